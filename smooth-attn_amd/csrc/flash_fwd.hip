// Host side of the fused attention forward for head dims up to 128 (bf16 /
// fp16, RoPE and fp8): argument checks, the choice of the kernel's key split
// and the launches; the K rotation of the RoPE forward.  The kernel is in
// flash_fwd_kernel.hpp.
#include <algorithm>

#include "flash_fwd_kernel.hpp"
#include "flash_f32.hpp"
#include "flash_wide.hpp"

namespace sa {
namespace {

// Rotates every row of K once into a contiguous [B, Hkv, T, D] buffer for the
// RoPE forward (each K tile is re-read by every query block of its head, so
// rotating K once beats rotating it in each block).  One thread per pair of
// 16-byte chunks (d, d + D/2).
template <typename T, int D>
__global__ __launch_bounds__(256) void rope_rotate_rows(const T* __restrict__ k, T* __restrict__ out,
                                                        const float* __restrict__ cs, const float* __restrict__ sn,
                                                        int Hkv, int T_, int64_t s0, int64_t s1, int64_t s2,
                                                        int64_t n_pairs) {
    constexpr int PPR = D / 16;  // chunk pairs per row
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (gid >= n_pairs) return;
    const int64_t row = gid / PPR;
    const int c = static_cast<int>(gid - row * PPR);
    const int64_t bh = row / T_;
    const int t = static_cast<int>(row - bh * T_);
    const int b = static_cast<int>(bh / Hkv);
    const int h = static_cast<int>(bh - static_cast<int64_t>(b) * Hkv);
    const T* src = k + b * s0 + h * s1 + t * s2 + c * 8;
    u32x4 a = load16(src);
    u32x4 bb = load16(src + D / 2);
    float cv[8], sv[8];
    const float* cr = cs + static_cast<int64_t>(t) * (D / 2) + c * 8;
    const float* sr = sn + static_cast<int64_t>(t) * (D / 2) + c * 8;
    *reinterpret_cast<float4*>(cv) = *reinterpret_cast<const float4*>(cr);
    *reinterpret_cast<float4*>(cv + 4) = *reinterpret_cast<const float4*>(cr + 4);
    *reinterpret_cast<float4*>(sv) = *reinterpret_cast<const float4*>(sr);
    *reinterpret_cast<float4*>(sv + 4) = *reinterpret_cast<const float4*>(sr + 4);
    rope_rotate8<T>(a, bb, cv, sv);
    T* dst = out + row * D + c * 8;
    *reinterpret_cast<u32x4*>(dst) = a;
    *reinterpret_cast<u32x4*>(dst + D / 2) = bb;
}

// The same rotation for any head dim D that is a multiple of 16 (pairs of
// 16-byte chunks (d, d + D/2)), from strided rows into a contiguous
// [B, H, T, D] buffer: the first pass of RoPE attention at head dims the
// fused Q rotation does not cover.
template <typename T>
__global__ __launch_bounds__(256) void rope_rotate_any(const T* __restrict__ x, T* __restrict__ out,
                                                       const float* __restrict__ cs, const float* __restrict__ sn,
                                                       int H, int T_, int D, int64_t s0, int64_t s1, int64_t s2,
                                                       int64_t n_pairs) {
    const int ppr = D / 16;  // chunk pairs per row
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (gid >= n_pairs) return;
    const int64_t row = gid / ppr;
    const int c = static_cast<int>(gid - row * ppr);
    const int64_t bh = row / T_;
    const int t = static_cast<int>(row - bh * T_);
    const int b = static_cast<int>(bh / H);
    const int h = static_cast<int>(bh - static_cast<int64_t>(b) * H);
    const T* src = x + b * s0 + h * s1 + t * s2 + c * 8;
    float cv[8], sv[8];
    const float* cr = cs + static_cast<int64_t>(t) * (D / 2) + c * 8;
    const float* sr = sn + static_cast<int64_t>(t) * (D / 2) + c * 8;
    *reinterpret_cast<float4*>(cv) = *reinterpret_cast<const float4*>(cr);
    *reinterpret_cast<float4*>(cv + 4) = *reinterpret_cast<const float4*>(cr + 4);
    *reinterpret_cast<float4*>(sv) = *reinterpret_cast<const float4*>(sr);
    *reinterpret_cast<float4*>(sv + 4) = *reinterpret_cast<const float4*>(sr + 4);
    T* dst = out + row * D + c * 8;
    if constexpr (std::is_same_v<T, float>) {  // 8 fp32 elements: two 16-byte loads per half
        float a[8], bb[8];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            *reinterpret_cast<float4*>(a + 4 * j) = *reinterpret_cast<const float4*>(src + 4 * j);
            *reinterpret_cast<float4*>(bb + 4 * j) = *reinterpret_cast<const float4*>(src + D / 2 + 4 * j);
        }
        float ra[8], rb[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            ra[e] = a[e] * cv[e] - bb[e] * sv[e];
            rb[e] = bb[e] * cv[e] + a[e] * sv[e];
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            *reinterpret_cast<float4*>(dst + 4 * j) = *reinterpret_cast<const float4*>(ra + 4 * j);
            *reinterpret_cast<float4*>(dst + D / 2 + 4 * j) = *reinterpret_cast<const float4*>(rb + 4 * j);
        }
    } else {
        u32x4 a = load16(src);
        u32x4 bb = load16(src + D / 2);
        rope_rotate8<T>(a, bb, cv, sv);
        *reinterpret_cast<u32x4*>(dst) = a;
        *reinterpret_cast<u32x4*>(dst + D / 2) = bb;
    }
}

// Estimated microseconds of the forward with key split KS, one block per CU:
// the longer of the longest block and all blocks shared out evenly, plus a
// part of the other (the ragged end).
struct SplitCosts {
    double setup, tile;        // the longest block: loads of Q and the first tile and the epilogue; per K/V tile
    double share_setup, share; // the same of a block in a full grid, per CU
};
struct ForwardCosts {
    SplitCosts ks1, ks2, ks4;
    double ragged, margin;
};
template <int KS>
double forward_estimate(const FlashParams& p, const SplitCosts& c, double ragged) {
    constexpr int kCus = 256;
    constexpr int BQ = Split<KS>::BQ, BKV = Split<KS>::BKV;
    const int nqb = (p.T + BQ - 1) / BQ, n_kv = (p.T + BKV - 1) / BKV;
    int64_t sum = 0;
    int longest = 0;
    for (int qb = 0; qb < nqb; ++qb) {
        const int q0 = qb * BQ;
        const int first = p.window > 0 ? std::max(0, q0 - p.window + 1) / BKV : 0;
        const int n = std::min((q0 + BQ + BKV - 1) / BKV, n_kv) - first;
        sum += n;
        longest = std::max(longest, n);
    }
    const double one = c.setup + longest * c.tile;
    const double all = static_cast<double>(p.B) * p.Hq * (nqb * c.share_setup + static_cast<double>(sum) * c.share) / kCus;
    return std::max(one, all) + ragged * std::min(one, all);
}

// Key split of a launch (1, 2 or 4).  A split shortens the blocks, for grids
// that leave CUs idle or waiting for the longest block, but costs a merge and
// more barriers per MFMA, so full grids keep KS = 1 at D = 128; at D = 64 two
// KS = 2 blocks fit a CU (under 128 registers) and it wins over most sizes.
// The constants (for D <= 128, 64 and 32, about us) are fitted to the 811
// measured shapes of profiles/attention_fwd_key_split_us.csv (bf16, T = 256 ..
// 8192, up to 1100 blocks of 256 rows, GQA 1 to 8, windows of none to most), on
// which the choice averages 0.5%, 0.5% and 1.0% over the fastest KS and takes
// 0.84, 0.80 and 0.76 of the time of KS = 1 throughout, at worst 1.09, 1.17 and
// 1.09.  KS = 1 / 2 / 4 in us,
// D = 128: [1,32/8,512] 18.7 / 15.3 / 13.1, [1,32/8,1024] 31.4 / 23.4 / 26.2,
// [1,32/8,2048] 58.0 / 52.4 / 69.9, [1,8,2048] 54.3 / 35.5 / 25.6,
// [2,32/8,1024] 34.0 / 35.3 / 49.4; D = 64: [1,32/8,5760] 207 / 179 / 251.
// Longer grids (over 512 blocks of 256 rows, 768 at D = 64) gain no more than
// their noise or lose ([1,32,8128] at D = 64, 1024 blocks, 350 / 374) and skip
// the estimate.  KS = 4 walks tiles of 128 rows, whose 32-bit offsets bound
// the row stride.
constexpr ForwardCosts kForwardCosts128 = {{6.5, 1.35, 7.7, 1.54}, {6.8, 0.78, 11.6, 1.01}, {4.7, 1.10, 9.2, 1.16}, 0.093, 1.16};
constexpr ForwardCosts kForwardCosts64 = {{9.7, 1.99, 4.6, 3.53}, {8.3, 0.85, 3.3, 1.25}, {7.1, 1.35, 8.1, 1.15}, 0.35, 1.02};
constexpr ForwardCosts kForwardCosts32 = {{4.0, 0.87, 0.0, 1.15}, {4.3, 0.53, 2.6, 0.53}, {4.1, 0.66, 3.1, 0.43}, 0.49, 1.0};
int key_split_for(const FlashParams& p, int qk_bytes, int v_bytes) {
    const int64_t limit = p.dr > 32 && p.dr <= 64 ? 768 : 512;
    if (static_cast<int64_t>(p.nqb) * p.B * p.Hq > limit) return 1;
    constexpr int64_t kMaxStride4 = int64_t(1) << 23;
    const ForwardCosts& c = p.dr > 64 ? kForwardCosts128 : p.dr > 32 ? kForwardCosts64 : kForwardCosts32;
    const double e1 = forward_estimate<1>(p, c.ks1, c.ragged);
    const double e2 = forward_estimate<2>(p, c.ks2, c.ragged);
    const double e4 = p.ks[2] * qk_bytes <= kMaxStride4 && p.vs[2] * v_bytes <= kMaxStride4
                          ? forward_estimate<4>(p, c.ks4, c.ragged)
                          : 2.0 * e2;
    if (std::min(e2, e4) >= c.margin * e1) return 1;
    return e4 < e2 ? 4 : 2;
}

template <typename T, int D, bool QK8, bool V8>
int launch_flash(FlashParams prm, int exact, hipStream_t st) {
    if (exact) {
        set_grid(prm, Split<1>::BQ, Split<1>::BKV);
        const dim3 grid(static_cast<unsigned>(prm.nqb) * prm.B * prm.Hq);
        flash_fwd_kernel<T, D, QK8, V8, true, false><<<grid, dim3(kThreads), 0, st>>>(prm);
        return status_from_launch();
    }
    const int ks = key_split_for(prm, QK8 ? 1 : 2, V8 ? 1 : 2);
    if (ks > 1) {
        const FlashKind kind = QK8 ? (V8 ? kFlashFp8V8 : kFlashFp8) : std::is_same_v<T, bf16> ? kFlashBf16 : kFlashF16;
        return flash_fwd_key_split(kind, ks, prm, st);
    }
    return launch_flash_split<T, D, QK8, V8, false, 1>(prm, st);
}

// RoPE forward: K rotated into k_rot (contiguous [B, Hkv, T, D]), then the
// forward with Q rotated in registers.
template <typename T, int D>
int launch_rope(FlashParams prm, T* k_rot, hipStream_t st) {
    const int64_t n_pairs = static_cast<int64_t>(prm.B) * prm.Hkv * prm.T * (D / 16);
    const dim3 rgrid(static_cast<unsigned>((n_pairs + 255) / 256));
    rope_rotate_rows<T, D><<<rgrid, 256, 0, st>>>(static_cast<const T*>(prm.k), k_rot, prm.rope_cos, prm.rope_sin,
                                                  prm.Hkv, prm.T, prm.ks[0], prm.ks[1], prm.ks[2], n_pairs);
    int stt = status_from_launch();
    if (stt != 0) return stt;
    prm.k = k_rot;
    prm.ks[0] = static_cast<int64_t>(prm.Hkv) * prm.T * D;
    prm.ks[1] = static_cast<int64_t>(prm.T) * D;
    prm.ks[2] = D;
    prm.ks[3] = 1;
    const int ks = key_split_for(prm, 2, 2);
    if (ks > 1) return flash_fwd_key_split(std::is_same_v<T, bf16> ? kFlashRopeBf16 : kFlashRopeF16, ks, prm, st);
    return launch_flash_split<T, D, false, false, true, 1>(prm, st);
}

// Head dims 8..128 (multiples of 8) run on the kernel for the next of 32,
// 64, 128 with the columns past prm.dr masked.
template <typename T, bool QK8, bool V8>
int launch_flash_d(const FlashParams& prm, int exact, hipStream_t st) {
    if (prm.dr <= 32) return launch_flash<T, 32, QK8, V8>(prm, exact, st);
    if (prm.dr <= 64) return launch_flash<T, 64, QK8, V8>(prm, exact, st);
    return launch_flash<T, 128, QK8, V8>(prm, exact, st);
}

// Largest K / V row stride (bytes) the tile loads address with 32-bit offsets.
constexpr int64_t kMaxRowStrideBytes = int64_t(1) << 24;

// (b, h, t) strides must keep every row start 16-byte aligned; d stride 1.
bool strides_ok(const int64_t* s, int elem_bytes) {
    const int64_t a = 16 / elem_bytes;
    return s[3] == 1 && s[0] % a == 0 && s[1] % a == 0 && s[2] % a == 0;
}

void set_sizes(FlashParams& prm, int B, int Hq, int Hkv, int T, int D, int window_size) {
    prm.B = B;
    prm.Hq = Hq;
    prm.Hkv = Hkv;
    prm.T = T;
    prm.G = Hq / Hkv;
    prm.window = window_size;
    prm.dr = D;
    prm.nqb = (T + Split<1>::BQ - 1) / Split<1>::BQ;
}

int fill_params(FlashParams& prm, const void* q, const void* k, const void* v, void* o, float* row_sums, int B,
                int Hq, int Hkv, int T, int D, const int64_t* q_strides, const int64_t* k_strides,
                const int64_t* v_strides, const int64_t* o_strides, float scale, int window_size, int qk_bytes,
                int v_bytes) {
    if (B < 0 || Hq <= 0 || Hkv <= 0 || T < 0 || Hq % Hkv != 0 || window_size < 0) return SA_ERR_BAD_SHAPE;
    if (!q || !k || !v || !o || !q_strides || !k_strides || !v_strides || !o_strides) return SA_ERR_NULL_POINTER;
    if (D < 8 || D > 128 || D % 8 != 0) return SA_ERR_UNSUPPORTED;
    if (!strides_ok(q_strides, qk_bytes) || !strides_ok(k_strides, qk_bytes) || !strides_ok(v_strides, v_bytes) ||
        !strides_ok(o_strides, 2) || !aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o))
        return SA_ERR_BAD_STRIDE;
    // K / V tile loads use 32-bit offsets within a tile of at most 128 rows.
    if (k_strides[2] * qk_bytes > kMaxRowStrideBytes || v_strides[2] * v_bytes > kMaxRowStrideBytes)
        return SA_ERR_BAD_STRIDE;
    prm.q = q;
    prm.k = k;
    prm.v = v;
    prm.o = o;
    prm.row_sums = row_sums;
    for (int i = 0; i < 4; ++i) {
        prm.qs[i] = q_strides[i];
        prm.ks[i] = k_strides[i];
        prm.vs[i] = v_strides[i];
        prm.os[i] = o_strides[i];
    }
    set_sizes(prm, B, Hq, Hkv, T, D, effective_window(window_size, T));
    prm.scale = scale;
    return 0;
}

}  // namespace
}  // namespace sa

extern "C" int sa_flash_fwd_key_split(int B, int Hq, int Hkv, int T, int D, int window_size, int exact_math,
                                      int64_t kv_row_bytes) {
    using namespace sa;
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || T <= 0 || Hq % Hkv != 0 || window_size < 0 || kv_row_bytes <= 0 ||
        kv_row_bytes > kMaxRowStrideBytes)
        return SA_ERR_BAD_SHAPE;
    if (D < 8 || D > 128 || D % 8 != 0) return SA_ERR_UNSUPPORTED;
    if (exact_math) return 1;
    FlashParams prm{};
    set_sizes(prm, B, Hq, Hkv, T, D, effective_window(window_size, T));
    prm.ks[2] = prm.vs[2] = kv_row_bytes;
    return key_split_for(prm, 1, 1);
}

extern "C" int sa_flash_fwd(const void* q, const void* k, const void* v, void* o, float* row_sums, int B, int Hq,
                            int Hkv, int T, int D, const int64_t* q_strides, const int64_t* k_strides,
                            const int64_t* v_strides, const int64_t* o_strides, float scale, int window_size,
                            int exact_math, int dtype, sa_stream_t stream) {
    using namespace sa;
    window_size = effective_window(window_size, T);
    if (dtype == SA_F32)
        return flash_fwd_f32(q, k, v, o, row_sums, B, Hq, Hkv, T, D, q_strides, k_strides, v_strides, o_strides,
                             scale, window_size, exact_math, reinterpret_cast<hipStream_t>(stream));
    if (dtype != SA_BF16 && dtype != SA_F16) return SA_ERR_BAD_DTYPE;
    if (D > 128)
        return flash_fwd_wide(q, k, v, o, row_sums, B, Hq, Hkv, T, D, q_strides, k_strides, v_strides, o_strides,
                              scale, window_size, exact_math, dtype, reinterpret_cast<hipStream_t>(stream));
    FlashParams prm{};
    const int st = fill_params(prm, q, k, v, o, row_sums, B, Hq, Hkv, T, D, q_strides, k_strides, v_strides,
                               o_strides, scale, window_size, 2, 2);
    if (st != 0) return st;
    if (B == 0 || T == 0) return 0;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int ex = exact_math ? 1 : 0;
    if (dtype == SA_BF16) return launch_flash_d<bf16, false, false>(prm, ex, s);
    return launch_flash_d<f16, false, false>(prm, ex, s);
}

extern "C" int sa_flash_fp8_fwd(const void* q8, const void* k8, const void* v, void* o, float* row_sums,
                                const float* q_scale, const float* k_scale, const float* v_scale, int B, int Hq,
                                int Hkv, int T, int D, const int64_t* q_strides, const int64_t* k_strides,
                                const int64_t* v_strides, const int64_t* o_strides, float attn_scale,
                                int window_size, int v_dtype, sa_stream_t stream) {
    using namespace sa;
    if (v_dtype != SA_FP8_E4M3FN && v_dtype != SA_BF16) return SA_ERR_BAD_DTYPE;
    const bool v8 = v_dtype == SA_FP8_E4M3FN;
    if (!q_scale || !k_scale || (v8 && !v_scale)) return SA_ERR_NULL_POINTER;
    FlashParams prm{};
    const int st = fill_params(prm, q8, k8, v, o, row_sums, B, Hq, Hkv, T, D, q_strides, k_strides, v_strides,
                               o_strides, attn_scale, window_size, 1, v8 ? 1 : 2);
    if (st != 0) return st;
    if (D != 32 && D != 64 && D != 128) return SA_ERR_UNSUPPORTED;  // fp8 kernels: native head dims only
    if (B == 0 || T == 0) return 0;
    prm.q_scale = q_scale;
    prm.k_scale = k_scale;
    prm.v_scale = v_scale;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (v8) return launch_flash_d<bf16, true, true>(prm, 0, s);
    return launch_flash_d<bf16, true, false>(prm, 0, s);
}

extern "C" int sa_rope_rotate(const void* x, void* out, const float* cos_table, const float* sin_table, int B,
                              int H, int T, int D, const int64_t* x_strides, int dtype, sa_stream_t stream) {
    using namespace sa;
    if (dtype != SA_BF16 && dtype != SA_F16 && dtype != SA_F32) return SA_ERR_BAD_DTYPE;
    if (B < 0 || H < 0 || T < 0 || D <= 0 || D % 16 != 0) return SA_ERR_BAD_SHAPE;
    if (!x || !out || !cos_table || !sin_table || !x_strides) return SA_ERR_NULL_POINTER;
    const int64_t* s = x_strides;
    const int64_t q16 = dtype == SA_F32 ? 4 : 8;  // elements per 16 bytes
    if (s[3] != 1 || s[0] % q16 || s[1] % q16 || s[2] % q16 || !aligned16(x) || !aligned16(out) ||
        !aligned16(cos_table) || !aligned16(sin_table))
        return SA_ERR_BAD_STRIDE;
    const int64_t n_pairs = static_cast<int64_t>(B) * H * T * (D / 16);
    if (n_pairs == 0) return 0;
    // one work-item per pair: the dispatch's grid x block count is 32-bit
    if ((n_pairs + 255) / 256 > INT32_MAX) return SA_ERR_BAD_SHAPE;
    const dim3 grid(static_cast<unsigned>((n_pairs + 255) / 256));
    if (!grid_fits(grid, dim3(256))) return SA_ERR_BAD_SHAPE;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (dtype == SA_F32)
        rope_rotate_any<float><<<grid, 256, 0, st>>>(static_cast<const float*>(x), static_cast<float*>(out),
                                                     cos_table, sin_table, H, T, D, s[0], s[1], s[2], n_pairs);
    else if (dtype == SA_BF16)
        rope_rotate_any<bf16><<<grid, 256, 0, st>>>(static_cast<const bf16*>(x), static_cast<bf16*>(out), cos_table,
                                                    sin_table, H, T, D, s[0], s[1], s[2], n_pairs);
    else
        rope_rotate_any<f16><<<grid, 256, 0, st>>>(static_cast<const f16*>(x), static_cast<f16*>(out), cos_table,
                                                   sin_table, H, T, D, s[0], s[1], s[2], n_pairs);
    return status_from_launch();
}

extern "C" int64_t sa_flash_rope_workspace_size(int B, int Hkv, int T, int D) {
    if (B < 0 || Hkv < 0 || T < 0 || D < 0) return -1;
    return static_cast<int64_t>(B) * Hkv * T * D * 2;
}

extern "C" int sa_flash_rope_fwd(const void* q, const void* k, const void* v, const float* cos_table,
                                 const float* sin_table, void* o, float* row_sums, void* k_rot_ws,
                                 int64_t ws_bytes, int B, int Hq, int Hkv, int T, int D,
                                 const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                 const int64_t* o_strides, float scale, int window_size, int dtype,
                                 sa_stream_t stream) {
    using namespace sa;
    if (dtype != SA_BF16 && dtype != SA_F16) return SA_ERR_BAD_DTYPE;
    if (!cos_table || !sin_table || !k_rot_ws) return SA_ERR_NULL_POINTER;
    FlashParams prm{};
    const int st = fill_params(prm, q, k, v, o, row_sums, B, Hq, Hkv, T, D, q_strides, k_strides, v_strides,
                               o_strides, scale, window_size, 2, 2);
    if (st != 0) return st;
    if (D != 32 && D != 64 && D != 128) return SA_ERR_UNSUPPORTED;  // fused RoPE: native head dims only
    if (B == 0 || T == 0) return 0;
    if (ws_bytes < sa_flash_rope_workspace_size(B, Hkv, T, D)) return SA_ERR_WORKSPACE;
    if (!aligned16(cos_table) || !aligned16(sin_table) || !aligned16(k_rot_ws)) return SA_ERR_BAD_STRIDE;
    prm.rope_cos = cos_table;
    prm.rope_sin = sin_table;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    switch (D) {
        case 32: return dtype == SA_BF16 ? launch_rope<bf16, 32>(prm, static_cast<bf16*>(k_rot_ws), s)
                                         : launch_rope<f16, 32>(prm, static_cast<f16*>(k_rot_ws), s);
        case 64: return dtype == SA_BF16 ? launch_rope<bf16, 64>(prm, static_cast<bf16*>(k_rot_ws), s)
                                         : launch_rope<f16, 64>(prm, static_cast<f16*>(k_rot_ws), s);
        case 128: return dtype == SA_BF16 ? launch_rope<bf16, 128>(prm, static_cast<bf16*>(k_rot_ws), s)
                                          : launch_rope<f16, 128>(prm, static_cast<f16*>(k_rot_ws), s);
        default: return SA_ERR_UNSUPPORTED;
    }
}
