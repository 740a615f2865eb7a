// Per-tensor absmax quantisation to float8_e4m3fn, entirely on the device
// (reference kernels.py:2592-2601, which synchronises through .item()):
//   scale = max(amax|x| / 448, 1e-12);  x8 = e4m3fn(clamp(x / scale, +-448))
// Both entry points run the same two passes.  The first leaves one maximum
// per block; the second reduces a tensor's maxima in every block and writes
// the codes.  sa_fp8_quantize_many puts up to kMaxTensors tensors into each
// pass, its blocks dealt out by size: a forward from 16-bit q, k and v takes
// two launches where a call per tensor takes nine (three each, the first to
// clear the one word that its blocks meet in).
// HBM binds the large sizes and the launches the small ones: q, k and v of a
// [2,32/8,8192,128] forward 103 -> 79 us, its whole call 945 -> 919 us; a
// [1,32/8,2048,128] call 83 -> 55 us.  Walking the second pass backwards,
// towards what the first read last, changed nothing.  Both passes
// read 16 bytes per lane and load when x is 16-byte aligned (the remainder,
// and unaligned inputs, element by element), several loads in flight per lane.
#include "common.hpp"

namespace sa {
namespace {

constexpr int kQThreads = 256;
constexpr int kMaxTensors = 4;
// Maxima kept per tensor, so also the most blocks of the amax pass on one.
constexpr unsigned kSlots = SA_FP8_AMAX_WORDS;
// Blocks of the amax pass over all tensors.  More cost (a single tensor of
// 2^24 fp32, 256 / 384 / 512 / 1024 blocks: 26.6 / 27.2 / 27.7 / 29.2 us; of 2^26
// bf16 52.3 / 52.5 / 53.6 / 56.1), fewer leave q, k and v of short calls waiting
// ([1,32/8,2048,128] 14.2 / 12.3 / 15.5 / 14.4).  A caller that brings one word
// instead of kSlots has the blocks meet in it by atomicMax (non-negative floats
// order like their bit patterns); those serialise, so that route keeps to one
// block per CU.
constexpr unsigned kAmaxBlocks = 384;
constexpr unsigned kAmaxAtomicBlocks = 256;
// Inputs up to this size are read through the caches, so that the second pass
// finds there what the first has just read (nontemporal loads -> these, whole
// calls, bf16 inputs: [1,32/8,2048,128] 61.1 -> 55.3 us, [8,32/8,1024,128] 124.7
// -> 120.5, [1,32/8,8192,128] 467.9 -> 463.7).  Past the size of the 256 MB
// last-level cache it finds nothing and the lines it left cost: nontemporal
// loads and one block per CU, as -> through the caches, 268 MB 113 -> 112 us,
// 402 MB 149 -> 165, 537 MB 196 -> 230.
constexpr int64_t kCachedBytes = int64_t(320) << 20;
constexpr int kAmaxUnroll = 8;
static_assert(kAmaxBlocks <= kSlots && kAmaxAtomicBlocks <= kSlots, "one word per block");
constexpr unsigned kQuantBlocks = 4096;

struct QuantTensor {
    const void* x;
    uint8_t* x8;
    int64_t n;
    uint32_t* maxima;  // bits of the blocks' maxima
    float* scale_out;
    unsigned amax_begin, amax_blocks;    // this tensor's blocks of the amax pass
    unsigned quant_begin, quant_blocks;  // and of the second
    int vec;                             // 16-byte loads
};

struct QuantArgs {
    QuantTensor t[kMaxTensors];
    int count;
    int shared_word;  // the maxima are one word, met by atomicMax
};

__global__ void fill_zero_u32(uint32_t* p) { p[0] = 0u; }

// 16-byte loads: nontemporal (STREAM), or leaving their lines in the caches
// (see kCachedBytes).
template <bool STREAM, typename T>
__device__ __forceinline__ void load_x(const T* p, uint32_t* words) {
    if constexpr (STREAM) {
        load_words(p, words);
    } else {
        const u32x4 v = *reinterpret_cast<const u32x4*>(p);
        words[0] = v.x;
        words[1] = v.y;
        words[2] = v.z;
        words[3] = v.w;
    }
}

template <typename T>
__device__ __forceinline__ float ld(const T* p, int64_t i) { return to_f32(p[i]); }

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    return v;
}

// The largest v of the block, in every thread.
__device__ __forceinline__ float block_max(float v) {
    __shared__ float part[kQThreads / 64];
    v = wave_max(v);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    float b = part[0];
#pragma unroll
    for (int w = 1; w < kQThreads / 64; ++w) b = fmaxf(b, part[w]);
    return b;
}

template <typename T, bool STREAM>
__global__ __launch_bounds__(kQThreads) void amax_kernel(const QuantArgs a) {
    int ti = 0;
    while (ti + 1 < a.count && blockIdx.x >= a.t[ti + 1].amax_begin) ++ti;
    const QuantTensor& qt = a.t[ti];
    const T* __restrict__ x = static_cast<const T*>(qt.x);
    const int64_t n = qt.n;
    const unsigned block = blockIdx.x - qt.amax_begin;
    constexpr int NV = 16 / sizeof(T);  // elements per 16-byte load
    float m = 0.f;
    const int64_t stride = static_cast<int64_t>(qt.amax_blocks) * kQThreads;
    const int64_t tid0 = static_cast<int64_t>(block) * kQThreads + threadIdx.x;
    const int64_t nv = qt.vec ? n / NV : 0;
    int64_t i = tid0;
    // kAmaxUnroll independent 16-byte loads in flight per lane: the grid is
    // small (see kSlots), so each lane must keep several loads going
    constexpr int U = kAmaxUnroll;
    for (; i + (U - 1) * stride < nv; i += U * stride) {
        uint32_t w[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) load_x<STREAM>(x + (i + u * stride) * NV, w[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < NV; ++e) m = fmaxf(m, fabsf(elem<T>(w[u], e)));
    }
    for (; i < nv; i += stride) {
        uint32_t w[4];
        load_x<STREAM>(x + i * NV, w);
#pragma unroll
        for (int e = 0; e < NV; ++e) m = fmaxf(m, fabsf(elem<T>(w, e)));
    }
    for (int64_t i = nv * NV + tid0; i < n; i += stride) m = fmaxf(m, fabsf(ld(x, i)));
    m = block_max(m);
    if (threadIdx.x != 0) return;
    if (a.shared_word) atomicMax(qt.maxima, __float_as_uint(m));
    else qt.maxima[block] = __float_as_uint(m);
}

// x / scale, clamped, as the correctly rounded quotient would be coded.  A
// true fp32 division is about ten operations per element, which the pass
// waited for.  For 16-bit x the quotient from the scale's reciprocal and one
// residual step (Markstein, 1990) takes three, and its codes equal the true
// division's for every pair of a 16-bit x and a 16-bit amax >= |x|; copysign
// keeps the sign of a zero, and an infinite scale takes no residual (finite x
// give zeros, infinite ones NaN, as the division does).  fp32 x divide.
template <typename T>
struct Quotient {
    float scale, inv;
    __device__ __forceinline__ explicit Quotient(float s) : scale(s), inv(1.f / s) {
        if constexpr (sizeof(T) == 2) scale = s == __builtin_inff() ? 0.f : s;
    }
    __device__ __forceinline__ float operator()(float x) const {
        float v;
        if constexpr (sizeof(T) == 2) {
            const float q = x * inv;
            v = copysignf(fmaf(fmaf(-q, scale, x), inv, q), x);
        } else {
            v = x / scale;
        }
        return fminf(fmaxf(v, -448.f), 448.f);
    }
};

// Round-to-nearest-even conversion of a value already clamped to +-448.
__device__ __forceinline__ uint32_t to_e4m3(float v) {
    return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(v, v, 0, false)) & 0xFFu;
}

// Four clamped values -> one word of e4m3fn codes (element e in byte e).
__device__ __forceinline__ uint32_t pack_e4m3(float v0, float v1, float v2, float v3) {
    const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(v0, v1, 0, false);
    return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(v2, v3, lo, true));
}

template <typename T, bool STREAM>
__global__ __launch_bounds__(kQThreads) void quant_kernel(const QuantArgs a) {
    constexpr int NV = 16 / sizeof(T);  // elements per 16-byte load
    int ti = 0;
    while (ti + 1 < a.count && blockIdx.x >= a.t[ti + 1].quant_begin) ++ti;
    const QuantTensor& qt = a.t[ti];
    const T* __restrict__ x = static_cast<const T*>(qt.x);
    uint8_t* __restrict__ x8 = qt.x8;
    const int64_t n = qt.n;
    const unsigned block = blockIdx.x - qt.quant_begin;
    float m = 0.f;
    const unsigned words = a.shared_word ? 1u : qt.amax_blocks;
    for (unsigned w = threadIdx.x; w < words; w += kQThreads) m = fmaxf(m, __uint_as_float(qt.maxima[w]));
    const float scale = fmaxf(block_max(m) / 448.f, 1e-12f);
    const Quotient<T> quotient(scale);
    if (block == 0 && threadIdx.x == 0) qt.scale_out[0] = scale;
    const int64_t stride = static_cast<int64_t>(qt.quant_blocks) * kQThreads;
    const int64_t tid0 = static_cast<int64_t>(block) * kQThreads + threadIdx.x;
    if (qt.vec) {
        // NV elements per thread and step: one 16-byte load, NV / 4 word stores
        const int64_t nv = n / NV;
        auto emit = [&](int64_t j, const uint32_t* w) {
            float v[NV];
#pragma unroll
            for (int e = 0; e < NV; ++e) v[e] = quotient(elem<T>(w, e));
            if constexpr (NV == 8) {
                *reinterpret_cast<uint2*>(x8 + j * NV) =
                    uint2{pack_e4m3(v[0], v[1], v[2], v[3]), pack_e4m3(v[4], v[5], v[6], v[7])};
            } else {
                *reinterpret_cast<uint32_t*>(x8 + j * NV) = pack_e4m3(v[0], v[1], v[2], v[3]);
            }
        };
        int64_t i = tid0;
        for (; i + stride < nv; i += 2 * stride) {  // two loads in flight per lane
            uint32_t w0[4], w1[4];
            load_x<STREAM>(x + i * NV, w0);
            load_x<STREAM>(x + (i + stride) * NV, w1);
            emit(i, w0);
            emit(i + stride, w1);
        }
        for (; i < nv; i += stride) {
            uint32_t w[4];
            load_x<STREAM>(x + i * NV, w);
            emit(i, w);
        }
        if (block == 0) {
            for (int64_t i = nv * NV + threadIdx.x; i < n; i += kQThreads) {
                const float v = quotient(ld(x, i));
                x8[i] = static_cast<uint8_t>(to_e4m3(v));
            }
        }
        return;
    }
    // four elements per thread and step, one 32-bit store
    const int64_t n4 = n / 4;
    for (int64_t i = tid0; i < n4; i += stride) {
        uint32_t word = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = quotient(ld(x, 4 * i + e));
            word |= to_e4m3(v) << (8 * e);
        }
        reinterpret_cast<uint32_t*>(x8)[i] = word;
    }
    if (block == 0) {
        for (int64_t i = 4 * n4 + threadIdx.x; i < n; i += kQThreads) {
            const float v = quotient(ld(x, i));
            x8[i] = static_cast<uint8_t>(to_e4m3(v));
        }
    }
}

// Deals out the blocks of both passes by size and launches them.
template <typename T>
int launch_quant(QuantArgs& a, hipStream_t st) {
    constexpr int NV = 16 / sizeof(T);
    constexpr int64_t kPerBlock = kQThreads * 4 * NV;
    double total = 0;
    for (int i = 0; i < a.count; ++i) total += static_cast<double>(a.t[i].n);
    const bool stream = total * sizeof(T) > static_cast<double>(kCachedBytes);
    const unsigned amax_limit = a.shared_word || stream ? kAmaxAtomicBlocks : kAmaxBlocks;
    unsigned amax_grid = 0, quant_grid = 0;
    for (int i = 0; i < a.count; ++i) {
        QuantTensor& t = a.t[i];
        // 16-byte steps need x 16-byte aligned and x8 aligned to the step's
        // output (8 or 4 bytes; the entry points require 4)
        t.vec = aligned16(t.x) && (reinterpret_cast<uintptr_t>(t.x8) % NV) == 0 ? 1 : 0;
        const int64_t want = (t.n + kPerBlock - 1) / kPerBlock;
        const double share = total > 0 ? static_cast<double>(t.n) / total : 0;
        auto blocks = [&](unsigned limit) {
            const int64_t most = static_cast<int64_t>(share * limit);
            const int64_t b = want < most ? want : most;
            return static_cast<unsigned>(b < 1 ? 1 : b);
        };
        t.amax_begin = amax_grid;
        t.quant_begin = quant_grid;
        amax_grid += t.amax_blocks = blocks(amax_limit);
        quant_grid += t.quant_blocks = blocks(kQuantBlocks);
    }
    if (stream) {
        amax_kernel<T, true><<<amax_grid, kQThreads, 0, st>>>(a);
        quant_kernel<T, true><<<quant_grid, kQThreads, 0, st>>>(a);
    } else {
        amax_kernel<T, false><<<amax_grid, kQThreads, 0, st>>>(a);
        quant_kernel<T, false><<<quant_grid, kQThreads, 0, st>>>(a);
    }
    return status_from_launch();
}

int launch_quant(QuantArgs& a, int dtype, hipStream_t st) {
    if (dtype != SA_F32 && dtype != SA_F16 && dtype != SA_BF16) return SA_ERR_BAD_DTYPE;
    if (a.shared_word) fill_zero_u32<<<1, 1, 0, st>>>(a.t[0].maxima);
    switch (dtype) {
        case SA_F32: return launch_quant<float>(a, st);
        case SA_F16: return launch_quant<f16>(a, st);
        default: return launch_quant<bf16>(a, st);
    }
}

}  // namespace
}  // namespace sa

extern "C" int sa_fp8_quantize(const void* x, void* x8, int64_t n, int dtype, float* amax_ws, float* scale_out,
                               sa_stream_t stream) {
    using namespace sa;
    if (n < 0) return SA_ERR_BAD_SHAPE;
    if (!amax_ws || !scale_out || (n > 0 && (!x || !x8))) return SA_ERR_NULL_POINTER;
    if ((reinterpret_cast<uintptr_t>(x8) & 3u) != 0) return SA_ERR_BAD_STRIDE;
    QuantArgs a{};
    a.count = 1;
    a.shared_word = 1;
    a.t[0].x = x;
    a.t[0].x8 = static_cast<uint8_t*>(x8);
    a.t[0].n = n;
    a.t[0].maxima = reinterpret_cast<uint32_t*>(amax_ws);
    a.t[0].scale_out = scale_out;
    return launch_quant(a, dtype, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int sa_fp8_quantize_many(int count, const void* const* x, void* const* x8, const int64_t* n, int dtype,
                                    float* amax_ws, float* scales_out, sa_stream_t stream) {
    using namespace sa;
    if (count < 1 || count > kMaxTensors) return SA_ERR_BAD_SHAPE;
    if (!x || !x8 || !n || !amax_ws || !scales_out) return SA_ERR_NULL_POINTER;
    QuantArgs a{};
    a.count = count;
    for (int i = 0; i < count; ++i) {
        if (n[i] < 0) return SA_ERR_BAD_SHAPE;
        if (n[i] > 0 && (!x[i] || !x8[i])) return SA_ERR_NULL_POINTER;
        if ((reinterpret_cast<uintptr_t>(x8[i]) & 3u) != 0) return SA_ERR_BAD_STRIDE;
        a.t[i].x = x[i];
        a.t[i].x8 = static_cast<uint8_t*>(x8[i]);
        a.t[i].n = n[i];
        a.t[i].maxima = reinterpret_cast<uint32_t*>(amax_ws) + static_cast<int64_t>(i) * kSlots;
        a.t[i].scale_out = scales_out + i;
    }
    return launch_quant(a, dtype, reinterpret_cast<hipStream_t>(stream));
}
