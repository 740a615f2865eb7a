// The fused attention forward's kernels with a key split (see
// flash_fwd_kernel.hpp), for grids too short to fill the GPU with 256-row
// blocks.
#include "flash_fwd_kernel.hpp"

namespace sa {
namespace {

template <typename T, bool QK8, bool V8, bool ROPE, int KS>
int launch_d(const FlashParams& prm, hipStream_t st) {
    if (prm.dr <= 32) return launch_flash_split<T, 32, QK8, V8, ROPE, KS>(prm, st);
    if (prm.dr <= 64) return launch_flash_split<T, 64, QK8, V8, ROPE, KS>(prm, st);
    return launch_flash_split<T, 128, QK8, V8, ROPE, KS>(prm, st);
}

template <int KS>
int launch_kind(FlashKind kind, const FlashParams& prm, hipStream_t st) {
    switch (kind) {
        case kFlashBf16: return launch_d<bf16, false, false, false, KS>(prm, st);
        case kFlashF16: return launch_d<f16, false, false, false, KS>(prm, st);
        case kFlashRopeBf16: return launch_d<bf16, false, false, true, KS>(prm, st);
        case kFlashRopeF16: return launch_d<f16, false, false, true, KS>(prm, st);
        case kFlashFp8: return launch_d<bf16, true, false, false, KS>(prm, st);
        case kFlashFp8V8: return launch_d<bf16, true, true, false, KS>(prm, st);
    }
    return SA_ERR_UNSUPPORTED;
}

}  // namespace

int flash_fwd_key_split(FlashKind kind, int ks, const FlashParams& prm, hipStream_t st) {
    return ks == 2 ? launch_kind<2>(kind, prm, st) : launch_kind<4>(kind, prm, st);
}

}  // namespace sa
