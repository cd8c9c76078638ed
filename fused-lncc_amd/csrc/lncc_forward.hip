// Instantiations and launcher of the forward-only LNCC kernel.
#include "lncc_forward_kernel.h"

namespace fl {

template <int HH, int NC>
static hipError_t launch_forward_h(int mode, bool bf16, const FusedArgs& a, uint32_t nblocks, hipStream_t st) {
    const dim3 grid(nblocks), block(FwdGeo<HH, NC>::LANES);
#define FL_LAUNCH(BF, MD) hipLaunchKernelGGL((lncc_forward_kernel<HH, NC, BF, MD>), grid, block, 0, st, a)
    if (mode == MODE_LOSS) {
        if (bf16) FL_LAUNCH(true, MODE_LOSS); else FL_LAUNCH(false, MODE_LOSS);
    } else if (mode == MODE_MAPS) {
        if (bf16) FL_LAUNCH(true, MODE_MAPS); else FL_LAUNCH(false, MODE_MAPS);
    } else {
        return hipErrorInvalidValue;
    }
#undef FL_LAUNCH
    return hipGetLastError();
}

hipError_t launch_forward(int halo, int cols, int mode, bool bf16, const FusedArgs& a, uint32_t nblocks, hipStream_t st) {
    switch (halo * 10 + cols) {
        case 13: return launch_forward_h<1, 3>(mode, bf16, a, nblocks, st);
        case 23: return launch_forward_h<2, 3>(mode, bf16, a, nblocks, st);
        case 33: return launch_forward_h<3, 3>(mode, bf16, a, nblocks, st);
        case 43: return launch_forward_h<4, 3>(mode, bf16, a, nblocks, st);
        case 14: return launch_forward_h<1, 4>(mode, bf16, a, nblocks, st);
        case 24: return launch_forward_h<2, 4>(mode, bf16, a, nblocks, st);
        case 34: return launch_forward_h<3, 4>(mode, bf16, a, nblocks, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace fl
