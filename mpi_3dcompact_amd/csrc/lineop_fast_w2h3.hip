// Fast line kernels of (W, H) = (2, 3): Penta10.
#include "lineop_fast_kernels.h"

namespace mc3d {

hipError_t lineop_launch_fast_w2h3(const OpDev &op, const LaunchArgs &a, int nfields, hipStream_t st) {
    return launch_fast_mm<2, 3>(op, a, nfields, st);
}

hipError_t lineop_launch_together_w2h3(const OpSet &o, const LaunchArgs &a, int nf, hipStream_t st) {
    switch (o.op[0].MM) {
        case 8: return launch_together<2, 3, 8>(o, a, nf, st);
        case 12: return launch_together<2, 3, 12>(o, a, nf, st);
        case 16: return launch_together<2, 3, 16>(o, a, nf, st);
        case 20: return launch_together<2, 3, 20>(o, a, nf, st);
        case 24: return launch_together<2, 3, 24>(o, a, nf, st);
        case 28: return launch_together<2, 3, 28>(o, a, nf, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mc3d
