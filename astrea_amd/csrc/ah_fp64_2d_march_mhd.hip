// 2D MHD flux kernels in marching form, double arithmetic.
#include "ah_inst.h"

namespace ah {
bool kernels_2d_march_mhd_fp64(int mask, int recon, int solver, KernelSet* ks) {
    if (mask == 0x77 && solver == HLLD) return set2d_march<0x77, HLLD>(recon, ks);
    return false;
}
}  // namespace ah
