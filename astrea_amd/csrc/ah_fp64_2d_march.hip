// 2D flux kernels in marching form, double arithmetic.
#include "ah_inst.h"

namespace ah {
bool kernels_2d_march_fp64(int mask, int recon, int solver, KernelSet* ks) {
    if (mask == 0x17 && solver == LLF) return set2d_march<0x17, LLF>(recon, ks);
    if (mask == 0x17 && solver == HLLC) return set2d_march<0x17, HLLC>(recon, ks);
    return kernels_2d_march_mhd_fp64(mask, recon, solver, ks);
}
}  // namespace ah
