// One instantiation family of the 2D kernels, compiled once per (dtype,
// prime class) by build.py with -DKYM_T=<float|double> -DKYM_P=<class>
// -DKYM_PICK=<function name> so the families build in parallel;
// -DKYM_GLOBAL_TW_ONLY for the family whose twiddles stay in global memory.
#include "kernels2d.h"

#ifdef KYM_GLOBAL_TW_ONLY
Scat2DKernel<KYM_T> KYM_PICK(int kind, int threads) { return pick_scat2d_global_tw<KYM_T, KYM_P>(kind, threads); }
#else
Scat2DKernel<KYM_T> KYM_PICK(int kind, int threads) { return pick_scat2d_p<KYM_T, KYM_P>(kind, threads); }
#endif
