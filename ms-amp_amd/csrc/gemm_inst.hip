// One pair of operand formats of the FP8 GEMM kernels (compiled four times: -DMSAMP_XF=5|6 -DMSAMP_YF=5|6), and once more
// per pair with -DMSAMP_GEMM_SECOND_UNIT for the small-tile and ragged-K instantiations, so that the eight units
// compile side by side.
#include "gemm_kernels.cuh"

namespace msamp {
#ifdef MSAMP_GEMM_SECOND_UNIT
template int run_gemm_ragged<MSAMP_XF, MSAMP_YF>(const GemmCall&);
template int run_gemm_small<MSAMP_XF, MSAMP_YF>(const GemmCall&);
template int run_gemm_pair128<MSAMP_XF, MSAMP_YF>(const GemmCall&);
template int run_gemm_parts<MSAMP_XF, MSAMP_YF>(const GemmCall&, const KSplit&);
#else
template int run_gemm_pair<MSAMP_XF, MSAMP_YF>(const GemmCall&);
#endif
}    // namespace msamp
