// z2h_wide.hip — the quantized GEMMs of wide passes (z2h_gemm.h, z2h_gemm_q.h) in a translation unit of their
// own: z2h.hip declares them extern, and its own kernels keep their code layout.
#define Z2H_TEMPLATES_ONLY
#include "z2h_gemm_q.h"

namespace z2d {
template __global__ void k_gemm_q4k<true>(GemmArgs);
template __global__ void k_gemm_q4k<false>(GemmArgs);
template __global__ void k_gemm_q80<true, 1>(GemmArgs);
template __global__ void k_gemm_q80<true, 2>(GemmArgs);
template __global__ void k_gemm_q80<false, 1>(GemmArgs);
template __global__ void k_gemm_q80<false, 2>(GemmArgs);
template __global__ void k_gemm_q6k<true, 1>(GemmArgs);
template __global__ void k_gemm_q6k<true, 2>(GemmArgs);
template __global__ void k_gemm_q6k<true, 4>(GemmArgs);
template __global__ void k_gemm_q6k<false, 1>(GemmArgs);
template __global__ void k_gemm_q6k<false, 2>(GemmArgs);
template __global__ void k_gemm_q6k<false, 4>(GemmArgs);
} // namespace z2d
