// Tiled linear layers in f16: instantiations of linear_gemm_kernels.hpp.
#include "linear_gemm_kernels.hpp"

namespace llaisys::kernels {

void gemmF16(GemmTile t, const GemmArgs &a, bool swiglu, hipStream_t s) { gemm16<F16>(t, a, swiglu, s); }

} // namespace llaisys::kernels
