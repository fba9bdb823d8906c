// Dense, and float MatMul, with too few output tiles to fill the chip with the tiled kernels (gemm_few.hip).
#pragma once

#include "gemm_rs.hpp"

namespace a4g {

enum FewKind { FEW_I8, FEW_I16X8, FEW_I16X16, FEW_BF16, FEW_F32, FEW_FP8 };

// g as the tiled kernels take it: K counts elements for the integer kinds and bytes for the floating-point ones, lda and
// stride_a are bytes, rows of A may start anywhere, rows of B are 16-byte aligned with a pitch that holds K rounded up to 16
// bytes. False where the kernel does not apply or the tiled kernels are ahead.
bool few_preferred(const GemmArgs& g, FewKind kind, int batch);
hipError_t launch_few(const GemmArgs& g, FewKind kind, int batch, hipStream_t stream);

}  // namespace a4g
