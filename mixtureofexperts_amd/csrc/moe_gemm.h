// moe_gemm.h -- rules of the fp32 grouped GEMMs that the layer's set-up shares.
#pragma once

namespace moe {
// Whether an fp32 call's expert segments are long enough for the bf16 matrix
// unit (moe_gemm_f32x3.h): at most `rows` rows that `experts` experts hold.
bool f32x3_rows(long long rows, int experts);
}  // namespace moe
