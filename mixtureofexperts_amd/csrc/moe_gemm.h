// moe_gemm.h -- rules of the fp32 grouped GEMMs that the layer's set-up shares.
#pragma once

namespace moe {
// Whether an fp32 call over m_tiles_grid M tiles (its rows / 128 + E) runs on
// the bf16 matrix unit (moe_gemm_f32x3.h).
bool f32x3_rows(int m_tiles_grid, int E);
}  // namespace moe
