// moe_decode.h -- the decode caller's device helpers and launchers
// (moe_decode.hip: routing, single tokens; moe_decode_batch.h: batches).
#pragma once
#include "moe_internal.h"

namespace moe {

__device__ __forceinline__ float readlane_f(float v, int i) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i));
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// Sum over each 16-lane row in a fixed order, every lane of the row ending
// with the same bits: pairs (quad_perm 1,0,3,2), quads (quad_perm 2,3,0,1),
// 8-lane halves (row_half_mirror), rows (row_mirror); additions commute
// exactly, so partner lanes hold identical values after every step.
__device__ __forceinline__ float row16_sum(float v) {
    v = v + dpp_f<0xb1>(v);
    v = v + dpp_f<0x4e>(v);
    v = v + dpp_f<0x141>(v);
    v = v + dpp_f<0x140>(v);
    return v;
}

// Wave sum (all 64 lanes active), uniform result: row sums, then the four rows
// in row order.
__device__ __forceinline__ float wave_sum(float v) {
    v = row16_sum(v);
    return ((readlane_f(v, 0) + readlane_f(v, 16)) + readlane_f(v, 32)) + readlane_f(v, 48);
}

__device__ __forceinline__ float4 zero_unless(bool v, float4 a) {
    return v ? a : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

__device__ __forceinline__ float dot4_acc(float acc, float4 a, float4 b) {
#pragma clang fp contract(off)
    acc = acc + a.x * b.x;
    acc = acc + a.y * b.y;
    acc = acc + a.z * b.z;
    acc = acc + a.w * b.w;
    return acc;
}

// 4 consecutive weights (element offset `o`, a multiple of 4) as fp32
template <int WT>
__device__ __forceinline__ float4 load_w4(const void *w, long long o) {
    if constexpr (WT == WT_F32) {
        return *(const float4 *)((const float *)w + o);
    } else if constexpr (WT == WT_BF16) {
        const uint2 q = *(const uint2 *)((const uint16_t *)w + o);
        return make_float4(__uint_as_float(q.x << 16), __uint_as_float(q.x & 0xffff0000u), __uint_as_float(q.y << 16),
                           __uint_as_float(q.y & 0xffff0000u));
    } else {
        const uint32_t q = *(const uint32_t *)((const uint8_t *)w + o);
        return make_float4(fp8e4m3_to_f32((uint8_t)q), fp8e4m3_to_f32((uint8_t)(q >> 8)),
                           fp8e4m3_to_f32((uint8_t)(q >> 16)), fp8e4m3_to_f32((uint8_t)(q >> 24)));
    }
}

// x = p[0] + p[1] + p[2], three bf16 values, exactly (the 24 significant bits
// in three groups of 8, cut off and not rounded, so no part overflows); an
// infinity or NaN goes to p[0] alone.  Exact for every x whose last bit is at
// least bf16's smallest subnormal, 2^-133.
__device__ __forceinline__ void split_bf16x3(float x, uint16_t (&p)[3]) {
    const uint32_t u = __float_as_uint(x);
    const bool finite = (u & 0x7f800000u) != 0x7f800000u;
    const bool nan = (u & 0x7fffffffu) > 0x7f800000u;
    const float r1 = finite ? x - __uint_as_float(u & 0xffff0000u) : 0.0f;
    const uint32_t u1 = __float_as_uint(r1);
    const float r2 = r1 - __uint_as_float(u1 & 0xffff0000u);
    p[0] = (uint16_t)((u >> 16) | (nan ? 0x40u : 0u));
    p[1] = (uint16_t)(u1 >> 16);
    p[2] = (uint16_t)(__float_as_uint(r2) >> 16);
}

// ---- batches of tokens ------------------------------------------------------------
constexpr int kDecodeChunk = 64;  // tokens per pass over the weights

struct DecodeBatch {
    const void *w1t, *w3t, *w2t;  // bf16 / fp8: the weights' tile images
    uint16_t *xs;                 // bf16 / fp8: x as three bf16 parts [n][3][Dpad]
    uint16_t *hs;                 // bf16 / fp8: h of each entry [n kt][3][Hpad]
    float *y;                     // [n kt][Dout]
};
// the routing of a.n tokens, one block each (wide: of 16 waves instead of 4);
// xs, when not null, receives their x as three bf16 parts
hipError_t launch_decode_route(const DecodeArgs &a, int wide, uint16_t *xs, hipStream_t s);
// the expert products of at most kDecodeChunk routed tokens; `done`, when not
// null, is recorded at the end
hipError_t launch_decode_batch(const DecodeArgs &a, const DecodeBatch &b, hipStream_t s, hipEvent_t done = nullptr);

}  // namespace moe
