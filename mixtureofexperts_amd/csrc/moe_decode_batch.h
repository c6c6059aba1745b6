// moe_decode_batch.h -- the decode caller's expert products for a batch of
// tokens (moe_ffn_forward! of n tokens, src/llama2/inference.jl:58-216),
// grouped by expert: each selected expert's matrices are read once per call
// (per up to kDecodeChunk tokens) instead of once per token that selected it.
// Part of moe_decode.hip.
//
//   decode_route_kernel : one block per token: its routing; bf16 / fp8
//        handles: x split into three bf16 parts (xs)
//   decode_up_*    : h of every (token, slot) entry of an expert
//   decode_down_*  : y of every entry
//   decode_combine_kernel : out, the entries of a token in slot order
//
// A block finds its expert and that expert's entries by itself from the
// call's indices (at most kDecodeChunk x MOE_MAX_TOPK of them): the a-th
// expert that some entry names, a = block / row tiles.  No list is built by
// a launch of its own; blocks past the last active expert end at once (the
// grid holds min(E, n k) + lsh experts).
//
// What bounds it: HBM, once the layer's matrices are a few tens of MB; below
// that the four launches.  Measured against the single-token kernels (one MoE
// call, host launches included, weights cold): 4096 / 14336, 2 of 8 experts,
// bf16: n = 1 148 -> 127 us, n = 16 1712 -> 452 to 505 us (5.6 to 6.2 TB/s), n = 64
// 5756 -> 765 us; fp8 n = 1 301 -> 78 us, n = 16 3842 -> 238 us; fp32 2048 / 1408, 6 of
// 64 experts: n = 1 100 -> 49 us, n = 64 1612 -> 433 us.
//
// bf16 / fp8 weights (MFMA): the weights are the MFMA's A operand (16 rows),
// up to 16 tokens its columns, and the fp32 activations enter exactly, as
// x = x0 + x1 + x2 (three bf16 parts of 8 significant bits each): three
// v_mfma_f32_16x16x32_bf16 per fragment, fp32 accumulation; products of bf16
// parts are exact in fp32, so nothing is dropped.  At 16 tokens the matrix
// unit needs 12 of the ~79 cycles that 1 KB of weights takes from HBM per CU.
// The weights stream from the tile images of the grouped GEMM straight into
// registers (16 rows x 64 B are contiguous there: every load instruction reads
// whole lines); the waves of a block split K and add their partial sums
// through LDS in wave order.  K ranges and row tiles depend on the layer's
// sizes only, and an MFMA column on its own token only, so a token's result
// does not depend on the batch it is in, as long as that runs here: calls of few
// tokens on small layers (decode_batched in moe_api.hip) sum in the order of
// the single-token kernels and differ in the last bits (2.5e-7 of the output's
// norm at 512 / 700).  Either order for every call of a layer costs more than it
// gives: grouped VALU kernels with a single call's sums took 75 us instead of 33
// for 64 tokens of 512 / 1376 in bf16 and 293 instead of 86 at 1024 / 4096, and
// one token grouped 19 instead of 10 and 30 instead of 21.
//
// fp32 weights (VALU): the arithmetic of decode_up_kernel / decode_down_kernel
// (one wave per row, chunks of 4 per lane in order, a fixed butterfly), each
// weight register used for up to 8 tokens: bitwise the results of single
// calls.
#pragma once
#include <algorithm>
#include <type_traits>

#include "moe_decode.h"
#include "moe_internal.h"

namespace moe {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// ---- the block's expert and its entries ------------------------------------------
struct DecodeGroupLds {
    int ids[kDecodeChunk * MOE_MAX_TOPK];   // the chunk's indices (1-based; 0: none)
    uint32_t act[MOE_MAX_EXPERTS / 32];     // experts that some entry names
    int list[kDecodeChunk];                 // the expert's entries (token * kt + slot), tokens ascending
};

// Expert of rank `ai` among the active ones (-1: fewer are active) and its
// entries; m of them.  All threads of the block call it (two barriers).
__device__ __forceinline__ int decode_group(const DecodeArgs &a, int ai, DecodeGroupLds &L, int &m) {
    const int ne = a.n * a.kt, Et = a.E + a.lsh, nw = (Et + 31) >> 5;
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid < MOE_MAX_EXPERTS / 32) L.act[tid] = 0u;
    __syncthreads();
    for (int i = tid; i < ne; i += blockDim.x) {
        const int id = a.idx[i];
        const bool ok = id >= 1 && id <= Et;
        L.ids[i] = ok ? id : 0;
        if (ok) atomicOr(&L.act[(id - 1) >> 5], 1u << ((id - 1) & 31));
    }
    __syncthreads();
    // every wave finds the expert on its own (same result): lane w holds word w
    const uint32_t word = lane < nw ? L.act[lane] : 0u;
    int before = 0;  // active experts in the words before this lane's
    for (int w = 0; w < nw; ++w) {
        const int c = __popc((uint32_t)__builtin_amdgcn_readlane((int)word, w));
        before += w < lane ? c : 0;
    }
    const unsigned long long here = __ballot(lane < nw && before <= ai && ai < before + __popc(word));
    if (!here) {
        m = 0;
        return -1;
    }
    const int wl = __builtin_ctzll(here);
    uint32_t bits = (uint32_t)__builtin_amdgcn_readlane((int)word, wl);
    for (int r = ai - __builtin_amdgcn_readlane(before, wl); r > 0; --r) bits &= bits - 1;
    const int e = 32 * wl + __builtin_ctz(bits);
    // a token names an expert at most once: lane t looks for it in token t's slots
    int slot = -1;
    if (lane < a.n)
        for (int s = 0; s < a.kt; ++s)
            if (L.ids[lane * a.kt + s] == e + 1) slot = s;
    const unsigned long long mask = __ballot(slot >= 0);
    m = __popcll(mask);
    if (slot >= 0 && tid < 64) L.list[__popcll(mask & ((1ull << lane) - 1))] = lane * a.kt + slot;
    __syncthreads();
    return e;
}

// ---- bf16 / fp8 weights -------------------------------------------------------------
// One wave's share of C[rows][tokens] += W[rows][K range] X[tokens][K range]^T:
// NM matrices x 2 row tiles of 16 rows, NT column tiles of 16 tokens, K steps
// [s0, s1) of KS K values (32 bf16, 64 fp8).  wsrc[m]: lane address of row tile
// 0 of matrix m at step 0; row tile 1 at + wrow bytes, step s at + s * wstep.
// xsrc[j]: lane address of column tile j's tokens at step 0, part p at
// + p * xpart elements.  Steps run in batches of P: a batch's loads are all
// issued before the previous batch's products, so P to 2 P steps are in
// flight per wave.  The products with x0 are summed from zero over kAccK K
// values and then added to the running sum (one addition at its magnitude per
// 128 K), those with the small parts in a sum of their own, added last: the
// error against 64 bits stays at or below that of one FMA chain per lane
// (every product added to one running sum had twice that at K = 4096).
constexpr int kAccK = 128;

template <int WF8, int NM, int NT, int P>
__device__ __forceinline__ void stream_rows(const uint8_t *const (&wsrc)[NM], long long wrow, long long wstep,
                                            const uint16_t *const (&xsrc)[NT], long long xpart, int s0, int s1,
                                            f32x4_t (&acc)[NM][2][NT]) {
    constexpr int KS = WF8 ? 64 : 32;
    constexpr int G = kAccK / KS;    // steps per group
    constexpr int XL = WF8 ? 2 : 1;  // 8-value fragments per lane, part and step
    u32x4_t wc[P][NM][2], wn[P][NM][2];
    bf16x8_t xc[P][NT][3][XL], xn[P][NT][3][XL];
    f32x4_t grp[NM][2][NT], low[NM][2][NT];
    auto load = [&](int s, u32x4_t (&w)[P][NM][2], bf16x8_t (&x)[P][NT][3][XL]) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int st = min(s + p, s1 - 1);  // past the range: a step already read, not used
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int i = 0; i < 2; ++i) w[p][m][i] = *(const u32x4_t *)(wsrc[m] + i * wrow + st * wstep);
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < 3; ++q)
#pragma unroll
                    for (int u = 0; u < XL; ++u)
                        x[p][j][q][u] = *(const bf16x8_t *)(xsrc[j] + q * xpart + (long long)st * KS + 8 * u);
        }
    };
    auto clear = [&](f32x4_t (&c)[NM][2][NT]) {
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) c[m][i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    };
    clear(acc);
    clear(grp);
    clear(low);
    if (s0 >= s1) return;
    load(s0, wc, xc);
    for (int s = s0; s < s1; s += P) {
        load(s + P, wn, xn);
#pragma unroll
        for (int p = 0; p < P; ++p) {
            if (s + p >= s1) break;  // wave-uniform
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int u = 0; u < XL; ++u) {
                        bf16x8_t wf;
                        if constexpr (WF8) wf = widen_fp8x8(wc[p][m][i][2 * u], wc[p][m][i][2 * u + 1]);
                        else __builtin_memcpy(&wf, &wc[p][m][i], 16);
#pragma unroll
                        for (int j = 0; j < NT; ++j) {
                            low[m][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xc[p][j][2][u], low[m][i][j], 0, 0, 0);
                            low[m][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xc[p][j][1][u], low[m][i][j], 0, 0, 0);
                            grp[m][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xc[p][j][0][u], grp[m][i][j], 0, 0, 0);
                        }
                    }
            if ((s + p - s0) % G == G - 1 || s + p == s1 - 1) {  // the group's end (wave-uniform)
#pragma unroll
                for (int m = 0; m < NM; ++m)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < NT; ++j)
#pragma unroll
                            for (int v = 0; v < 4; ++v) acc[m][i][j][v] = acc[m][i][j][v] + grp[m][i][j][v];
                clear(grp);
            }
        }
#pragma unroll
        for (int p = 0; p < P; ++p) {
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int i = 0; i < 2; ++i) wc[p][m][i] = wn[p][m][i];
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < 3; ++q)
#pragma unroll
                    for (int u = 0; u < XL; ++u) xc[p][j][q][u] = xn[p][j][q][u];
        }
    }
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[m][i][j][v] = acc[m][i][j][v] + low[m][i][j][v];
}

// Lane address of rows r0 .. r0 + 15 (r0 a multiple of 16) in a tile image of
// RB-row blocks and KTT 32-wide stages, at step 0.  bf16: lane (r, q) = (l %
// 16, l / 16) takes 16-byte chunk q of its row's stage; fp8 (a step is two
// stages): chunk q % 2 of stage q / 2.
template <int WF8, int RB>
__device__ __forceinline__ const uint8_t *image_lane(const void *img, long long estride, int e, int r0, long long KTT,
                                                     int lane) {
    constexpr int BROWB = WF8 ? 32 : 64;
    const int r = lane & 15, q = lane >> 4;
    const long long nb = r0 / RB, rin = r0 - nb * RB + r;
    const long long st = WF8 ? (q >> 1) : 0;
    const int pos = WF8 ? ((q & 1) ^ ((r >> 3) & 1)) : (q ^ ((r >> 2) & 3));
    return (const uint8_t *)img + (long long)e * estride * (WF8 ? 1 : 2) + ((nb * KTT + st) * RB + rin) * BROWB +
           pos * 16;
}

constexpr int kDecRows = 32;  // rows of a block's row tile (two MFMA row tiles)

// A block's row tile of NM matrices against entries j0 .. j0 + 16 NT - 1 of
// L.list: each wave's sums over its K range to red, [wave][matrix][row
// tile][column tile][lane] of f32x4.
template <int WF8, int NM, int RB, int NT, int P>
__device__ __forceinline__ void decode_tile(const void *const (&img)[NM], long long estride, int e, int r0, int Kpad,
                                            const uint16_t *xs, bool by_entry, int kt, const DecodeGroupLds &L, int m,
                                            int j0, int nwave, f32x4_t *red) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long long KTT = Kpad / 32;
    const int steps = Kpad / (WF8 ? 64 : 32);
    const int s0 = (int)((long long)steps * w / nwave), s1 = (int)((long long)steps * (w + 1) / nwave);
    const uint8_t *wsrc[NM];
#pragma unroll
    for (int q = 0; q < NM; ++q) wsrc[q] = image_lane<WF8, RB>(img[q], estride, e, r0, KTT, lane);
    constexpr long long BROWB = WF8 ? 32 : 64;
    const uint16_t *xsrc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int ent = L.list[min(j0 + 16 * j + (lane & 15), m - 1)];  // columns past m repeat the last entry
        const long long row = by_entry ? ent : ent / kt;
        xsrc[j] = xs + row * 3 * Kpad + (lane >> 4) * (WF8 ? 16 : 8);
    }
    f32x4_t acc[NM][2][NT];
    stream_rows<WF8, NM, NT, P>(wsrc, 16 * BROWB, (WF8 ? 2 : 1) * RB * BROWB, xsrc, Kpad, s0, s1, acc);
#pragma unroll
    for (int q = 0; q < NM; ++q)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) red[(((w * NM + q) * 2 + i) * NT + j) * 64 + lane] = acc[q][i][j];
}

// Sum over the waves, in wave order, of row r (0 .. 31) of matrix q, column c.
template <int NM, int NT>
__device__ __forceinline__ float wave_total(const f32x4_t *red, int nwave, int q, int r, int c) {
    const int i = r >> 4, j = c >> 4, l = (c & 15) + 16 * ((r & 15) >> 2);
    const float *p = (const float *)(red + ((q * 2 + i) * NT + j) * 64 + l) + (r & 3);
    float s = p[0];
    for (int w = 1; w < nwave; ++w) s = s + p[(long long)w * NM * 2 * NT * 64 * 4];
    return s;
}

// A bf16 weight row with 4 nch fp32 values (x4(c): chunk c of four), by a whole
// wave in a single call's arithmetic: an output whose sum is not finite is
// recomputed by it.  An infinite weight gives NaN with the zero parts of a
// finite x (and infinities of both signs with parts of both signs), where the
// product itself is an infinity.  One infinity or NaN in x makes every row of
// its token's experts such an output, in the same launches as the other
// tokens, so the row is read in coalesced chunks, eight per lane in flight, up
// to the first batch that makes it NaN.  Sixteen tokens on a 4096 / 14336
// layer, us: 515; one of them with a NaN 620, with an infinity 710 (3530 and
// 4670 by one thread per row and one load per value).
template <typename X4>
__device__ __forceinline__ float wave_row_bf16(const uint16_t *w, int nch, X4 x4) {
    const int lane = threadIdx.x & 63;
    float s = 0.0f;
    for (int c0 = 0; c0 < nch; c0 += 64 * 8) {
        float4 wv[8], xv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int c = min(c0 + 64 * u + lane, nch - 1);
            wv[u] = load_w4<WT_BF16>(w, 4 * c);
            xv[u] = x4(c);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const bool v = c0 + 64 * u + lane < nch;
            s = dot4_acc(s, zero_unless(v, wv[u]), zero_unless(v, xv[u]));
        }
        if (__any(s != s)) break;  // the row's sum is NaN
    }
    return wave_sum(s);
}

constexpr int kUpWaves = 4;
constexpr int kBatchNT = 2;  // column tiles of 16 entries per pass over the weights

// h of 32 rows for the entries of one expert, as three bf16 parts.
template <int WF8, int NT, int P>
__device__ __forceinline__ void up_tile(const DecodeArgs &a, const DecodeBatch &b, int e, int r0,
                                        const DecodeGroupLds &L, int m, int j0, f32x4_t *red) {
#pragma clang fp contract(off)
    const void *img[2] = {b.w1t, b.w3t};
    decode_tile<WF8, 2, kNPadGated, NT, P>(img, a.w1_stride, e, r0, a.Dpad, b.xs, false, a.kt, L, m, j0, kUpWaves, red);
    __syncthreads();
    // thread: column c, rows 2 rr, 2 rr + 1 (one 4-byte store per part); whole
    // waves run each pass, for wave_row_bf16
    const int lane = threadIdx.x & 63, nu = 16 * min(m - j0, 16 * NT);
    for (int u0 = threadIdx.x - lane; u0 < nu; u0 += 64 * kUpWaves) {
        const bool on = u0 + lane < nu;
        const int u = on ? u0 + lane : u0, c = u >> 4, rr = (u & 15) * 2;
        uint32_t part[3] = {0u, 0u, 0u};
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int r = rr + k;
            float g = wave_total<2, NT>(red, kUpWaves, 0, r, c);
            float up = wave_total<2, NT>(red, kUpWaves, 1, r, c);
            if constexpr (WF8) {
                g = g * a.s1[(long long)e * a.Hpad + r0 + r];
                up = up * a.s3[(long long)e * a.Hpad + r0 + r];
            } else {
                unsigned long long bad =
                    __ballot(on && r0 + r < a.H && !(__builtin_isfinite(g) && __builtin_isfinite(up)));
                while (bad) {
                    const int l = __builtin_ctzll(bad), ub = u0 + l, rb = r0 + (ub & 15) * 2 + k;
                    bad &= bad - 1;
                    const float4 *x = (const float4 *)(a.x + (long long)(L.list[j0 + (ub >> 4)] / a.kt) * a.D);
                    const long long wo = (long long)e * a.w1_stride + (long long)rb * a.Dpad;
                    auto x4 = [&](int i) { return x[i]; };
                    const float gb = wave_row_bf16((const uint16_t *)a.w1 + wo, a.D >> 2, x4);
                    const float vb = wave_row_bf16((const uint16_t *)a.w3 + wo, a.D >> 2, x4);
                    g = lane == l ? gb : g;
                    up = lane == l ? vb : up;
                }
            }
            // pad rows: 0 whatever x holds
            const float h = r0 + r < a.H ? (g * (1.0f / (1.0f + expf(-g)))) * up : 0.0f;
            uint16_t p3[3];
            split_bf16x3(h, p3);
#pragma unroll
            for (int q = 0; q < 3; ++q) part[q] |= (uint32_t)p3[q] << (16 * k);
        }
        if (!on) continue;
        uint16_t *dst = b.hs + (long long)L.list[j0 + c] * 3 * a.Hpad + r0 + rr;
#pragma unroll
        for (int q = 0; q < 3; ++q) *(uint32_t *)(dst + (long long)q * a.Hpad) = part[q];
    }
}

// y of 32 rows for the entries of one expert.
template <int WF8, int NW, int NT, int P>
__device__ __forceinline__ void down_tile(const DecodeArgs &a, const DecodeBatch &b, int e, int r0,
                                          const DecodeGroupLds &L, int m, int j0, f32x4_t *red) {
#pragma clang fp contract(off)
    const void *img[1] = {b.w2t};
    decode_tile<WF8, 1, kNPad, NT, P>(img, a.w2_stride, e, r0, a.Hpad, b.hs, true, a.kt, L, m, j0, NW, red);
    __syncthreads();
    const int lane = threadIdx.x & 63, nu = 32 * min(m - j0, 16 * NT);
    for (int u0 = threadIdx.x - lane; u0 < nu; u0 += 64 * NW) {  // whole waves, for wave_row_bf16
        const int u = min(u0 + lane, nu - 1), c = u >> 5, r = u & 31;
        const bool on = u0 + lane < nu && r0 + r < a.Dout;
        float y = wave_total<1, NT>(red, NW, 0, r, c);
        if constexpr (WF8) {
            y = y * a.s2[(long long)e * a.Dout_npad + r0 + r];
        } else {
            unsigned long long bad = __ballot(on && !__builtin_isfinite(y));
            while (bad) {
                const int l = __builtin_ctzll(bad), ub = u0 + l;
                bad &= bad - 1;
                const uint16_t *h = b.hs + (long long)L.list[j0 + (ub >> 5)] * 3 * a.Hpad;
                auto h4 = [&](int i) {
                    const float4 p0 = load_w4<WT_BF16>(h, 4 * i), p1 = load_w4<WT_BF16>(h, a.Hpad + 4 * i),
                                 p2 = load_w4<WT_BF16>(h, 2 * a.Hpad + 4 * i);
                    return make_float4((p2.x + p1.x) + p0.x, (p2.y + p1.y) + p0.y, (p2.z + p1.z) + p0.z, (p2.w + p1.w) + p0.w);
                };
                const float yb = wave_row_bf16((const uint16_t *)a.w2 + (long long)e * a.w2_stride +
                                                   (long long)(r0 + (ub & 31)) * a.Hpad, a.Hpad >> 2, h4);
                y = lane == l ? yb : y;
            }
        }
        if (on) b.y[(long long)L.list[j0 + c] * a.Dout + r0 + r] = y;
    }
}

template <int WF8>
__global__ __launch_bounds__(64 * kUpWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void decode_up_mfma_kernel(
    DecodeArgs a, DecodeBatch b) {
    __shared__ DecodeGroupLds L;
    __shared__ f32x4_t red[kUpWaves * 2 * 2 * kBatchNT * 64];
    const int nt = a.Hpad / kDecRows;
    const int ai = blockIdx.x / nt, r0 = (blockIdx.x - ai * nt) * kDecRows;
    int m;
    const int e = decode_group(a, ai, L, m);
    if (e < 0) return;
    for (int j0 = 0; j0 < m; j0 += 16 * kBatchNT) {
        if (j0 > 0) __syncthreads();  // red is read
        if (m - j0 <= 16) up_tile<WF8, 1, 2>(a, b, e, r0, L, m, j0, red);
        else up_tile<WF8, 2, 1>(a, b, e, r0, L, m, j0, red);
    }
}

template <int WF8, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2))) void decode_down_mfma_kernel(
    DecodeArgs a, DecodeBatch b) {
    __shared__ DecodeGroupLds L;
    __shared__ f32x4_t red[NW * 2 * kBatchNT * 64];
    const int nt = (a.Dout + kDecRows - 1) / kDecRows;
    const int ai = blockIdx.x / nt, r0 = (blockIdx.x - ai * nt) * kDecRows;
    int m;
    const int e = decode_group(a, ai, L, m);
    if (e < 0) return;
    for (int j0 = 0; j0 < m; j0 += 16 * kBatchNT) {
        if (j0 > 0) __syncthreads();  // red is read
        if (m - j0 <= 16) down_tile<WF8, NW, 1, WF8 ? 2 : 4>(a, b, e, r0, L, m, j0, red);
        else down_tile<WF8, NW, 2, WF8 ? 1 : 2>(a, b, e, r0, L, m, j0, red);
    }
}

// ---- fp32 weights ----------------------------------------------------------------------
// Rows j0, j0 + 1 of W1 and W3 of expert e for entries [c0, c0 + TM) of the
// list (past m: the last one again, not stored): decode_up_units' arithmetic.
template <int TM>
__device__ __forceinline__ void up_rows_f32(const DecodeArgs &a, int e, int j0, const DecodeGroupLds &L, int m, int c0) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const int nch = a.D >> 2;
    const float *w1 = (const float *)a.w1 + (long long)e * a.w1_stride + (long long)j0 * a.Dpad;
    const float *w3 = (const float *)a.w3 + (long long)e * a.w1_stride + (long long)j0 * a.Dpad;
    const float4 *x4[TM];
#pragma unroll
    for (int q = 0; q < TM; ++q) x4[q] = (const float4 *)(a.x + (long long)(L.list[min(c0 + q, m - 1)] / a.kt) * a.D);
    float g[TM][2], up[TM][2];
#pragma unroll
    for (int q = 0; q < TM; ++q) g[q][0] = g[q][1] = up[q][0] = up[q][1] = 0.0f;
    // chunks k0 + lane, k0 + 64 + lane; TAIL: those past nch enter as zeros
    auto chunks = [&](int k0, auto TAIL) {
        const int c = k0 + lane;
        const bool va = !TAIL || c < nch, vb = !TAIL || c + 64 < nch;
        const int ca = TAIL ? min(c, nch - 1) : c, cb = TAIL ? min(c + 64, nch - 1) : c + 64;
        float4 ga[2], gb[2], ua[2], ub[2], xa[TM], xb[TM];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            ga[r] = *(const float4 *)(w1 + (long long)r * a.Dpad + 4 * ca);
            gb[r] = *(const float4 *)(w1 + (long long)r * a.Dpad + 4 * cb);
            ua[r] = *(const float4 *)(w3 + (long long)r * a.Dpad + 4 * ca);
            ub[r] = *(const float4 *)(w3 + (long long)r * a.Dpad + 4 * cb);
        }
#pragma unroll
        for (int q = 0; q < TM; ++q) {
            xa[q] = zero_unless(va, x4[q][ca]);
            xb[q] = zero_unless(vb, x4[q][cb]);
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const float4 wga = zero_unless(va, ga[r]), wua = zero_unless(va, ua[r]);
            const float4 wgb = zero_unless(vb, gb[r]), wub = zero_unless(vb, ub[r]);
#pragma unroll
            for (int q = 0; q < TM; ++q) {
                g[q][r] = dot4_acc(g[q][r], wga, xa[q]);
                up[q][r] = dot4_acc(up[q][r], wua, xa[q]);
                g[q][r] = dot4_acc(g[q][r], wgb, xb[q]);
                up[q][r] = dot4_acc(up[q][r], wub, xb[q]);
            }
        }
    };
    int k0 = 0;
    for (; k0 + 128 <= nch; k0 += 128) chunks(k0, std::false_type{});
    if (k0 < nch) chunks(k0, std::true_type{});
#pragma unroll
    for (int q = 0; q < TM; ++q)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const float gs = wave_sum(g[q][r]), us = wave_sum(up[q][r]);
            if (lane == 0 && c0 + q < m && j0 + r < a.Hpad)
                a.h[(long long)L.list[c0 + q] * a.Hpad + j0 + r] =
                    j0 + r < a.H ? (gs * (1.0f / (1.0f + expf(-gs)))) * us : 0.0f;
        }
}

// Rows i0 .. i0 + R - 1 of W2 of expert e for entries [c0, c0 + TM):
// decode_down_kernel's arithmetic.  (That kernel also adds the zero products
// of its batch's chunks past the row's end: a sum that starts at +0 is never
// -0, so they change no bit and are left out here.)  R rows share the h
// reads: at 8 entries one row per wave needs nine 1 KB reads through the L1
// per KB of weights, four rows three.
template <int TM, int R, int U>
__device__ __forceinline__ void down_rows_f32(const DecodeArgs &a, const DecodeBatch &b, int e, int i0,
                                              const DecodeGroupLds &L, int m, int c0) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    const int nch = a.Hpad >> 2;
    const float4 *w[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
        w[r] = (const float4 *)((const float *)a.w2 + (long long)e * a.w2_stride +
                                (long long)min(i0 + r, a.Dout - 1) * a.Hpad);
    const float4 *h4[TM];
#pragma unroll
    for (int q = 0; q < TM; ++q) h4[q] = (const float4 *)(a.h + (long long)L.list[min(c0 + q, m - 1)] * a.Hpad);
    float y[TM][R];
#pragma unroll
    for (int q = 0; q < TM; ++q)
#pragma unroll
        for (int r = 0; r < R; ++r) y[q][r] = 0.0f;
    // U chunks per lane from k0; TAIL: those past nch enter as zeros
    auto chunks = [&](int k0, auto TAIL) {
        float4 wv[U][R], hv[U][TM];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = TAIL ? min(k0 + u * 64 + lane, nch - 1) : k0 + u * 64 + lane;
#pragma unroll
            for (int r = 0; r < R; ++r) wv[u][r] = w[r][c];
#pragma unroll
            for (int q = 0; q < TM; ++q) hv[u][q] = h4[q][c];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool v = !TAIL || k0 + u * 64 + lane < nch;
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int q = 0; q < TM; ++q)
                    y[q][r] = dot4_acc(y[q][r], zero_unless(v, wv[u][r]), zero_unless(v, hv[u][q]));
        }
    };
    int k0 = 0;
    for (; k0 + 64 * U <= nch; k0 += 64 * U) chunks(k0, std::false_type{});
    if (k0 < nch) chunks(k0, std::true_type{});
#pragma unroll
    for (int q = 0; q < TM; ++q)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float s = wave_sum(y[q][r]);
            if (lane == 0 && c0 + q < m && i0 + r < a.Dout) b.y[(long long)L.list[c0 + q] * a.Dout + i0 + r] = s;
        }
}

constexpr int kUpRowsF32 = 8;  // rows of a block: 4 waves x 2

__global__ __launch_bounds__(256) void decode_up_f32_kernel(DecodeArgs a, DecodeBatch b) {
    __shared__ DecodeGroupLds L;
    const int nt = (a.Hpad + kUpRowsF32 - 1) / kUpRowsF32;
    const int ai = blockIdx.x / nt, j0 = (blockIdx.x - ai * nt) * kUpRowsF32 + 2 * (threadIdx.x >> 6);
    int m;
    const int e = decode_group(a, ai, L, m);
    if (e < 0) return;
    if (m == 1) up_rows_f32<1>(a, e, j0, L, m, 0);
    else if (m == 2) up_rows_f32<2>(a, e, j0, L, m, 0);
    else if (m <= 4) up_rows_f32<4>(a, e, j0, L, m, 0);
    else
        for (int c0 = 0; c0 < m; c0 += 8) up_rows_f32<8>(a, e, j0, L, m, c0);
}

template <int R>
__global__ __launch_bounds__(256) void decode_down_f32_kernel(DecodeArgs a, DecodeBatch b) {
    __shared__ DecodeGroupLds L;
    const int nt = (a.Dout + 4 * R - 1) / (4 * R);
    const int ai = blockIdx.x / nt, i0 = ((blockIdx.x - ai * nt) * 4 + (threadIdx.x >> 6)) * R;
    int m;
    const int e = decode_group(a, ai, L, m);
    if (e < 0 || i0 >= a.Dout) return;
    if (m == 1) down_rows_f32<1, R, R == 1 ? 8 : 2>(a, b, e, i0, L, m, 0);
    else if (m == 2) down_rows_f32<2, R, R == 1 ? 4 : 2>(a, b, e, i0, L, m, 0);
    else if (m <= 4) down_rows_f32<4, R, 2>(a, b, e, i0, L, m, 0);
    else
        for (int c0 = 0; c0 < m; c0 += 8) down_rows_f32<8, R, R == 1 ? 2 : 1>(a, b, e, i0, L, m, c0);
}

// ---- out: a token's entries in slot order (decode_down_kernel's end) --------------------
__global__ __launch_bounds__(256) void decode_combine_kernel(DecodeArgs a, DecodeBatch b) {
#pragma clang fp contract(off)
    const int t = blockIdx.x, i = blockIdx.y * 256 + threadIdx.x;
    if (i >= a.Dout) return;
    const float sw = a.lsh > 0 ? 1.0f / (float)a.lsh : 0.0f;
    float yv[MOE_MAX_TOPK];
#pragma unroll
    for (int s = 0; s < MOE_MAX_TOPK; ++s)
        if (s < a.kt) yv[s] = b.y[((long long)t * a.kt + s) * a.Dout + i];
    float acc = 0.0f, sh = 0.0f;
#pragma unroll
    for (int s = 0; s < MOE_MAX_TOPK; ++s)
        if (s < a.kt) {
            const int id = a.idx[(long long)t * a.kt + s];
            if (id < 1 || id > a.E + a.lsh) continue;
            if (s < a.lsh) sh = sh + sw * yv[s];
            else acc = acc + a.gates[(long long)t * a.kt + s] * yv[s];
        }
    if (a.lsh > 0) acc = 0.5f * sh + 0.5f * acc;
    a.out[(long long)t * a.Dout + i] = acc;
}

// One chunk (a.n <= kDecodeChunk tokens, routed by launch_decode_route).
hipError_t launch_decode_batch(const DecodeArgs &a, const DecodeBatch &b, hipStream_t s, hipEvent_t done) {
    if (a.n < 1 || a.n > kDecodeChunk || !b.y) return hipErrorInvalidValue;
    const unsigned na = (unsigned)(std::min(a.E, a.n * a.k) + a.lsh);  // at most this many active experts
    hipError_t e = hipSuccess;
    if (a.wt == WT_F32) {
        hipLaunchKernelGGL(decode_up_f32_kernel, dim3(na * ((a.Hpad + kUpRowsF32 - 1) / kUpRowsF32)), dim3(256), 0, s, a, b);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        // four rows per wave where that still leaves about four waves per SIMD
        if ((long long)na * a.Dout >= 16 * 1024)
            hipLaunchKernelGGL(decode_down_f32_kernel<4>, dim3(na * ((a.Dout + 15) / 16)), dim3(256), 0, s, a, b);
        else
            hipLaunchKernelGGL(decode_down_f32_kernel<1>, dim3(na * ((a.Dout + 3) / 4)), dim3(256), 0, s, a, b);
    } else {
        if (!b.xs || !b.hs || !b.w1t || !b.w3t || !b.w2t || a.Dpad % 64 || a.Hpad % 64) return hipErrorInvalidValue;
        const dim3 gu(na * (unsigned)(a.Hpad / kDecRows)), gd(na * (unsigned)((a.Dout + kDecRows - 1) / kDecRows));
        if (a.wt == WT_FP8) hipLaunchKernelGGL(decode_up_mfma_kernel<1>, gu, dim3(64 * kUpWaves), 0, s, a, b);
        else hipLaunchKernelGGL(decode_up_mfma_kernel<0>, gu, dim3(64 * kUpWaves), 0, s, a, b);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        // K ranges of the down tiles: eight waves where each still has 16
        // steps or more, else four
        const bool deep = a.Hpad >= 8 * 16 * (a.wt == WT_FP8 ? 64 : 32);
        if (a.wt == WT_FP8) {
            if (deep) hipLaunchKernelGGL((decode_down_mfma_kernel<1, 8>), gd, dim3(512), 0, s, a, b);
            else hipLaunchKernelGGL((decode_down_mfma_kernel<1, 4>), gd, dim3(256), 0, s, a, b);
        } else {
            if (deep) hipLaunchKernelGGL((decode_down_mfma_kernel<0, 8>), gd, dim3(512), 0, s, a, b);
            else hipLaunchKernelGGL((decode_down_mfma_kernel<0, 4>), gd, dim3(256), 0, s, a, b);
        }
    }
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid(a.n, (a.Dout + 255) / 256);
    hipExtLaunchKernelGGL(decode_combine_kernel, grid, dim3(256), 0, s, nullptr, done, 0, a, b);
    return hipGetLastError();
}

}  // namespace moe
