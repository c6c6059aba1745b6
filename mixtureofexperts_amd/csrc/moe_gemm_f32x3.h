// moe_gemm_f32x3.h -- the fp32 grouped GEMM on the bf16 matrix unit, for expert
// segments of many rows.  Part of moe_gemm.hip.
//
// An fp32 value of 2^-110 or more is the sum of three bf16 ones (8 significant
// bits each, rounded to nearest: |x1| <= 2^-9 |x|, |x2| <= 2^-17 |x|), and an
// fp32 product to fp32 accuracy the sum of the six products of parts i + j <=
// 2: the three left out are below 2^-25 of it, random in sign, under the
// rounding of the fp32 sum.  Smaller values keep their bits down to 2^-133,
// bf16's smallest (an error of 2^-22 at 2^-112, 2^-14 at 2^-120), so sums below
// 2^-90 are redone too.  Per 32 x 32 outputs and 16 K, six bf16 products take 192 cycles of the matrix unit, eight
// v_mfma_f32_32x32x2_f32 512; the running sums stay fp32.
//
// What bounds it: the work besides the MFMAs (splits, LDS), which keep the
// matrix unit busy 64 to 67 % of cycles at 1.8 GHz at 4096 / 14336, 43 to 54 % at
// 2.2 to 2.3 GHz at 768 / 3072 with its 24 and 96 stages per tile.  Against
// grouped_gemm_kernel (whole layer forward, 8 experts, top-2, 4096 tokens):
// 4096 / 14336 gated 25.4 -> 14.2 ms, 768 / 3072 standard 722 -> 428 us, 1024 / 4096
// gated 1861 -> 1040 us; error against 64 bits 2.8e-6 -> 2.4e-6, 1.13e-6 ->
// 0.99e-6, 1.44e-6 -> 1.24e-6.  Two 128 x 128 workgroups per CU instead of one
// took 4 % longer, 32x32x16 instead of 16x16x32 MFMAs 5 %, and splitting the last
// round's tiles into K ranges gained nothing (467 and 463 us).
//
// Tile 128 rows x 256 weight rows (gated: 128 of W1 and the same 128 of W3), 8
// waves as 2 (rows) x 4 (columns), two per SIMD, each 64 x 64.  A stage is 32
// K: every thread loads 8 K values of three rows (one of A, two of the
// weights) two stages ahead, splits them one stage ahead and writes them to
// the other of two LDS buffers (72 KB each), so the split's vector
// instructions, the LDS writes and the reads of the next half's fragments run
// between the MFMAs and there is one barrier per stage (192 MFMAs per SIMD).
// Splitting in the kernel repeats it for every tile that reads an operand, but
// keeps weights, xp and h at 4 bytes in memory and in L2.
//
// LDS rows are 64 B (32 bf16 of one part), 16-byte chunk c of row r at c ^
// ((r >> 2) & 3), as in the bf16 kernel.
//
// Infinities, NaN and values that round up to an infinity: their parts give
// NaN or infinite sums, and a wave that holds such a sum, or one that is not
// 0 and below 2^-90, takes it from fp32 MFMAs over the fp32 operands (redo).
//
// STAGE_SUMS: the six products of a stage start from zero, the smallest first,
// and are added to the running sum with one rounded addition.  An MFMA adds its
// products to its accumulator in several steps, each rounded at the
// accumulator's size, without a bias: a chain of 4096 random bf16 products has
// an error of 3.9e-7 in a running accumulator, 2.1e-7 in sums of 32 from zero
// and one addition each, 6.0e-7 with v_mfma_f32_16x16x4_f32 (the mean along the
// sum's sign below 1e-8 in all).  Six instructions of the running size per 32 K
// cost more accuracy at small K than grouped_gemm_kernel's 16 smaller ones:
// error against 64 bits at 300 / 300 gated 2.5e-7 there, 5.0e-7 with running
// sums, 1.6e-7 with stage sums; 64 / 64 2.0e-7, 2.9e-7, 1.0e-7; 128 / 256 standard
// 1.8e-7, 3.4e-7, 1.2e-7; and no more from 512 on: 520 / 2731 gated 8.2e-7, 5.3e-7
// with running sums in the up GEMM; 768 / 3072 standard 11.3e-7, 9.9e-7, 2.6e-7.
// The additions wait for the matrix unit and cost 6 % where it is the bound
// (768 / 3072 standard, 4096 tokens: 427 -> 453 us), 0 to 2 % elsewhere, so the running sums
// stay for large calls of large K (launch_f32x3).
//
// K split (g.ksplit = S > 1): as in grouped_gemm_kernel, blocks of BM x 256
// floats.

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// Eight fp32 -> three chunks of eight bf16.
__device__ __forceinline__ void split8(const f32x4_t &a, const f32x4_t &b, u32x4_t (&p)[3]) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float x = i < 2 ? a[2 * i] : b[2 * i - 4], y = i < 2 ? a[2 * i + 1] : b[2 * i - 3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const bf16x2_t h = {(__bf16)x, (__bf16)y};
            uint32_t u;
            __builtin_memcpy(&u, &h, 4);
            p[q][i] = u;
            if (q < 2) {
                x = x - __uint_as_float(u << 16);
                y = y - __uint_as_float(u & 0xffff0000u);
            }
        }
    }
}

template <int MODE, bool STAGE_SUMS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void grouped_gemm_f32x3_kernel(GemmArgs g) {
    constexpr int NB = (MODE == MODE_GATED_UP) ? 2 : 1;
    constexpr int BM = kGemmBM, BR = 256;         // tile rows, weight rows
    constexpr int BN = BR / NB;                   // output columns
    constexpr int ROWS = BM + BR;                 // LDS rows of a part
    constexpr int PART = ROWS * 64, STAGE = 3 * PART;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * STAGE];

    // tile order as in grouped_gemm_kernel
    const int L = blockIdx.x;
    const int per = gridDim.x >> 3;
    const int S = g.ksplit;
    const int id0 = (L & 7) * per + (L >> 3);
    const int ks = id0 % S, id = id0 / S;
    const int mt = id % g.m_tiles_grid;
    const int nt = id / g.m_tiles_grid;
    if (nt >= g.n_tiles) return;
    if (mt >= g.num_tiles[0]) return;
    const int2 te = g.tiles[mt];
    const int e = te.x, m0 = te.y;
    const int rows = min(BM, g.counts[e] - m0);
    const long long arow0 = (long long)g.offsets[e] + m0;
    const int n0 = nt * BN;

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = w & 1, wn = w >> 1;
    const int q4 = lane >> 4, r16 = lane & 15;

    // this thread's three rows: row tid / 4 of A, of the first and of the
    // second 128 weight rows; K values 8 (tid % 4) .. + 8 of each stage
    const int tr = tid >> 2, tc = tid & 3;
    const float *A = (const float *)g.A;
    const float *B0 = (const float *)g.B0 + (long long)e * g.b_stride + (long long)n0 * g.ldb;
    const float *B1 = NB == 2 ? (const float *)g.B1 + (long long)e * g.b_stride + (long long)n0 * g.ldb
                              : B0 + 128 * g.ldb;
    const float *src[3] = {A + (arow0 + min(tr, rows - 1)) * g.lda + 8 * tc, B0 + (long long)tr * g.ldb + 8 * tc,
                           B1 + (long long)tr * g.ldb + 8 * tc};
    // (rows tr, 128 + tr and 256 + tr of a part share their swizzle)
    const int wofs = tr * 64 + ((tc ^ ((tr >> 2) & 3)) << 4);
    f32x4_t ra[3][2];
    auto load = [&](int i, int kt) {
        ra[i][0] = *(const f32x4_t *)(src[i] + (long long)kt * 32);
        ra[i][1] = *(const f32x4_t *)(src[i] + (long long)kt * 32 + 4);
    };
    auto split_store = [&](int buf, int i) {
        u32x4_t p[3];
        split8(ra[i][0], ra[i][1], p);
#pragma unroll
        for (int q = 0; q < 3; ++q) *(u32x4_t *)(lds + buf * STAGE + q * PART + i * 128 * 64 + wofs) = p[q];
    };

    // fragments (16 rows x 32 K): A row blocks 2 i, 2 i + 1 of the 32 rows wm +
    // 2 i (so a tile of few rows is shared by both wave rows), weight blocks j
    // of the wave's columns (gated: W1 and W3 rows of 16 h columns in turn)
    const int sw = (q4 ^ ((r16 >> 2) & 3)) << 4;
    const int afr = (wm * 32 + r16) * 64 + sw;
    const int bfr = (BM + wn * (NB == 2 ? 32 : 64) + r16) * 64 + sw;
    f32x4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int KTT = g.K / 32;
    const int kb = (ks * KTT) / S, ke = ((ks + 1) * KTT) / S;
    const int kl = ke - 1;  // the loads past the range repeat its last stage, into a buffer that nothing reads

    // Stage s is in buffer (s - kb) % 2.  Its MFMAs run in two halves of the
    // wave's columns, rows in order; a row block's fragments are replaced by
    // the next stage's once the second half is past it.  Per stage:
    //   columns 0, 1 | reads of (s, columns 2, 3)        | the weight rows of stage s + 1: split, written, loaded for s + 2
    //   barrier: stage s + 1 is written, and nothing more is read from buffer s
    //   columns 2, 3 | reads of (s + 1, rows, columns 0, 1) | the A row of stage s + 2: split, written, loaded for s + 3
    auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
#pragma unroll
    for (int i = 0; i < 3; ++i) load(i, kb);
#pragma unroll
    for (int i = 0; i < 3; ++i) split_store(0, i);
#pragma unroll
    for (int i = 0; i < 3; ++i) load(i, min(kb + 1, kl));
    split_store(1, 0);
    load(0, min(kb + 2, kl));
    barrier();

    auto run = [&](auto NV_) {
        constexpr int NV = decltype(NV_)::value;  // row blocks of this wave that hold rows of the tile
        constexpr int NF = 2 * NV;
        bf16x8_t fa[4][3], fb[2][2][3];
        auto read_a = [&](int buf, int i) {
#pragma unroll
            for (int q = 0; q < 3; ++q)
                fa[i][q] = *(const bf16x8_t *)(lds + buf * STAGE + q * PART + afr + ((i >> 1) * 64 + (i & 1) * 16) * 64);
        };
        auto read_b = [&](int buf, int hf) {
            if constexpr (NV > 0)
#pragma unroll
                for (int q = 0; q < 3; ++q)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        fb[hf][j][q] = *(const bf16x8_t *)(lds + buf * STAGE + q * PART + bfr +
                                                           (NB == 2 ? j * 128 + hf * 16 : (2 * hf + j) * 16) * 64);
        };
        auto row_mfmas = [&](int i, int hf) {
            f32x4_t t2[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) t2[j] = STAGE_SUMS ? f32x4_t{0.0f, 0.0f, 0.0f, 0.0f} : acc[i][2 * hf + j];
#pragma unroll
            for (int t = 0; t < 6; ++t) {
                constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    t2[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[hf][j][PB[t]], fa[i][PA[t]], t2[j], 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][2 * hf + j] = STAGE_SUMS ? acc[i][2 * hf + j] + t2[j] : t2[j];
        };
        // after each pair of MFMAs: VA vector instructions of the split, an LDS
        // read, at the end the LDS writes
        auto interleave = [&](auto VA_, auto NR_, auto NW_) {
            constexpr int NM = 6 * NF, NR = decltype(NR_)::value, NW = decltype(NW_)::value;
#pragma unroll
            for (int t = 0; t < NM; ++t) {
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                     // MFMAs
                __builtin_amdgcn_sched_group_barrier(0x002, decltype(VA_)::value, 0);  // vector instructions
                if (t < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);         // LDS read
                if (t >= NM - NW) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);   // LDS write
            }
        };
#pragma unroll
        for (int i = 0; i < NF; ++i) read_a(0, i);
        read_b(0, 0);
        for (int kt = kb; kt < ke; ++kt) {
            const int cur = (kt - kb) & 1;
            read_b(cur, 1);
            split_store(cur ^ 1, 1);
            split_store(cur ^ 1, 2);
            load(1, min(kt + 2, kl));
            load(2, min(kt + 2, kl));
#pragma unroll
            for (int i = 0; i < NF; ++i) row_mfmas(i, 0);
            if constexpr (NV > 0)
                interleave(std::integral_constant<int, (STAGE_SUMS ? 12 : 10) / NV>{}, std::integral_constant<int, 6>{},
                           std::integral_constant<int, 6>{});
            barrier();
            read_b(cur ^ 1, 0);
            split_store(cur, 0);
            load(0, min(kt + 3, kl));
#pragma unroll
            for (int i = 0; i < NF; ++i) {
                row_mfmas(i, 1);
                read_a(cur ^ 1, i);
            }
            if constexpr (NV > 0)
                interleave(std::integral_constant<int, (STAGE_SUMS ? 8 : 6) / NV>{}, std::integral_constant<int, 6 * NF>{},
                           std::integral_constant<int, 3>{});
        }
    };
    const int nv = (rows > wm * 32 ? 1 : 0) + (rows > wm * 32 + 64 ? 1 : 0);  // wave-uniform
    if (nv == 2) run(std::integral_constant<int, 2>{});
    else if (nv == 1) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 0>{});

    // ---- epilogue: lane holds row r16 of each row block and the columns 4 q4
    // .. + 3 of each weight block.
    const long long sofs = (long long)e * g.s_stride;
    auto row_of = [&](int i) { return (wm + 2 * (i >> 1)) * 32 + (i & 1) * 16 + r16; };
    // first column of the lane in column block j (gated: of h, from blocks 2 j and 2 j + 1)
    auto col_of = [&](int j) { return wn * (NB == 2 ? 32 : 64) + j * 16 + 4 * q4; };
    constexpr int NJ = 4 / NB;

    // redo: the wave's 64 x 64 sums on v_mfma_f32_16x16x4_f32, operands straight
    // from memory; those that the parts do not give are replaced.  It takes about
    // four times the tile's own MFMAs and runs for whole waves, whatever the
    // number of such sums: 768 / 3072 standard, 4096 tokens, us a call: 545; with
    // an infinity in one row 945, in every row 1300 (1720 and 46070 by one lane
    // per output and one K value after the other).
    auto good = [](float v) { return __builtin_isfinite(v) && (fabsf(v) >= 0x1p-90f || v == 0.0f); };
    // first in two instructions per sum: 0 v is not 0 for infinities and NaN, and
    // the smallest size, which zeros (rows of zeros, row blocks past the tile)
    // bring below the line too
    float nil[4] = {0.0f, 0.0f, 0.0f, 0.0f}, least = INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                nil[c] = fmaf(acc[i][j][c], 0.0f, nil[c]);
                least = fminf(least, fabsf(acc[i][j][c]));
            }
    bool all_good = (nil[0] + nil[1]) + (nil[2] + nil[3]) == 0.0f && least >= 0x1p-90f;
    if (!all_good) {
        all_good = true;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) all_good = all_good && (good(acc[i][j][c]) || row_of(i) >= rows);
    }
    if (__any(!all_good)) {
        const float *ap[4], *bp[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) ap[i] = A + (arow0 + min(row_of(i), rows - 1)) * g.lda + 4 * q4;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            bp[j] = NB == 2 ? ((j & 1) ? B1 : B0) + (long long)(wn * 32 + (j >> 1) * 16 + r16) * g.ldb + 4 * q4
                            : B0 + (long long)(wn * 64 + j * 16 + r16) * g.ldb + 4 * q4;
        f32x4_t sum[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) sum[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int k = kb * 32; k < ke * 32; k += 16) {  // lane (r16, q4): K k + 4 q4 .. + 3 of its rows
            f32x4_t av[4], bv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = *(const f32x4_t *)(ap[i] + k);
#pragma unroll
            for (int j = 0; j < 4; ++j) bv[j] = *(const f32x4_t *)(bp[j] + k);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[j][t], av[i][t], sum[i][j], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[i][j][c] = good(acc[i][j][c]) ? acc[i][j][c] : sum[i][j][c];
    }

    float *ws = S > 1 ? g.split_ws + ((long long)(mt * g.n_tiles + nt) * S + ks) * (BM * BR) : nullptr;
    const bool vec4 = (g.ldc & 3) == 0;
    // the activation is picked once per tile (picked per output, it was a
    // branch and a wait for each of a lane's 64 outputs)
    auto tile = [&](auto &&out) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int n = n0 + col_of(j);
            float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (MODE != MODE_GATED_UP && g.bias)
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (n + c < g.N) bias[c] = g.bias[sofs + n + c];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                f32x4_t v;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float v0 = acc[i][NB == 2 ? 2 * j : j][c], v1 = acc[i][NB == 2 ? 2 * j + 1 : j][c];
                    v[c] = out(arow0 + row_of(i), n + c, bias[c], v0, v1);
                }
                if (row_of(i) >= rows) continue;
                float *p = (float *)g.C + (arow0 + row_of(i)) * g.ldc + n;
                if (vec4 && n + 3 < g.N) {
                    *(f32x4_t *)p = v;
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (n + c < g.N) p[c] = v[c];
                }
            }
        }
    };
    auto tile_act = [&](auto ACT_) {
        constexpr int ACT = decltype(ACT_)::value;
        if constexpr (MODE == MODE_GATED_UP) {
            tile([](long long, int, float, float v0, float v1) { return act_apply(ACT, v0) * v1; });
        } else if constexpr (MODE == MODE_STD_UP) {
            if (g.drop_p > 0.0f)
                tile([&](long long row, int n, float bias, float v0, float) {
                    return dropout_h(g, row, n, act_apply(ACT, v0 + bias));
                });
            else tile([](long long, int, float bias, float v0, float) { return act_apply(ACT, v0 + bias); });
        } else {
            tile([](long long, int, float bias, float v0, float) { return v0 + bias; });
        }
    };
    if (S > 1) {  // a K range: its raw sums, [b][row][column] of split_ws block (tile, ks)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (row_of(i) >= rows) continue;
#pragma unroll
                for (int b = 0; b < NB; ++b) *(f32x4_t *)(ws + (b * BM + row_of(i)) * BN + col_of(j)) = acc[i][NB * j + b];
            }
    } else if constexpr (MODE == MODE_DOWN) {
        tile_act(std::integral_constant<int, MOE_ACT_IDENTITY>{});
    } else {
        switch (g.act) {
        case MOE_ACT_SILU: tile_act(std::integral_constant<int, MOE_ACT_SILU>{}); break;
        case MOE_ACT_GELU: tile_act(std::integral_constant<int, MOE_ACT_GELU>{}); break;
        case MOE_ACT_RELU: tile_act(std::integral_constant<int, MOE_ACT_RELU>{}); break;
        default: tile_act(std::integral_constant<int, MOE_ACT_IDENTITY>{});
        }
    }
}
