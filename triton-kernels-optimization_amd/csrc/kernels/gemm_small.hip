// gemm_small.hip -- MFMA GEMMs for few rows (decode steps, short prompts, the tiers of
// a small routed batch) on gfx950.
//
// What bounds them: the weights are read once, and a CU holds only ~100 requests open, so
// the read goes at chip rate only when every CU takes part.  A 128 x 128 tile gives M <= 128
// rows ceil(N / 128) workgroups (32 of 256 CUs at N = 4096), each also loading 128 rows of A.
// Here a tile is up to 64 rows by NWV column groups of 16 (FP8: 32, its MFMA's block):
//   compute waves (NWV = 1, 2 or 4): one column group each, all rows.  B, which no other wave
//     uses, goes from global memory straight into registers, D 128-byte K stages ahead.
//   one loader wave: A, which all of them use, by direct-to-LDS loads into a ring of four
//     16 KB chunks (1024 bytes of K for 16 rows, 256 for 64); one barrier per chunk.
// A tile of the last rows runs on the 16-, 32- or 64-row form that holds them.
// Measured (us per launch, 128-tile kernel before, this one now): INT8 4 x 4096 x 4096 13.8 /
// 5.5 (3 TB/s of weights), FP8 13.3 / 8.4, W8A16 22.2 / 9.2; W8A16 4 x 4096 x 14336 35 / 12.9
// (4.6 TB/s).  Also measured: one wave per 32 x 32 block with A and B through its own LDS ring, 8.4 (INT8,
// first shape: two LDS round trips per stage in one wave); A in registers too, 5.6 but 33 us for W8A16 16 x
// 4096 x 14336 (every wave pulls A through L1); B in whole 128-byte lines of 8 rows, exchanged by
// row_ror:8, 6.4 (the halves of a line already merge).
//
// Every block sums K in the order of the other kernels (the same MFMA on the same K slices, which is
// why K is never split and FP8 keeps its 32-wide blocks), so each tier's rows have the same
// bits whatever the tile.  EE_GEMM_W8A16 reads int8 codes and dequantises them in registers to the
// values eek_pack_b_f16 writes, in EE_GEMM_F16's order: its bits from half the bytes.
#include "../common/ee_device.h"
#include "../common/ee_gemm_dev.h"

#pragma clang fp contract(off)

#define SM_NC 4                         // chunks of A in the LDS ring
#define SM_CHUNK 16384                  // bytes of a chunk: 64 KB rings, two workgroups per CU ...
#define SM_DENSE 8192                   // ... or 32 KB, four, for routed grids of many workgroups per CU: 8 x
                                        // 2048 x 32000 20/40/40 % tiers 43.3 -> 39.4 us; but 8 x 4096 x 4096 (2.5 per
                                        // CU, better dealt two at a time) 12.7 -> 13.9
#define SM_ROWS 64                      // rows of a tile

// NI row groups by BJ column groups per wave (SwiGLU: BJ = 2, gate and up of the same outputs).
template <int KIND, int NI, int BJ, int SW, int NWV, int CHUNK>
struct SmallTile {
    static constexpr bool W8 = KIND == EE_GEMM_W8A16;
    static constexpr bool F16T = KIND == EE_GEMM_F16 || W8;
    static constexpr bool F8 = KIND == EE_GEMM_F8;
    static constexpr int R = F8 ? 32 : 16;                     // rows and columns of a block
    static constexpr int ESZ = F16T ? 2 : 1;
    static constexpr int BROW = W8 ? 64 : BKB;
    static constexpr int ROWS = NI * R;                        // A rows in LDS
    static constexpr int STG = ROWS * BKB;
    static constexpr int CH = CHUNK / STG;                  // stages per chunk
    // FP8 SwiGLU at 64 rows holds 64 accumulators.  The routed kernel has to fit 256 registers for four workgroups a
    // CU: four stages of B beside one buffer of A fragments, read just before use (two stages of B beside two buffers
    // fit too, but hold too few bytes in flight).  us, all rows FP8, 128-tile grid / two stages / this, with the
    // epilogue's loads below: 33 x 4096 x 4096 16.5 / 20.9 / 17.1, 64 x 4096 x 11264 18.3 / 22.5 / 18.4.
    static constexpr int NA = F8 && BJ == 2 && NI == 2 ? 1 : 2;
    static constexpr int D0 = F8 ? (BJ == 2 ? 4 : NI == 1 ? 8 : 6) : W8 ? (BJ == 2 ? 8 : 16) : (BJ == 2 ? 6 : 8);
    static constexpr int D = D0 / CH * CH > 0 ? D0 / CH * CH : CH;   // stages of B in registers: whole chunks
    typedef std::conditional_t<F8, i32x8, i32x4> frag_t;
    typedef std::conditional_t<F8, f32x16, std::conditional_t<F16T, f32x4, i32x4>> acc_t;
    // Raw B of a stage, 16 bytes per lane and load: one load per slice, whole 64-byte pieces of 16
    // rows (W8: one for both slices; FP8: two, the lane's two 16-byte chunks of its row)
    static constexpr int NL = W8 ? 1 : F8 ? 4 : 2;
    struct BStage { u32x4 v[BJ][NL]; };
    struct AStage { frag_t a[2][NI]; };

    const EeGemmArgs& g;
    uint8_t* smem;
    const uint8_t* pb[BJ];
    f16x2 s2[W8 ? BJ : 1];
    uint32_t ao;                                               // LDS offset of the lane's row 0 fragment
    __device__ __forceinline__ SmallTile(const EeGemmArgs& g_, uint8_t* s) : g(g_), smem(s) {}

    __device__ __forceinline__ void load(BStage& f, int i) {
#pragma unroll
        for (int l = 0; l < NL; ++l)
#pragma unroll
            for (int j = 0; j < BJ; ++j)
                f.v[j][l] = *(const u32x4*)(pb[j] + i * BROW + (F8 ? (l >> 1) * 64 + (l & 1) * 16 : l * 64));
    }
    // v_permlane16_swap: the odd 16-lane rows of x change places with the even ones of y
    static __device__ __forceinline__ void swap16(uint32_t& x, uint32_t& y) {
        const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
        x = r[0];
        y = r[1];
    }
    // B fragment of slice sl, column group j.
    // W8: lane group c loaded bytes 16 p(c) .. +15 of its row's 64, p = 0, 2, 1, 3; the swap leaves
    // slice 0's codes 8 (l >> 4) .. +7 in the first half and slice 1's in the second.
    __device__ __forceinline__ void frags(const BStage& f, int j, frag_t (&b)[2]) {
        if constexpr (W8) {
            uint32_t x0 = f.v[j][0][0], x1 = f.v[j][0][1], y0 = f.v[j][0][2], y1 = f.v[j][0][3];
            swap16(x0, y0);
            swap16(x1, y1);
            uint32_t w0, w1, w2, w3;
            dq4(x0, s2[j], w0, w1);
            dq4(x1, s2[j], w2, w3);
            b[0] = i32x4{(int)w0, (int)w1, (int)w2, (int)w3};
            dq4(y0, s2[j], w0, w1);
            dq4(y1, s2[j], w2, w3);
            b[1] = i32x4{(int)w0, (int)w1, (int)w2, (int)w3};
        } else if constexpr (F8) {
#pragma unroll
            for (int sl = 0; sl < 2; ++sl) {
                const i32x4 x = as_i32x4(f.v[j][2 * sl]), y = as_i32x4(f.v[j][2 * sl + 1]);
                b[sl] = i32x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
            }
        } else {
            b[0] = as_i32x4(f.v[j][0]);
            b[1] = as_i32x4(f.v[j][1]);
        }
    }
    // fragments of the stage at s; slice 1's chunks are slice 0's with bit 6 flipped, row r + R's lie R * 128 on
    __device__ __forceinline__ void read(AStage& f, const uint8_t* s) {
#pragma unroll
        for (int sl = 0; sl < 2; ++sl)
#pragma unroll
            for (int r = 0; r < NI; ++r) {
                const uint8_t* q = s + (ao ^ (sl * 64)) + r * R * BKB;
                if constexpr (F8) {
                    const i32x4 x = *(const i32x4*)q, y = *(const i32x4*)(s + ((ao ^ (sl * 64)) ^ 16) + r * R * BKB);
                    f.a[sl][r] = i32x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
                } else {
                    f.a[sl][r] = *(const i32x4*)q;
                }
            }
    }
    __device__ __forceinline__ void compute(const BStage& fb, const AStage& fa, acc_t (&acc)[NI][BJ]) {
        frag_t b[BJ][2];
#pragma unroll
        for (int j = 0; j < BJ; ++j) frags(fb, j, b[j]);
#pragma unroll
        for (int sl = 0; sl < 2; ++sl)
#pragma unroll
            for (int j = 0; j < BJ; ++j)
#pragma unroll
                for (int r = 0; r < NI; ++r) {
                    if constexpr (F8)
                        acc[r][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(b[j][sl], fa.a[sl][r], acc[r][j], 0, 0, 0, 0, 0, 0);
                    else if constexpr (F16T)
                        acc[r][j] = PipeF16x16::m16(b[j][sl], fa.a[sl][r], acc[r][j]);
                    else
                        acc[r][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b[j][sl], fa.a[sl][r], acc[r][j], 0, 0, 0);
                }
    }
    static __device__ __forceinline__ void barrier() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }

    // The loader wave: A chunks into the ring.  Barrier c: chunk c has landed and chunk c - 1 has been read.
    __device__ __forceinline__ void loader(int m0, int M, int64_t off, int nk) {
        constexpr int NG = ROWS / 8;
        const int lane = (int)(threadIdx.x & 63);
        const uint8_t* pa[NG];
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const int r = i * 8 + (lane >> 3), m = min(m0 + r, M - 1);
            const int64_t ar = g.a_idx ? (int64_t)g.a_idx[off + m] : off + m;
            pa[i] = (const uint8_t*)g.a + ar * g.lda * ESZ + ((lane & 7) ^ swz(r)) * 16;
        }
        const int nc = (nk + CH - 1) / CH;
        // every chunk issues CH * NG loads (a constant count for the waits): past K they repeat the last stage
        auto issue = [&](int c) {
            const uint32_t s = lds_addr(smem) + (uint32_t)((c % SM_NC) * CHUNK);
#pragma unroll
            for (int st = 0; st < CH; ++st) {
                const int64_t kb = (int64_t)min(c * CH + st, nk - 1) * BKB;
#pragma unroll
                for (int i = 0; i < NG; ++i) dma16(pa[i] + kb, s + st * STG + i * 1024);
            }
        };
        constexpr int L = CH * NG;
        static_assert(L * 1024 == CHUNK && SM_NC >= 2 && (SM_NC - 1) * L < 64, "");
#pragma unroll
        for (int c = 0; c < SM_NC; ++c)
            if (c < nc) issue(c);
        for (int c = 0; c < nc; ++c) {
            const int last = c == 0 ? SM_NC - 1 : c + SM_NC - 2;   // chunks issued so far
            const int after = min(last, nc - 1) - c;
            if (after >= 3) WAITCNT_VM(3 * L);
            else if (after == 2) WAITCNT_VM(2 * L);
            else if (after == 1) WAITCNT_VM(L);
            else WAITCNT_VM(0);
            barrier();
            if (c >= 1 && c - 1 + SM_NC < nc) issue(c - 1 + SM_NC);
        }
    }

    __device__ __forceinline__ void run(int m0, int tn, int M, int64_t off) {
        const int nk = (int)((int64_t)g.K * ESZ / BKB);
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        if (wave == NWV) {
            loader(m0, M, off, nk);
            return;
        }
        const int lane = (int)(threadIdx.x & 63);
        const int lr = lane & (R - 1), lk = lane / R;          // row of the block, K group of the lane
        const int cg = tn * NWV + wave;                        // the wave's column group
        int nb[BJ];
#pragma unroll
        for (int j = 0; j < BJ; ++j)
            nb[j] = SW ? (F8 ? cg * 64 + j * 32 : (cg >> 1) * 64 + (cg & 1) * 16 + j * 32) : (cg * BJ + j) * R;
        // byte of its row where the lane's part of a B load starts
        const int bo = (W8 ? (lk & 1) << 1 | lk >> 1 : F8 ? 2 * lk : lk) * 16;
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
            const int n = min(nb[j] + lr, g.N - 1);
            pb[j] = (const uint8_t*)g.b + (int64_t)n * g.ldb * (W8 ? 1 : ESZ) + bo;
            if constexpr (W8) {
                const float s = g.b_scale[n];
                s2[j] = f16x2{(f16)s, (f16)s};
            }
        }
        ao = lds_off(lr, lk * (F8 ? 2 : 1));                   // swz(r + 16 i) == swz(r)
        acc_t acc[NI][BJ];
#pragma unroll
        for (int r = 0; r < NI; ++r)
#pragma unroll
            for (int j = 0; j < BJ; ++j) acc[r][j] = acc_t{};
        BStage f[D];                                           // B, D stages ahead
#pragma unroll
        for (int i = 0; i < D; ++i)
            if (i < nk) load(f[i], i);
        AStage fa[NA];                                         // A, one stage ahead with two buffers (D is even)
        barrier();                                             // chunk 0 has landed
        if constexpr (NA == 2) read(fa[0], smem);
        // D stages from k0; FULL: all of them are below nk, RELOAD: so are the next D
        auto pass = [&](int k0, auto full, auto reload) {
            constexpr bool FULL = decltype(full)::value, RELOAD = decltype(reload)::value;
#pragma unroll
            for (int j = 0; j < BJ; ++j) pb[j] += D * BROW;
#pragma unroll
            for (int i = 0; i < D; ++i) {
                if constexpr (NA == 1) {
                    if (FULL || k0 + i < nk) {
                        if (i % CH == 0 && k0 + i > 0) {       // the chunk before has been read, this one has landed
                            WAITCNT_LGKM0();
                            barrier();
                        }
                        read(fa[0], smem + ((k0 + i) / CH % SM_NC) * CHUNK + i % CH * STG);
                        compute(f[i], fa[0], acc);
                    }
                } else if (FULL || k0 + i < nk) {
                    if ((RELOAD || (FULL && i + 1 < D)) || k0 + i + 1 < nk) {
                        if ((i + 1) % CH == 0) {
                            WAITCNT_LGKM0();                   // this chunk has been read
                            barrier();                         // ... by every wave, and the next one has landed
                        }
                        read(fa[(i + 1) & 1], smem + ((k0 + i + 1) / CH % SM_NC) * CHUNK + (i + 1) % CH * STG);
                    }
                    compute(f[i], fa[i & 1], acc);
                }
                if (FULL && (RELOAD || k0 + D + i < nk)) load(f[i], i);
                __builtin_amdgcn_sched_barrier(0);             // the loads stay D stages ahead of their use
            }
        };
        int k0 = 0;
        for (; k0 + 2 * D <= nk; k0 += D) pass(k0, std::true_type{}, std::true_type{});
        if (k0 + D <= nk) {
            pass(k0, std::true_type{}, std::false_type{});
            k0 += D;
        }
        if (k0 < nk) pass(k0, std::false_type{}, std::false_type{});

        // epilogue: lane holds row lr, columns 4 lk .. +3 (FP8: 8 q + 4 lk .. +3) of each block
        constexpr int NQ = F8 ? 4 : 1;
        // What the stores need from memory, all of it at once: row group by row group under the branch below,
        // each waited for its own (FP8 SwiGLU 128 x 256 x 2048 7.6 us, now 6.3).
        int64_t crow[NI];
        float as[NI];
        f32x4 bs[BJ][NQ];
#pragma unroll
        for (int r = 0; r < NI; ++r) {
            const int m = min(m0 + r * R + lr, M - 1);
            crow[r] = g.c_idx ? (int64_t)g.c_idx[off + m] : (int64_t)m;
            as[r] = F16T ? 0.0f : g.a_scale[off + m];
        }
        if constexpr (!F16T) {
#pragma unroll
            for (int j = 0; j < BJ; ++j)
#pragma unroll
                for (int q = 0; q < NQ; ++q) bs[j][q] = *(const f32x4*)(g.b_scale + min(nb[j] + 8 * q + 4 * lk, g.N - 4));
        }
#pragma unroll
        for (int r = 0; r < NI; ++r) {
            if (m0 + r * R + lr >= M) continue;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                uint32_t o[BJ][2];
#pragma unroll
                for (int j = 0; j < BJ; ++j) {
                    const int n = nb[j] + 8 * q + 4 * lk;
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if constexpr (F16T) v[e] = acc[r][j][4 * q + e];
                        else v[e] = deq<KIND>(acc[r][j][4 * q + e], as[r], bs[j][q][e]);
                    }
                    o[j][0] = pack_f16x2(v[0], v[1]);
                    o[j][1] = pack_f16x2(v[2], v[3]);
                    if constexpr (!SW) {
                        if (n < g.N) {                         // N is a multiple of 4
                            *(u32x2*)(g.c + crow[r] * g.ldc + n) = u32x2{o[j][0], o[j][1]};
                            if constexpr (KIND == EE_GEMM_I8) {
                                if (g.acc) *(i32x4*)(g.acc + crow[r] * g.ldc + n) = acc[r][j];
                            }
                        }
                    }
                }
                if constexpr (SW) {
                    const int n = cg * R + 8 * q + 4 * lk;
                    if (n < (g.N >> 1))
                        *(u32x2*)(g.c + crow[r] * g.ldc + n) = u32x2{silu_mul2(o[0][0], o[1][0]), silu_mul2(o[0][1], o[1][1])};
                }
            }
        }
    }
};

// Up to 64 rows of C by the 16- or 32-row groups they need.
template <int KIND, int SW, int NWV, int CHUNK>
EE_DEV void tile_small(const EeGemmArgs& g, int tm, int tn, uint8_t* smem) {
    const int M = g.counts ? g.counts[g.tier] : g.M;
    const int64_t off = g.counts ? tier_offset(g.counts, g.tier) : 0;
    const int m0 = tm * SM_ROWS, rows = M - m0;
    constexpr int BJ = SW ? 2 : 1;
    if (rows <= 0) return;
    if constexpr (KIND == EE_GEMM_F8) {
        if (rows <= 32) SmallTile<KIND, 1, BJ, SW, NWV, CHUNK>(g, smem).run(m0, tn, M, off);
        else SmallTile<KIND, 2, BJ, SW, NWV, CHUNK>(g, smem).run(m0, tn, M, off);
    } else {
        if (rows <= 16) SmallTile<KIND, 1, BJ, SW, NWV, CHUNK>(g, smem).run(m0, tn, M, off);
        else if (rows <= 32) SmallTile<KIND, 2, BJ, SW, NWV, CHUNK>(g, smem).run(m0, tn, M, off);
        else SmallTile<KIND, 4, BJ, SW, NWV, CHUNK>(g, smem).run(m0, tn, M, off);
    }
}

// M fastest: the M-tiles of a column panel read its weights through one L2.
template <int KIND, int SW, int NWV>
EE_DEV void gemm_small(const EeGemmArgs& g) {
    __shared__ __attribute__((aligned(1024))) uint8_t smem[SM_NC * SM_CHUNK];
    const int tiles_m = (g.M + SM_ROWS - 1) / SM_ROWS;
    int i = (int)blockIdx.x >> 3;
    if (xcd_share((int)gridDim.x, i)) {
        const int tn = tile_div(i, tiles_m);
        tile_small<KIND, SW, NWV, SM_CHUNK>(g, i - tn * tiles_m, tn, smem);
    }
}

// The routed linear's tier GEMMs as one grid of at least as many workgroups as the tiers
// have tiles (the counts are on the device; the surplus exits).  Every XCD gets an eighth of
// each tier's tiles, the W8A16 ones (t[2]: int8 codes), which take longest, first.
template <int SW, int NWV, int CHUNK>
EE_DEV void gemm_small_routed(const EeRoutedGemmArgs& r) {
    __shared__ __attribute__((aligned(1024))) uint8_t smem[SM_NC * CHUNK];
    const int32_t* counts = r.t[0].counts;
    const int T0 = (counts[0] + SM_ROWS - 1) / SM_ROWS, T1 = (counts[1] + SM_ROWS - 1) / SM_ROWS;
    const int T2 = (counts[2] + SM_ROWS - 1) / SM_ROWS;
    constexpr int C = 16 * NWV * (SW ? 2 : 1);                 // columns of a tile; FP8: 2 C
    const int n = (r.t[0].N + C - 1) / C, n8 = (r.t[0].N + 2 * C - 1) / (2 * C);
    int i = (int)blockIdx.x >> 3;
    if (xcd_share(T2 * n, i)) {
        const int tn = tile_div(i, T2);
        tile_small<EE_GEMM_W8A16, SW, NWV, CHUNK>(r.t[2], i - tn * T2, tn, smem);
    } else if (xcd_share(T1 * n8, i)) {
        const int tn = tile_div(i, T1);
        tile_small<EE_GEMM_F8, SW, NWV, CHUNK>(r.t[1], i - tn * T1, tn, smem);
    } else if (xcd_share(T0 * n, i)) {
        const int tn = tile_div(i, T0);
        tile_small<EE_GEMM_I8, SW, NWV, CHUNK>(r.t[0], i - tn * T0, tn, smem);
    }
}

#define EE_SMALL_ENTRY(SUFFIX, KIND, W)                                                                         \
    extern "C" __global__ void __launch_bounds__(64 * (W + 1)) eek_gemm_m64w##W##_##SUFFIX(EeGemmArgs g) {      \
        gemm_small<KIND, 0, W>(g);                                                                              \
    }
#define EE_SMALL_ENTRY_SW(SUFFIX, KIND, W)                                                                      \
    extern "C" __global__ void __launch_bounds__(64 * (W + 1)) eek_gemm_m64w##W##_##SUFFIX##_swiglu(EeGemmArgs g) { \
        gemm_small<KIND, 1, W>(g);                                                                              \
    }
#define EE_SMALL_ROUTED(NAME, SW, W, CHUNK)                                                                     \
    extern "C" __global__ void __launch_bounds__(64 * (W + 1)) __attribute__((amdgpu_waves_per_eu(2)))           \
    NAME(EeRoutedGemmArgs r) {                                                                                  \
        gemm_small_routed<SW, W, CHUNK>(r);                                                                     \
    }
#define EE_SMALL_WAVES(W)                                                                                       \
    EE_SMALL_ENTRY(i8, EE_GEMM_I8, W)                                                                           \
    EE_SMALL_ENTRY(f8, EE_GEMM_F8, W)                                                                           \
    EE_SMALL_ENTRY(f16, EE_GEMM_F16, W)                                                                         \
    EE_SMALL_ENTRY(w8a16, EE_GEMM_W8A16, W)
#define EE_SMALL_WAVES_SW(W)                                                                                    \
    EE_SMALL_ENTRY_SW(i8, EE_GEMM_I8, W)                                                                        \
    EE_SMALL_ENTRY_SW(f8, EE_GEMM_F8, W)                                                                        \
    EE_SMALL_ENTRY_SW(f16, EE_GEMM_F16, W)                                                                      \
    EE_SMALL_ENTRY_SW(w8a16, EE_GEMM_W8A16, W)
EE_SMALL_WAVES(1)
EE_SMALL_WAVES(2)
EE_SMALL_WAVES(4)
EE_SMALL_WAVES_SW(1)
EE_SMALL_WAVES_SW(2)
EE_SMALL_ROUTED(eek_gemm_routed_m64w1, 0, 1, SM_CHUNK)
EE_SMALL_ROUTED(eek_gemm_routed_m64w2, 0, 2, SM_CHUNK)
EE_SMALL_ROUTED(eek_gemm_routed_m64w2_dense, 0, 2, SM_DENSE)
EE_SMALL_ROUTED(eek_gemm_routed_m64w1_swiglu, 1, 1, SM_DENSE)
