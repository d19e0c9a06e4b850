// softmax_entropy.hip -- fused row softmax + Shannon entropy for gfx950.
//
// Computes, for every row r of fp16 logits x (S columns, causal optional):
//   m = max x,  s = x - m,  Z = sum e^s,  p = e^s / Z  (stored fp16, RNE)
//   H = ln Z - sum p*s   (masked columns contribute 0)
// which is the function of the reference's fused_softmax_entropy_kernel
// (EE/python/kernels.py:264-312).  H is evaluated in the cancellation-free
// form  H = ln(c0) + log1p(Z'/c0) - T/(c0 + Z')  with c0 = number of entries
// equal to the max, Z' = sum of e^s over the other entries and T = sum e^s*s;
// every term is non-negative, so nearly one-hot rows keep full relative
// precision (the plain ln Z form loses ~1e-4 relative at H ~ 5e-4 in f32).
//
// Layout: row-major rows, unit column stride.  One to eight wave64s per row;
// each lane holds VPT 16-byte vectors (8 fp16) of the row in registers, so
// the row is read from HBM exactly once and the probabilities are written
// once: 2 bytes in + 2 bytes out per element + 4 bytes of H per row.
#include "../common/ee_device.h"
#include "../common/ee_softmax_dev.h"

// 16 bytes of a row, which starts at any multiple of 2 bytes: gfx950 loads and stores them at any
// address (the compiler emits the same global_load_dwordx4 for either alignment).
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(2)));

// Rows per block for WPR waves per row (the block holds RPB * WPR waves).
template <int WPR>
struct SeGeom {
    static constexpr int RPB = WPR == 1 ? 4 : (WPR == 2 ? 2 : 1);
    static constexpr int BLOCK = RPB * WPR * 64;
};

EE_DEV int tier_of(float h, double tl, double th) {
    const double d = (double)h;
    return d < tl ? 0 : (d < th ? 1 : 2);
}

// (x - m) log2 e in one v_fma_mix_f32: x * log2e + (-m log2e), one rounding.
// The waves of a row that hold no entry equal to the max take this form (one
// instruction per element instead of two); it is within 2^-24 |m log2 e| of
// the two-step value, so e changes by at most a few f32 ulps.
EE_DEV float sub2_lo(uint32_t u, float l2e, float negml) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(u), "s"(l2e), "v"(negml));
    return r;
}
EE_DEV float sub2_hi(uint32_t u, float l2e, float negml) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(u), "s"(l2e), "v"(negml));
    return r;
}
// A row whose max is within 104 of the lowest fp16 value: -inf entries (masked or padding) clamped to
// -65504 would count beside it (e^-104 is the first e that is 0 in f32), so the row is moved up by 32768
// first, exactly (its finite entries are multiples of 32 from -65504 up; -inf stays).
#define NEAR_LOWEST(m) ((m) < -65376.0f)
#define LOW_SHIFT 32768.0f
EE_DEV uint32_t shift_up(uint32_t u) {
    const f16x2 s = {(f16)LOW_SHIFT, (f16)LOW_SHIFT};
    return bits_of(f16x2_from_bits(u) + s);
}

// Row kernel: WPR wave64s per row (one to eight), VPT 16-byte vectors per lane
// (S <= VPT * WPR * 512).  Passes over the registers:
//  1. max with packed fp16 IEEE maximum (NaN anywhere, or no finite entry,
//     makes the row NaN, as the reference's e^(x - m) / Z does);
//  2. -inf (masked or padded) entries clamped to -65504 with a packed max, so
//     they give e = 0 and e * s = 0 without a per-element guard;
//  3. e = 2^((x - m) log2 e), Z' and T = sum e * s.  Only a wave whose lanes
//     hold an entry equal to the row max (one wave of the row, typically) needs
//     the per-element test that keeps those entries out of Z' and counts them
//     (c0); the others take the test-free loop;
//  4. probabilities p = fp16(e / Z) from the kept e (VPT <= 4) or recomputed e,
//     stored before
//  5. H, which only the row's first wave evaluates (its stores drain meanwhile).
// The row's registers: lane l of wave wr of the row holds 16-byte vectors
// j = 0 .. VPT-1 at column ((j * WPR + wr) * 64 + l) * 8; entries past the row
// (or past the causal limit) read as -inf and are not loaded.
// NT: non-temporal loads (the _nt kernels: logits read once from HBM).
template <int VPT, int WPR, bool NT = false>
EE_DEV void se_load(const EeSoftmaxArgs& a, int64_t r, int wr, int lane, u32x4 (&v)[VPT]) {
    const int S = a.S;
    const int nvalid = a.causal ? min(S, (int)(r % S) + 1) : S;
    const uint16_t* xr = a.x + r * a.ld_x;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int c0 = ((j * WPR + wr) * 64 + lane) * 8;
        if (c0 + 8 <= nvalid) {
            if constexpr (NT) v[j] = __builtin_nontemporal_load((const u32x4_u*)(xr + c0));
            else v[j] = *(const u32x4_u*)(xr + c0);
        } else {
            uint16_t e[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) e[i] = (c0 + i < nvalid) ? xr[c0 + i] : (uint16_t)0xFC00u;  // -inf
            v[j] = u32x4{e[0] | ((uint32_t)e[1] << 16), e[2] | ((uint32_t)e[3] << 16),
                         e[4] | ((uint32_t)e[5] << 16), e[6] | ((uint32_t)e[7] << 16)};
        }
    }
}

// H of a row from its reduced sums, and its tier, written by lane 0.
EE_DEV void se_entropy_out(const EeSoftmaxArgs& a, int64_t row, bool dead, float cz, float z, float t, int lane) {
    const float H = dead ? NAN : entropy_from(cz, z, t);
    if (lane == 0) {
        a.h[row] = H;
        if (a.tier) a.tier[row] = tier_of(H, a.tau_low, a.tau_high);
    }
}

// Steps 1-5 for one row held in v (red: the block's cross-wave partials when WPR > 1).
template <int VPT, int WPR>
EE_DEV void se_process(const EeSoftmaxArgs& a, u32x4 (&v)[VPT], int64_t row, bool valid, int w, int wr, int lane,
                       float (*red)[4]) {
    constexpr bool KEEP_E = VPT <= 4;
    const int S = a.S;

    // ---- 1. max
    f16x2 mx2 = f16x2_from_bits(0xFC00FC00u);
#pragma unroll
    for (int j = 0; j < VPT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx2 = __builtin_elementwise_maximum(mx2, f16x2_from_bits(v[j][i]));
    const float m_lane = fmaximum((float)mx2.x, (float)mx2.y);
    float m = wave_maximum(m_lane);
    if constexpr (WPR > 1) {
        if (lane == 0) red[w][0] = m;
        __syncthreads();
        const int base = (w / WPR) * WPR;
        m = red[base][0];
#pragma unroll
        for (int i = 1; i < WPR; ++i) m = fmaximum(m, red[base + i][0]);
    }
    const bool dead = !(m > -INFINITY);
    const bool has_max = __builtin_amdgcn_ballot_w64(m_lane == m) != 0;   // wave-uniform
    if (dead) m = 0.0f;
    if (NEAR_LOWEST(m)) {                             // (wave-uniform)
#pragma unroll
        for (int j = 0; j < VPT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) v[j][i] = shift_up(v[j][i]);
        m += LOW_SHIFT;
    }
    const float negm = -m;

    // ---- 2. -inf -> -65504 (after the max, so NaN rows stay dead).  IEEE maximum
    // (NaN-propagating) needs no canonicalising max of its input first, as maxnum
    // does: one v_pk_maximum3_f16 per two elements.
    const f16x2 lowest = f16x2_from_bits(0xFBFFFBFFu);
#pragma unroll
    for (int j = 0; j < VPT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[j][i] = bits_of(__builtin_elementwise_maximum(f16x2_from_bits(v[j][i]), lowest));

    // ---- 3. sums
    float ek[KEEP_E ? VPT * 8 : 1];
    float z0 = 0.f, z1 = 0.f, t0 = 0.f, t1 = 0.f;
    int cnt = 0;
    const float negml = negm * LOG2E;
    if (!has_max) {
        // s2 = (x - m) log2 e; T accumulates e * s2 and is scaled by ln 2 below
#pragma unroll
        for (int j = 0; j < VPT; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t u = v[j][i >> 1];
                const float s2 = (i & 1) ? sub2_hi(u, LOG2E, negml) : sub2_lo(u, LOG2E, negml);
                const float e = __builtin_amdgcn_exp2f(s2);
                if (i & 1) { z1 += e; t1 = fmaf(e, s2, t1); }
                else       { z0 += e; t0 = fmaf(e, s2, t0); }
                if (KEEP_E) ek[j * 8 + i] = e;
            }
    } else {
#pragma unroll
        for (int j = 0; j < VPT; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t u = v[j][i >> 1];
                const float s = (i & 1) ? sub_hi(u, negm) : sub_lo(u, negm);
                const float e = __builtin_amdgcn_exp2f(s * LOG2E);
                const bool at_max = (s == 0.0f);
                cnt += at_max ? 1 : 0;
                if (i & 1) { z1 += at_max ? 0.0f : e; t1 = fmaf(e, s, t1); }
                else       { z0 += at_max ? 0.0f : e; t0 = fmaf(e, s, t0); }
                if (KEEP_E) ek[j * 8 + i] = e;
            }
    }
    float z = wave_sum(z0 + z1);
    float t = wave_sum(t0 + t1);
    if (!has_max) t *= LN2;
    float cz = has_max ? (float)wave_sum_i32(cnt) : 0.0f;   // cnt is 0 in every lane elsewhere
    if constexpr (WPR > 1) {
        if (lane == 0) { red[w][1] = z; red[w][2] = t; red[w][3] = cz; }
        __syncthreads();
        const int base = (w / WPR) * WPR;
        z = red[base][1]; t = red[base][2]; cz = red[base][3];
#pragma unroll
        for (int i = 1; i < WPR; ++i) { z += red[base + i][1]; t += red[base + i][2]; cz += red[base + i][3]; }
    }
    if (!valid) return;
    // One wave x 4 vectors (eight waves per SIMD, 64 VGPRs) has no registers to keep
    // the row sums through the stores: it evaluates H first.
    constexpr bool H_FIRST = WPR == 1 && VPT == 4;
    if constexpr (H_FIRST) se_entropy_out(a, row, dead, cz, z, t, lane);

    // ---- 4. one write of the probabilities, issued before H is evaluated so that
    // the stores drain while the row's first wave computes it (1/Z from v_rcp_f32,
    // within 1 ulp; Z >= 1)
    if (a.p != nullptr) {
        const float invZ = dead ? NAN : __builtin_amdgcn_rcpf(cz + z);
        uint16_t* pr = a.p + row * a.ld_p;
    #pragma unroll
        for (int j = 0; j < VPT; ++j) {
            const int c0 = ((j * WPR + wr) * 64 + lane) * 8;
            if (c0 >= S) continue;
            float ev[8];
    #pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (KEEP_E) {
                    ev[i] = ek[j * 8 + i];
                } else {                                  // the e of step 3, recomputed
                    const uint32_t u = v[j][i >> 1];
                    ev[i] = __builtin_amdgcn_exp2f(has_max ? ((i & 1) ? sub_hi(u, negm) : sub_lo(u, negm)) * LOG2E
                                                           : ((i & 1) ? sub2_hi(u, LOG2E, negml) : sub2_lo(u, LOG2E, negml)));
                }
            }
            const u32x4 o{scale_pack_f16x2(ev[0], ev[1], invZ), scale_pack_f16x2(ev[2], ev[3], invZ),
                          scale_pack_f16x2(ev[4], ev[5], invZ), scale_pack_f16x2(ev[6], ev[7], invZ)};
            if (c0 + 8 <= S) {
                // written once, read by a later kernel: non-temporal (measured 5% faster
                // at [4096, 14336], where the kernel runs at ~93% of a plain copy)
                __builtin_nontemporal_store(o, (u32x4_u*)(pr + c0));
            } else {
    #pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (c0 + i < S) pr[c0 + i] = (uint16_t)(o[i >> 1] >> ((i & 1) * 16));
            }
        }
    }
    // ---- 5. H and the tier, by the row's first wave
    if (!H_FIRST && wr == 0) se_entropy_out(a, row, dead, cz, z, t, lane);
}

template <int VPT, int WPR, bool NT = false>
EE_DEV void softmax_entropy_vec(const EeSoftmaxArgs& a) {
    typedef SeGeom<WPR> G;
    __shared__ float red[G::RPB * WPR][4];
    const int lane = lane_id();
    const int w = wave_id();
    const int wr = w % WPR;
    const int64_t row = (int64_t)blockIdx.x * G::RPB + w / WPR;
    const bool valid = row < a.rows;
    const int64_t r = valid ? row : a.rows - 1;    // keep every wave in the barriers
    u32x4 v[VPT];
    se_load<VPT, WPR, NT>(a, r, wr, lane, v);
    se_process<VPT, WPR>(a, v, row, valid, w, wr, lane, red);
}

// Short rows (one wave per row): each wave takes RPW consecutive rows and
// issues all their loads before working on the first, so a wave keeps
// RPW x VPT x 1 KB of the input in flight instead of VPT x 1 KB.
template <int VPT, int RPW>
EE_DEV void softmax_entropy_rows(const EeSoftmaxArgs& a) {
    const int lane = lane_id();
    const int w = wave_id();
    const int64_t row0 = ((int64_t)blockIdx.x * (EE_BLOCK / 64) + w) * RPW;
    u32x4 v[RPW][VPT];
#pragma unroll
    for (int q = 0; q < RPW; ++q) se_load<VPT, 1>(a, min(row0 + q, a.rows - 1), 0, lane, v[q]);
#pragma unroll
    for (int q = 0; q < RPW; ++q) {
        if (row0 + q >= a.rows) break;                // wave-uniform; no barriers in se_process<., 1>
        se_process<VPT, 1>(a, v[q], row0 + q, true, w, 0, lane, nullptr);
    }
}

// Rows of up to 1024 columns in groups of LPR lanes (16 or 32): a wave works on 64 / LPR
// consecutive rows at once, each lane holding VPT vectors of its row (S <= 8 LPR VPT).
// With one wave per row the kernel is bound by its instructions there, not by memory: per row the
// wave reductions (max, Z', T, c0: ~130 instructions) cost as much as the row's 8 elements per
// lane.  Here they serve 4 (2) rows, over 16 lanes by DPP alone.  Vectors past every row's
// causal limit are neither loaded nor evaluated.  Measured at [131072, 512] with
// probabilities: causal 59.9 -> 35.4 us (5.7 TB/s of the bytes the rows cannot do
// without), all columns 54.0 -> 42.4 us (6.3 TB/s, a large copy's rate).
// Same steps, per-element arithmetic and results as se_process (the sums in another order).
template <int LPR>
EE_DEV float grp_max(float v) {                    // IEEE maximum over the lane's group
    v = fmaximum(v, dpp_f32<0xB1>(v));
    v = fmaximum(v, dpp_f32<0x4E>(v));
    v = fmaximum(v, dpp_f32<0x141>(v));
    v = fmaximum(v, dpp_f32<0x140>(v));
    if constexpr (LPR == 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = fmaximum(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    return v;
}
template <int LPR>
EE_DEV float grp_sum(float v) {
    v += dpp_f32<0xB1>(v);
    v += dpp_f32<0x4E>(v);
    v += dpp_f32<0x141>(v);
    v += dpp_f32<0x140>(v);
    if constexpr (LPR == 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    return v;
}

template <int VPT, int LPR>
EE_DEV void softmax_entropy_group(const EeSoftmaxArgs& a) {
    constexpr int RPW = 64 / LPR;
    const int lane = lane_id(), gl = lane & (LPR - 1), grp = lane / LPR;
    const int S = a.S;
    // (the launcher keeps rows below 2^31 and S >= 16)
    const uint32_t row0 = __builtin_amdgcn_readfirstlane((blockIdx.x * (EE_BLOCK / 64) + wave_id()) * RPW);
    if (row0 >= (uint32_t)a.rows) return;
    const uint32_t row = min(row0 + grp, (uint32_t)a.rows - 1);   // past the end: the last row again, not stored
    int nvalid = S, nmax = S;                      // columns of the row, and of the wave's longest row
    if (a.causal) {
        const int p0 = __builtin_amdgcn_readfirstlane((int)(row0 % (uint32_t)S));
        const int p = p0 + (int)(row - row0);
        nvalid = (p >= S ? p - S : p) + 1;
        nmax = min(S, p0 + RPW);                   // (a wave that wraps holds row S - 1)
    }
    const uint16_t* xr = a.x + (int64_t)row * a.ld_x;
    u32x4 v[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        v[j] = u32x4{0xFC00FC00u, 0xFC00FC00u, 0xFC00FC00u, 0xFC00FC00u};
        if (j * LPR * 8 < nmax) {                  // uniform
            const int c0 = (j * LPR + gl) * 8;
            if (c0 < nvalid) {
                if (c0 + 8 <= S) {
                    v[j] = *(const u32x4_u*)(xr + c0);
                } else {                           // the row's last, partial vector
                    uint16_t e[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) e[i] = c0 + i < S ? xr[c0 + i] : (uint16_t)0xFC00u;
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[j][i] = e[2 * i] | ((uint32_t)e[2 * i + 1] << 16);
                }
            }
        }
    }
    if (a.causal) {                                // -inf past the limit, in the vector that it cuts
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            const int k = nvalid - (j * LPR + gl) * 8;
            if (j * LPR * 8 < nmax && k > 0 && k < 8) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (k < 2 * i + 2) v[j][i] = k == 2 * i + 1 ? (v[j][i] & 0xffffu) | 0xFC000000u : 0xFC00FC00u;
                }
            }
        }
    }
    f16x2 mx2 = f16x2_from_bits(0xFC00FC00u);
#pragma unroll
    for (int j = 0; j < VPT; ++j)
        if (j * LPR * 8 < nmax) {
#pragma unroll
            for (int i = 0; i < 4; ++i) mx2 = __builtin_elementwise_maximum(mx2, f16x2_from_bits(v[j][i]));
        }
    float m = grp_max<LPR>(fmaximum((float)mx2.x, (float)mx2.y));
    const bool dead = !(m > -INFINITY);
    if (dead) m = 0.0f;
    if (__builtin_amdgcn_ballot_w64(NEAR_LOWEST(m)) != 0) {
        if (NEAR_LOWEST(m)) {
#pragma unroll
            for (int j = 0; j < VPT; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[j][i] = shift_up(v[j][i]);
            m += LOW_SHIFT;
        }
    }
    const float negm = -m;
    const f16x2 lowest = f16x2_from_bits(0xFBFFFBFFu);
    float ek[VPT * 8];
    float z0 = 0.f, z1 = 0.f, t0 = 0.f, t1 = 0.f;
    int cnt = 0;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        if (j * LPR * 8 < nmax) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t u = bits_of(__builtin_elementwise_maximum(f16x2_from_bits(v[j][i >> 1]), lowest));
                const float s = (i & 1) ? sub_hi(u, negm) : sub_lo(u, negm);
                const float e = __builtin_amdgcn_exp2f(s * LOG2E);
                const bool at_max = s == 0.0f;
                cnt += at_max ? 1 : 0;
                if (i & 1) { z1 += at_max ? 0.0f : e; t1 = fmaf(e, s, t1); }
                else       { z0 += at_max ? 0.0f : e; t0 = fmaf(e, s, t0); }
                ek[j * 8 + i] = e;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) ek[j * 8 + i] = 0.0f;
        }
    }
    const float z = grp_sum<LPR>(z0 + z1), t = grp_sum<LPR>(t0 + t1), cz = grp_sum<LPR>((float)cnt);
    const bool mine = row0 + grp < (uint32_t)a.rows;
    if (a.p != nullptr && mine) {
        const float invZ = dead ? NAN : __builtin_amdgcn_rcpf(cz + z);
        uint16_t* pr = a.p + (int64_t)row * a.ld_p;
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            const int c0 = (j * LPR + gl) * 8;
            if (c0 >= S) continue;
            const float* ev = ek + j * 8;
            const u32x4 o{scale_pack_f16x2(ev[0], ev[1], invZ), scale_pack_f16x2(ev[2], ev[3], invZ),
                          scale_pack_f16x2(ev[4], ev[5], invZ), scale_pack_f16x2(ev[6], ev[7], invZ)};
            if (c0 + 8 <= S) {
                __builtin_nontemporal_store(o, (u32x4_u*)(pr + c0));
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (c0 + i < S) pr[c0 + i] = (uint16_t)(o[i >> 1] >> ((i & 1) * 16));
            }
        }
    }
    const float H = dead ? NAN : entropy_from(cz, z, t);
    if (gl == 0 && mine) {
        a.h[row] = H;
        if (a.tier) a.tier[row] = tier_of(H, a.tau_low, a.tau_high);
    }
}

// Any row length, any alignment: one wave per row, three passes over the row
// (max, sums, store) with 2-byte loads.  Used for rows that the vector kernels do not
// hold (S > 8 * 8 * 512).
EE_DEV void softmax_entropy_generic(const EeSoftmaxArgs& a) {
    const int lane = lane_id();
    const int64_t row = (int64_t)blockIdx.x * 4 + wave_id();
    if (row >= a.rows) return;                     // no barriers below
    const int S = a.S;
    const int nvalid = a.causal ? min(S, (int)(row % S) + 1) : S;
    const uint16_t* xr = a.x + row * a.ld_x;
    float m = -INFINITY;
    for (int c = lane; c < nvalid; c += 64) m = fmaximum(m, f16_lo(xr[c]));
    m = wave_maximum(m);
    const bool dead = !(m > -INFINITY);                // NaN or no finite entry: NaN row
    if (dead) m = 0.0f;
    float cz = 0.f, z = 0.f, t = 0.f;
    for (int c = lane; c < nvalid; c += 64) {
        const float s = fmaxf(f16_lo(xr[c]) - m, -256.0f);
        const float e = __builtin_amdgcn_exp2f(s * LOG2E);
        const bool at_max = (s == 0.0f);
        cz += at_max ? 1.0f : 0.0f;
        z += at_max ? 0.0f : e;
        t = fmaf(e, s, t);
    }
    z = wave_sum(z);
    t = wave_sum(t);
    cz = wave_sum(cz);
    const float H = dead ? NAN : entropy_from(cz, z, t);
    if (lane == 0) {
        a.h[row] = H;
        if (a.tier) a.tier[row] = tier_of(H, a.tau_low, a.tau_high);
    }
    if (a.p == nullptr) return;
    const float invZ = dead ? NAN : 1.0f / (cz + z);
    uint16_t* pr = a.p + row * a.ld_p;
    for (int c = lane; c < S; c += 64) {
        float e = 0.0f;
        if (c < nvalid) e = __builtin_amdgcn_exp2f(fmaxf(f16_lo(xr[c]) - m, -256.0f) * LOG2E);
        pr[c] = (uint16_t)pack_f16x2(e * invZ, 0.0f);
    }
}

#define EE_SE_VEC(V, W)                                                                        \
    extern "C" __global__ void __launch_bounds__(SeGeom<W>::BLOCK) eek_softmax_entropy_v##V##_w##W( \
        EeSoftmaxArgs a) {                                                                     \
        softmax_entropy_vec<V, W>(a);                                                          \
    }
// The same within 64 VGPRs, for eight waves per SIMD: with 4 vectors per lane the
// kept e values take the kernel to 65-72 VGPRs (seven waves per SIMD), and at
// [4096, 4096] (8192 waves for 7168 slots) the last 1024 waves ran as a second
// round: 15.1 -> 14.2 us cold at 63 VGPRs.  (Three, five, six and seven waves per
// row do not fit 64 without spilling and keep the plain form.)
#define EE_SE_VEC_8W(V, W)                                                                     \
    extern "C" __global__ void __launch_bounds__(SeGeom<W>::BLOCK)                             \
        __attribute__((amdgpu_waves_per_eu(8))) eek_softmax_entropy_v##V##_w##W(EeSoftmaxArgs a) { \
        softmax_entropy_vec<V, W>(a);                                                          \
    }
// Non-temporal twins of the multi-wave layouts, for logits too large to have
// stayed in cache (the launcher's choice): from HBM 3-5% faster, from the caches
// ~13% slower (configs 0-2, measured both ways).
#define EE_SE_VEC_NT(V, W, EPU)                                                                \
    extern "C" __global__ void __launch_bounds__(SeGeom<W>::BLOCK)                             \
        __attribute__((amdgpu_waves_per_eu(EPU))) eek_softmax_entropy_v##V##_w##W##_nt(EeSoftmaxArgs a) { \
        softmax_entropy_vec<V, W, true>(a);                                                    \
    }
#define EE_SE_VEC_W(V) EE_SE_VEC(V, 1) EE_SE_VEC(V, 2) EE_SE_VEC(V, 3) EE_SE_VEC(V, 4) \
                       EE_SE_VEC(V, 5) EE_SE_VEC(V, 6) EE_SE_VEC(V, 7) EE_SE_VEC(V, 8)
EE_SE_VEC_W(1)
EE_SE_VEC_W(2)
EE_SE_VEC_W(3)
EE_SE_VEC_8W(4, 1)
EE_SE_VEC_8W(4, 2)
EE_SE_VEC(4, 3)
EE_SE_VEC_8W(4, 4)
EE_SE_VEC(4, 5)
EE_SE_VEC(4, 6)
EE_SE_VEC(4, 7)
EE_SE_VEC_8W(4, 8)
// short rows, several per wave
#define EE_SE_ROWS(V, R) \
    extern "C" __global__ void __launch_bounds__(EE_BLOCK) eek_softmax_entropy_v##V##_r##R(EeSoftmaxArgs a) { \
        softmax_entropy_rows<V, R>(a);                                                                  \
    }
EE_SE_ROWS(1, 2)
EE_SE_ROWS(1, 4)
EE_SE_ROWS(2, 2)
#define EE_SE_GROUP(V, L) \
    extern "C" __global__ void __launch_bounds__(EE_BLOCK) eek_softmax_entropy_g##L##_v##V(EeSoftmaxArgs a) { \
        softmax_entropy_group<V, L>(a);                                                                 \
    }
EE_SE_GROUP(1, 16)
EE_SE_GROUP(2, 16)
EE_SE_GROUP(3, 16)
EE_SE_GROUP(4, 16)
EE_SE_GROUP(3, 32)
EE_SE_GROUP(4, 32)
// rows longer than 4 * 8 * 512: eight waves, probabilities from recomputed e
EE_SE_VEC(5, 8)
EE_SE_VEC(6, 8)
EE_SE_VEC(7, 8)
EE_SE_VEC(8, 8)
EE_SE_VEC_NT(4, 2, 8)
EE_SE_VEC_NT(4, 4, 8)
EE_SE_VEC_NT(4, 8, 8)
EE_SE_VEC_NT(5, 8, 1)
EE_SE_VEC_NT(6, 8, 1)
EE_SE_VEC_NT(7, 8, 1)
EE_SE_VEC_NT(8, 8, 1)

extern "C" __global__ void __launch_bounds__(EE_BLOCK) eek_softmax_entropy_generic(EeSoftmaxArgs a) {
    softmax_entropy_generic(a);
}
