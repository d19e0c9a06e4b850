// ee_softmax_dev.h -- the arithmetic of a softmax row that the softmax + entropy kernels and the
// fused attention share: the same bits of p and the same form of H in both.
#pragma once
#include "ee_device.h"

#define LOG2E 1.4426950408889634f
#define LN2 0.69314718055994531f

// ln x for x >= 1: v_log_f32 (log2, within 1 ulp of the result) times ln 2.
EE_DEV float ln_ge1(float x) { return __builtin_amdgcn_logf(x) * LN2; }
// log1p(x) for x >= 0 (Goldberg): u = 1 + x; x ln(u) / (u - 1) with u - 1 exact,
// which cancels u's rounding, or x where u rounds to 1.  A few ulps relative.
EE_DEV float log1p_ge0(float x) {
    const float u = 1.0f + x;
    return u == 1.0f ? x : ln_ge1(u) * (x * __builtin_amdgcn_rcpf(u - 1.0f));
}
// Entropy from the reduced partial sums (softmax_entropy.hip says why in this form): c0 >= 1 counts the
// entries at the max, z >= 0, t <= 0, so every term is >= 0; the quotients take
// v_rcp_f32 (1 ulp).  Within ~1e-6 relative of the libm form (logf, log1pf and
// IEEE divisions: ~120 dependent instructions, evaluated once per row).
EE_DEV float entropy_from(float c0, float z, float t) {
    return ln_ge1(c0) + log1p_ge0(z * __builtin_amdgcn_rcpf(c0)) - t * __builtin_amdgcn_rcpf(c0 + z);
}

// s = x - m for the low / high fp16 half of a packed word: one v_fma_mix_f32
// (x * 1 + (-m), a single rounding, the same value as converting x and then
// subtracting).
EE_DEV float sub_lo(uint32_t u, float negm) {
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(u), "v"(negm));
    return r;
}
EE_DEV float sub_hi(uint32_t u, float negm) {
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(u), "v"(negm));
    return r;
}
// fp16(e0 * s) | fp16(e1 * s) << 16, each product rounded once to fp16
// (v_fma_mixlo_f16 / v_fma_mixhi_f16 with a zero addend).
EE_DEV uint32_t scale_pack_f16x2(float e0, float e1, float s) {
    uint32_t r;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(r) : "v"(e0), "v"(s));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(r) : "v"(e1), "v"(s));
    return r;
}
