// Argument block of the attention core and the requantisation of its probabilities, shared by the attention kernel and
// the single-launch program.
#pragma once
#include "conv_epilogue.h"
#include "requant.h"

namespace hipie {

struct AttentionArgs {
    const int8_t *q, *k, *v;
    int64_t ldq, sq, oq, ldk, sk, ok, ldv, sv, ov;   // row pitch, inner / outer batch stride (bytes)
    void* out;
    int64_t ldo, so, oo;                              // elements
    const float* mask;                                // optional additive mask row [S] per batch element, or null
    int64_t mask_inner, mask_outer;                   // its batch strides (elements)
    float* scores;                                    // optional [batch][S][S] dumps (inspection), or null
    float* probs;
    int S, batch_inner;
    float scale1, scale2;
    Requant fq_p, fq_o;                               // fq_o.levels == 0: f32 output
    float p_zh, p_zl;                                 // probabilities: two-operation division by fq_p.p.d
    int p_div2;                                       // ... verified against IEEE division on the device
    int p_sat;                                        // input_low of the probabilities' FakeQuantize is +0 and it has 256 levels
    int p_inside;                                     // ... or input_low <= 0 and input_high >= 1: a probability never leaves the interval
    int qblocks;                                      // workgroups (128 queries, beyond kPlainSoftmax keys 64) per batch element
    int xcd_groups;                                   // 1: a one-dimensional grid that keeps the blocks of two neighbouring batch elements on one XCD
#ifdef HIPIE_ATT_STAMPS
    long long* stamps;                                // probe builds only: cycle stamps per workgroup
#endif
    uint32_t p_xor, p_add;                            // stored byte = level + out_low (mod 256): XOR 0x80 per byte, or bytewise add
    int p_bias;                                       // 128 when the probabilities are u8 levels (stored as level - 128), else 0
};

// level index k of four probabilities as four unsigned bytes (rounded to nearest-even and packed by
// v_cvt_pk_u8_f32), then the output offset applied bytewise
// PFORM 2: input_low is +0 and there are 256 levels - a probability is never below input_low, and the packing
// conversion's saturation at 255 is the branch for values above input_high: no clamp, no subtraction.
// PFORM 1: input_low <= 0 and input_high >= 1 - a probability (0 <= e / sum <= 1: the largest e is 2^0 and counted in
// the sum) takes neither of the reference's saturating branches: no clamp.  PFORM 0: any interval.
template <bool DIV2, int PFORM>
__device__ __forceinline__ uint32_t prob_levels4(const AttentionArgs& a, float p0, float p1, float p2, float p3) {
    const FqChannel& c = a.fq_p.p;
    constexpr int M = DIV2 ? 2 : 1;
    constexpr bool IL0 = PFORM == 2, NOCLAMP = PFORM != 0;
    uint32_t w = 0;
    w = __builtin_amdgcn_cvt_pk_u8_f32(fq_level_fast<M, IL0, NOCLAMP>(p0, c.il, c.ih, c.d, DIV2 ? a.p_zh : c.r, a.p_zl, a.fq_p.lm1), 0, w);
    w = __builtin_amdgcn_cvt_pk_u8_f32(fq_level_fast<M, IL0, NOCLAMP>(p1, c.il, c.ih, c.d, DIV2 ? a.p_zh : c.r, a.p_zl, a.fq_p.lm1), 1, w);
    w = __builtin_amdgcn_cvt_pk_u8_f32(fq_level_fast<M, IL0, NOCLAMP>(p2, c.il, c.ih, c.d, DIV2 ? a.p_zh : c.r, a.p_zl, a.fq_p.lm1), 2, w);
    w = __builtin_amdgcn_cvt_pk_u8_f32(fq_level_fast<M, IL0, NOCLAMP>(p3, c.il, c.ih, c.d, DIV2 ? a.p_zh : c.r, a.p_zl, a.fq_p.lm1), 3, w);
    return a.p_add ? add_bytes(w, a.p_add) : (w ^ a.p_xor);
}

// 4 x 4 byte transpose: t[e] = bytes e of p0 .. p3
__device__ __forceinline__ void transpose_bytes(uint32_t p0, uint32_t p1, uint32_t p2, uint32_t p3, uint32_t (&t)[4]) {
    const uint32_t lo01 = __builtin_amdgcn_perm(p1, p0, 0x05010400u), hi01 = __builtin_amdgcn_perm(p1, p0, 0x07030602u);      // p0.b0 p1.b0 p0.b1 p1.b1 ...
    const uint32_t lo23 = __builtin_amdgcn_perm(p3, p2, 0x05010400u), hi23 = __builtin_amdgcn_perm(p3, p2, 0x07030602u);
    t[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
    t[1] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
    t[2] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
    t[3] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
}

// Rows longer than this have the Softmax of the stand-alone kernel bit for bit (softmax_rows_reg: exp(x - max), sums of
// four keys, the chunks of 256 keys, then a tree over the groups of four), so that their levels do not depend on whether
// the core is one kernel.  Up to it exp2 of one fused multiply-add, a serial sum and the reciprocal, within the same
// tolerance: a third of the instructions.
constexpr int kPlainSoftmax = 384;

// e / sum rounded once, from inv = 1 / sum rounded once: quotient, exact residual, correction.  Equal to the IEEE
// quotient for e in [2^-60, 1] and sum in [1, 1024): tests/test_quotient_cpu.py derives which pairs of significands could round
// the other way and compares all of them.  Below that range of e the level is that of zero.
__device__ __forceinline__ float quotient(float e, float sum, float inv) {
    const float q = e * inv;
    return fmaf(fmaf(-q, sum, e), inv, q);
}

}  // namespace hipie

struct hipie_attention;
namespace hipie {
// everything of the kernel's arguments but the operands
const AttentionArgs& attention_prototype(const hipie_attention* att);
}  // namespace hipie
