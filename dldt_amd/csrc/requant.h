// Per-tensor FakeQuantize to i8 levels evaluated inside the kernel that produces its input (the
// transformer glue kernels and the attention kernel).
#pragma once
#include "common.h"
#include "fq.h"

namespace hipie {

// The level index of the reference's expression (fake_quantize.hpp:175-194) by IEEE division, or by
// the reciprocal sequence when that was proven to give the same index on both sides of every level
// boundary; stored as out_low + k.  levels == 0: no quantized output.
struct Requant {
    FqChannel p;
    float lm1;
    int levels;
    int rcp;   // the reciprocal evaluation was proven equal to the division on every level boundary
};

__device__ __forceinline__ int requant_level(const Requant& f, float x) {
    // x <= il -> level 0, x > ih -> level L - 1 through the clamp
    const float k = f.rcp ? fq_level_clamped<true>(f.p, f.lm1, x) : fq_level_clamped<false>(f.p, f.lm1, x);
    return static_cast<int>(k + f.p.ol);
}

// four of them in a dword: the packing conversion rounds to the nearest level and places it (nine instructions a value instead
// of fourteen), the offset of the stored bytes is one bytewise addition
__device__ __forceinline__ uint32_t requant4(const Requant& f, const float4& v) {
    const float x[4] = {v.x, v.y, v.z, v.w};
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float n = __builtin_amdgcn_fmed3f(x[j], f.p.il, f.p.ih) - f.p.il;
        float q;
        if (f.rcp) {                                    // fq_level_rcp
            const float q0 = n * f.p.r, q1 = fmaf(fmaf(-f.p.d, q0, n), f.p.r, q0);
            q = fmaf(fmaf(-f.p.d, q1, n), f.p.r, q1);
        } else {
            q = n / f.p.d;
        }
        w = __builtin_amdgcn_cvt_pk_u8_f32(q * f.lm1, j, w);
    }
    const uint32_t off = (static_cast<uint32_t>(static_cast<int>(f.p.ol)) & 0xffu) * 0x01010101u;
    return ((w & 0x7f7f7f7fu) + (off & 0x7f7f7f7fu)) ^ ((w ^ off) & 0x80808080u);
}

// x / d for the values x of a row that share d: by the reciprocal, rounded once, with two residual corrections - the IEEE
// quotient (Markstein, as fq_level_rcp) where no intermediate leaves the range of normal numbers and x is no zero, at five
// instructions instead of eleven.  Four values with one outside [2^-60, 2^60], zeros among them, and a d outside it divide: the
// residual of smaller ones would be rounded, and -0 would lose its sign.
struct RowDivisor {
    float d, r;
    bool fast;
    static __device__ __forceinline__ bool in_range(float least, float most) { return least >= 0x1p-60f && most <= 0x1p60f; }
    __device__ __forceinline__ explicit RowDivisor(float by) : d(by), r(1.0f / by), fast(in_range(by, by)) {}
    __device__ __forceinline__ float operator()(float x) const {
        const float q0 = x * r, q1 = fmaf(fmaf(-d, q0, x), r, q0);
        return fmaf(fmaf(-d, q1, x), r, q1);
    }
    __device__ __forceinline__ float4 operator()(const float4& v) const {
        const float x = fabsf(v.x), y = fabsf(v.y), z = fabsf(v.z), w = fabsf(v.w);
        if (fast && in_range(fminf(fminf(x, y), fminf(z, w)), fmaxf(fmaxf(x, y), fmaxf(z, w))))
            return make_float4((*this)(v.x), (*this)(v.y), (*this)(v.z), (*this)(v.w));
        return make_float4(v.x / d, v.y / d, v.z / d, v.w / d);
    }
};

// Host side: checks that the reference's output expression yields the integers out_low + k and picks
// the evaluation of the level index.
inline Requant make_requant(const hipie_requant* r, const char* what) {
    Requant f{};
    if (!r) return f;
    HIPIE_REQUIRE(r->levels >= 2 && r->levels <= 256 && r->in_low < r->in_high, HIPIE_PARAMETER_MISMATCH,
                  "%s: requantisation needs 2..256 levels and in_low < in_high", what);
    f.p.il = f.p.lo = r->in_low;
    f.p.ih = f.p.hi = r->in_high;
    f.p.d = r->in_high - r->in_low;
    f.p.r = fq_rounded_reciprocal(f.p.d);
    f.lm1 = static_cast<float>(r->levels - 1);
    f.p.ol = r->out_low;
    f.p.oh = r->out_low + f.lm1;
    f.levels = static_cast<int>(r->levels);
    f.rcp = fq_reciprocal_exact_on_boundaries(f.p, f.lm1) ? 1 : 0;
    const float oh = f.p.oh;
    HIPIE_REQUIRE(f.p.ol == std::nearbyintf(f.p.ol) && f.p.ol >= -128.f && oh <= 127.f, HIPIE_NOT_IMPLEMENTED,
                  "%s: output levels must be the i8 integers out_low .. out_low + levels - 1", what);
    for (int k = 0; k < f.levels; ++k)   // the reference's own output expression yields these integers
        HIPIE_REQUIRE(static_cast<float>(k) / f.lm1 * (oh - f.p.ol) + f.p.ol == f.p.ol + static_cast<float>(k),
                      HIPIE_NOT_IMPLEMENTED, "%s: output level %d is not an integer", what, k);
    return f;
}

// Softmax, MVN (LayerNorm) and Gelu over dense f32 rows (glue.hip): f32 result y, i8 levels q by `r`, either may be null.  A
// plan keeps its Requant: make_requant compares the reciprocal form with the division on every level boundary, 28 us of host
// time, and an encoder has two a layer: 3 layers of 8 x 128 tokens, three requests in flight, 239.7 us a pass with a check in
// each call, 99.9 without.
void run_softmax(const float* x, float* y, int8_t* q, int64_t rows, int64_t axis, const Requant* r, hipStream_t s, const char* what);
void run_mvn(const float* x, float* y, int8_t* q, int64_t rows, int64_t axis, int normalize_variance, float eps, int eps_inside_sqrt, const float* gamma,
             const float* beta, const Requant* r, hipStream_t s, const char* what);
void run_gelu(const float* x, float* y, int8_t* q, int64_t n, const Requant* r, hipStream_t s, const char* what);

}  // namespace hipie
