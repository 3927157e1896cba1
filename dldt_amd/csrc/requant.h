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

__device__ __forceinline__ uint32_t requant4(const Requant& f, const float4& v) {
    return (static_cast<uint32_t>(requant_level(f, v.x)) & 0xffu) | ((static_cast<uint32_t>(requant_level(f, v.y)) & 0xffu) << 8) |
           ((static_cast<uint32_t>(requant_level(f, v.z)) & 0xffu) << 16) | (static_cast<uint32_t>(requant_level(f, v.w)) << 24);
}

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
