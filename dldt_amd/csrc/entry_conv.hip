// A FakeQuantize on a graph input and the convolution behind it, whose f32 values are the graph's result, in one launch: f32 (or u8)
// [N, C, H, W] in, f32 [N, OC, H, W] out, and the levels between them into their own tensor for whoever else reads them.
//
// What bounds the two layers apart is not their work (12 x 72 x 45 x 45 to 100 channels: 17 MB and 2.8 GOP, 2.7 us at the
// rates of this device) but two dependent launches: 2.7 us of host time each, and a cold start on either side.
//
// A workgroup owns R whole rows of one image and walks groups of 32 wo output channels.  It requests the f32 rows under them - a
// wave's load is 64 neighbouring values of a channel - quantises them into an LDS patch [row][column][channel] with the padding
// around it, and the waves multiply from there by v_mfma_i32_32x32x32_i8: weights as rows, packed in fragment order (1 KB a load,
// straight into operand registers, requested two K steps of four ahead), 32 neighbouring pixels as columns, so that a value's 32
// lanes store 128 contiguous bytes of a channel's plane.  Rows that two workgroups share are quantised by both, and every channel
// group of blockIdx.y quantises the patch again: 1.2 - 3 times the work of a FakeQuantize that is bound by its loads, which L2 serves.
//
// Measured, us, as two launches and as one (three requests in flight; one launch behind the other): 12 x 72 x 45 x 45 to 100 9.5 / 16.2
// and 7.5 / 15.1 (6.3 tuned against 8.4, by a caller that waits at the end only); 1 x 64 x 56 x 56 to 64 7.0 / 14.4 and 4.0 / 8.1;
// 24 x 40 x 20 x 20 to 90 7.3 / 13.6 and 4.2 / 7.3; 32 x 256 x 7 x 7 to 512 9.7 / 21.5 and 9.9 / 14.3; 2 x 8 x 107 x 107 to 301
// 9.8 / 18.3 and 9.8 / 16.1.  4.0 is what the call and one launch cost the host.  Large layers of many channels stay two launches.
// Of a workgroup's 8.7 us for the first of these 3.7 are the way to the patch (1.5 until the requests are out, the rest latency and 45
// instructions an item, which two workgroups of a unit wait for together), 2.6 the sums, 1.2 - 2 the values' way out.
// Reference semantics: as fq.hip and conv_epilogue.h, the same f32 operations in the same order.
#include <memory>
#include <type_traits>

#include "conv.h"
#include "conv_epilogue.h"
#include "conv_dispatch.h"
#include "entry_conv.h"
#include "fq.h"

namespace hipie {
namespace {

constexpr int kThreads = 512, kWaves = kThreads / 64;
constexpr int kMostFragments = 2;            // of 32 pixels that a wave multiplies (104 registers, 110 with BOTH: two workgroups a compute unit; three fragments take 140)
constexpr int kAhead = 4;                    // K steps of 32 bytes in a group: one is multiplied while the next one's weights come

struct Args {
    const void* x;
    const FqChannel* tab;
    float lm1, off;
    uint8_t* levels;                         // of pixel (0, 0, 0), channel 0
    int64_t lv_sn;
    int32_t lv_sh, cs;                       // bytes from row to row and from pixel to pixel
    const int8_t* wgt;                       // [32 channels][K step of 32 bytes][lane] x 16 bytes
    const int32_t* corr;
    const float *bias, *scale;
    float* out;
    float* tensor;                           // (BOTH) the values channels innermost as well
    int64_t t_sn, t_sh;
    int32_t t_sw;                            // its strides in elements: image, row, pixel
    int32_t C, H, W, HW, OC;
    int32_t kh, kw, pad_h, pad_w;
    int32_t R, row_tiles, tiles, per_xcd;    // rows of a tile, tiles of an image and of all, of an XCD
    int32_t PW, pcs;                         // patch: pixels of a row, bytes of a pixel
    int32_t koff_at, chan_at, tables_at;     // where the tables are in LDS: K offsets, input channels, output channels
    int32_t steps, pieces;                   // K steps (a multiple of kAhead), 16-byte pieces of K that exist
    int32_t o_groups, wo_shift;              // groups of 32 << wo_shift output channels; log2 of the waves side by side in channels
    uint32_t flags, fill;                    // fill: four bytes of the padding's level
    float clamp_lo, clamp_hi, inv_W;
};

typedef uint32_t v4u __attribute__((ext_vector_type(4)));
#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t Buffer;
__device__ __forceinline__ Buffer make_buffer(void* p, uint32_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(p, 0, static_cast<int>(bytes), 0x00020000); }
__device__ __forceinline__ void store4(Buffer b, uint32_t o, float v) { __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v), b, static_cast<int>(o), 0, 0); }
#else
typedef void* Buffer;
__device__ __forceinline__ Buffer make_buffer(void* p, uint32_t) { return p; }
__device__ __forceinline__ void store4(Buffer, uint32_t, float) {}
#endif

// PF: fragments of 32 pixels a wave multiplies; U8: bytes in; SMALL: pixels of four bytes (rows of taps contiguous, 4-byte aligned);
// BOTH: the values into a.tensor as well (its instructions beside the others' cost 12 x 72 x 45 x 45 to 100 1 %, taken or not)
template <int PF, bool U8, bool SMALL, bool BOTH>
__global__ __launch_bounds__(kThreads, 4) void entry_conv_kernel(const Args a) {
    extern __shared__ __attribute__((aligned(16))) int8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // neighbouring tiles share rows: each XCD takes a contiguous run of them
    const int tile = static_cast<int>(blockIdx.x & 7) * a.per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (tile >= a.tiles) return;
    const int n = tile / a.row_tiles, y0 = (tile - n * a.row_tiles) * a.R;
    const int rows = min(a.R, a.H - y0), count = rows * a.W;
    int32_t* const koff = reinterpret_cast<int32_t*>(lds + a.koff_at);          // [half][step]
    float4* const chan = reinterpret_cast<float4*>(lds + a.chan_at);            // il, ih, d, r

    float* const bias = reinterpret_cast<float*>(lds + a.tables_at);
    // the first group's weights, on their way before anything else
    const int l32 = lane & 31, h = lane >> 5, wo = 1 << a.wo_shift, wp = kWaves >> a.wo_shift;
    const int o_wave = wave & (wo - 1), p_wave = wave >> a.wo_shift, o_tiles = (a.OC + 31) / 32;
    float* const scale = bias + 32 * o_tiles;
    auto weights = [&](int og) { return a.wgt + (static_cast<int64_t>(min(og * wo + o_wave, o_tiles - 1)) * a.steps * 1024 + lane * 16); };
    const int8_t* wp0 = weights(blockIdx.y);
    v4i w[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) w[k] = *reinterpret_cast<const v4i*>(wp0 + k * 1024);

    // the input rows under the patch that exist: contiguous in every channel
    const int iy0 = max(y0 - a.pad_h, 0), iy1 = min(y0 + rows + a.kh - 1 - a.pad_h, a.H), values = (iy1 - iy0) * a.W;
    const int row0 = iy0 - (y0 - a.pad_h);                                       // their first row in the patch
    const int c4s = a.cs / 4, items = (values + 63) / 64 * c4s;
    const int64_t image = static_cast<int64_t>(n) * a.C * a.HW + static_cast<int64_t>(iy0) * a.W;
    typedef typename std::conditional<U8, uint8_t, float>::type In;
    const In* const x = static_cast<const In*>(a.x) + image;
    // An item: four channels of 64 neighbouring values.  A wave takes every eighth, channels first, U of them in flight.  (Where it
    // is goes along by additions, and a lane's place by a branch where the values change: divisions in every item were a third of
    // its instructions.)
    constexpr int U = 8;
    float v[U][4];
    int ask_c4 = wave, ask_at = 0;                                               // the item that is requested next: channel quad, first value
    uint32_t from = static_cast<uint32_t>(min(lane, values - 1));
    auto request = [&](float (&to)[4]) {
        if (ask_c4 >= c4s) {
            do {
                ask_c4 -= c4s;
                ask_at += 64;
            } while (ask_c4 >= c4s);
            from = static_cast<uint32_t>(min(ask_at + lane, values - 1));        // (behind the last value: there, and not stored)
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const In* const channel = x + static_cast<int64_t>(min(4 * ask_c4 + j, a.C - 1)) * a.HW;
            to[j] = static_cast<float>(channel[from]);
        }
        ask_c4 += kWaves;
    };
#pragma unroll
    for (int u = 0; u < U; ++u) request(v[u]);
    for (int i = tid; i < a.cs; i += kThreads) {                                 // (channels that do not exist: level 0 of any value)
        const FqChannel p = a.tab[min(i, a.C - 1)];
        chan[i] = i < a.C ? make_float4(p.il, p.ih, p.d, p.r) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    for (int i = tid; i < 32 * o_tiles; i += kThreads) {
        if (a.flags & CF_BIAS) bias[i] = a.bias[i];
        if (a.flags & CF_SCALE) scale[i] = a.scale[i];
    }
    for (int i = tid; i < 2 * a.steps; i += kThreads) {
        const int half = i >= a.steps ? 1 : 0, piece = min(2 * (i - half * a.steps) + half, a.pieces - 1);      // (behind the last: zero weights)
        int32_t o;
        if constexpr (SMALL) {
            const int per = (4 * a.kw + 15) / 16;
            o = (piece / per) * a.PW * 4 + (piece % per) * 16;
        } else {
            const int tap = piece / (a.cs / 16);
            o = ((tap / a.kw) * a.PW + tap % a.kw) * a.pcs + (piece - tap * (a.cs / 16)) * 16;
        }
        koff[i] = o;
    }
    for (int i = tid * 16; i < a.koff_at; i += kThreads * 16) *reinterpret_cast<v4u*>(lds + i) = v4u{a.fill, a.fill, a.fill, a.fill};
    __syncthreads();
    // (a packed conversion rounds a level and puts it in its byte; the offset of the stored bytes is one bytewise addition)
    const uint32_t off = (static_cast<uint32_t>(static_cast<int>(a.off)) & 0xffu) * 0x01010101u;
    int c4 = wave, first = 0, place = 0;
    bool on = false;
    auto locate = [&] {
        int y, xx;
        on = first + lane < values;
        fast_divmod(min(first + lane, values - 1), a.W, a.inv_W, y, xx);
        place = ((row0 + y) * a.PW + a.pad_w + xx) * a.pcs;
    };
    locate();
    for (int i0 = wave; i0 < items; i0 += kWaves * U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (i0 + kWaves * u >= items) break;
            if (c4 >= c4s) {
                do {
                    c4 -= c4s;
                    first += 64;
                } while (c4 >= c4s);
                locate();
            }
            uint32_t dw = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float4 t = chan[4 * c4 + j];                               // il, ih, d, r: fq_level_clamped
                const float d = __builtin_amdgcn_fmed3f(v[u][j], t.x, t.y) - t.x;
                const float q0 = d * t.w, q1 = fmaf(fmaf(-t.z, q0, d), t.w, q0), q = fmaf(fmaf(-t.z, q1, d), t.w, q1);
                dw = __builtin_amdgcn_cvt_pk_u8_f32(q * a.lm1, j, dw);
            }
            if (on) *reinterpret_cast<uint32_t*>(lds + place + 4 * c4) = add_bytes(dw, off);
            c4 += kWaves;
            if (i0 + kWaves * (u + U) < items) request(v[u]);
        }
    }
    __syncthreads();

    // the levels of the tile's own rows, pixel by pixel
    if (blockIdx.y == 0) {
        const int unit = SMALL ? 4 : 16, per = a.cs / unit;
        for (int i = tid; i < count * per; i += kThreads) {
            const int m = SMALL ? i : i / per, q = i - m * per;
            int y, xx;
            fast_divmod(m, a.W, a.inv_W, y, xx);
            const int8_t* from = lds + ((y + a.pad_h) * a.PW + a.pad_w + xx) * a.pcs + unit * q;
            uint8_t* to = a.levels + static_cast<int64_t>(n) * a.lv_sn + static_cast<int64_t>(y0 + y) * a.lv_sh + xx * a.cs + unit * q;
            if constexpr (SMALL) *reinterpret_cast<uint32_t*>(to) = *reinterpret_cast<const uint32_t*>(from);
            else *reinterpret_cast<v4u*>(to) = *reinterpret_cast<const v4u*>(from);
        }
    }

    int base[PF];
#pragma unroll
    for (int f = 0; f < PF; ++f) {
        int y, xx;
        fast_divmod(min((p_wave + f * wp) * 32 + l32, count - 1), a.W, a.inv_W, y, xx);
        base[f] = (y * a.PW + xx) * a.pcs;
    }
    const int32_t* const ko = koff + h * a.steps;
    float* const out = a.out + (static_cast<int64_t>(n) * a.OC * a.HW + static_cast<int64_t>(y0) * a.W);
    for (int og = blockIdx.y; og < a.o_groups; og += gridDim.y) {
        const int oc0 = min((og * wo + o_wave) * 32, 32 * o_tiles - 32) + 4 * h;
        if (og != static_cast<int>(blockIdx.y)) {
            wp0 = weights(og);
#pragma unroll
            for (int k = 0; k < kAhead; ++k) w[k] = *reinterpret_cast<const v4i*>(wp0 + k * 1024);
        }
        v16i acc[PF];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const v4i c = *reinterpret_cast<const v4i*>(a.corr + oc0 + 8 * q);
#pragma unroll
            for (int f = 0; f < PF; ++f)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[f][4 * q + j] = c[j];
        }
        auto multiply = [&](const v4i (&wt)[kAhead], int k0) {
            const v4i o4 = *reinterpret_cast<const v4i*>(ko + k0);
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {
#pragma unroll
                for (int f = 0; f < PF; ++f) {
                    const int8_t* p = lds + base[f] + o4[k];
                    v4i px;
                    if constexpr (SMALL) {
                        const int32_t* d = reinterpret_cast<const int32_t*>(p);
                        px = v4i{d[0], d[1], d[2], d[3]};
                    } else px = *reinterpret_cast<const v4i*>(p);
                    acc[f] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wt[k], px, acc[f], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        for (int k0 = 0; k0 < a.steps; k0 += kAhead) {
            v4i next[kAhead];
            const int at = min(k0 + kAhead, a.steps - kAhead) * 1024;
#pragma unroll
            for (int k = 0; k < kAhead; ++k) next[k] = *reinterpret_cast<const v4i*>(wp0 + at + k * 1024);
            multiply(w, k0);
#pragma unroll
            for (int k = 0; k < kAhead; ++k) w[k] = next[k];
        }
        const int left = a.OC - (og * wo + o_wave) * 32;                         // channels from here on
        if (left <= 0) continue;
        const Buffer plane = make_buffer(out + static_cast<int64_t>((og * wo + o_wave) * 32) * a.HW, static_cast<uint32_t>(min(left, 32)) * static_cast<uint32_t>(a.HW) * 4u);
#pragma unroll
        for (int f = 0; f < PF; ++f) {
            const int m = (p_wave + f * wp) * 32 + l32;
            float r[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) r[i] = static_cast<float>(acc[f][i]);
            if (a.flags & CF_BIAS) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 t = ld4f(bias + oc0 + 8 * q);
                    r[4 * q] += t.x; r[4 * q + 1] += t.y; r[4 * q + 2] += t.z; r[4 * q + 3] += t.w;
                }
            }
            if (a.flags & CF_SCALE) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 t = ld4f(scale + oc0 + 8 * q);
                    r[4 * q] *= t.x; r[4 * q + 1] *= t.y; r[4 * q + 2] *= t.z; r[4 * q + 3] *= t.w;
                }
            }
            if (a.flags & CF_RELU) {
#pragma unroll
                for (int i = 0; i < 16; ++i) r[i] = r[i] > 0.0f ? r[i] : 0.0f;
            }
            if (a.flags & CF_CLAMP) {
#pragma unroll
                for (int i = 0; i < 16; ++i) r[i] = r[i] < a.clamp_lo ? a.clamp_lo : (r[i] > a.clamp_hi ? a.clamp_hi : r[i]);
            }
            if constexpr (BOTH) {
                int y, xx;
                fast_divmod(min(m, count - 1), a.W, a.inv_W, y, xx);
                const int oc = (og * wo + o_wave) * 32 + 4 * h;
                float* const t = a.tensor + n * a.t_sn + (y0 + y) * a.t_sh + static_cast<int64_t>(xx) * a.t_sw + oc;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (m < count && oc + 8 * q + 4 <= a.t_sw) *reinterpret_cast<float4*>(t + 8 * q) = make_float4(r[4 * q], r[4 * q + 1], r[4 * q + 2], r[4 * q + 3]);
            }
            // (offsets beyond the plane's records store nothing: pixels behind the tile, channels behind the last)
            uint32_t to = m < count ? 4u * (static_cast<uint32_t>(4 * h) * static_cast<uint32_t>(a.HW) + static_cast<uint32_t>(m)) : 0x80000000u;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                store4(plane, to, r[i] + 0.f);                                   // (as a result that is copied out: no negative zero)
                to += (i & 3) == 3 ? 20u * static_cast<uint32_t>(a.HW) : 4u * static_cast<uint32_t>(a.HW);
            }
            __builtin_amdgcn_sched_barrier(0);                                   // (one fragment after the other: registers)
        }
    }
}

// constant weights [OCp][Kp] in the per-layer kernels' row order -> [32 channels][K step][lane] x 16 bytes
__global__ __launch_bounds__(256) void pack_entry_kernel(const int8_t* __restrict__ w, int8_t* __restrict__ f, int OCp, int Kp, int steps, int64_t pieces) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= pieces) return;
    const int l = static_cast<int>(i & 63), k = static_cast<int>((i >> 6) % steps), o = static_cast<int>((i >> 6) / steps);
    const int oc = 32 * o + (l & 31), at = 32 * k + 16 * (l >> 5);
    uint4 v = make_uint4(0, 0, 0, 0);
    if (oc < OCp && at < Kp) {
        const int e = oc & 63;
        const int row = (oc & ~63) + 32 * ((e >> 4) & 1) + 8 * ((e >> 2) & 3) + 4 * (e >> 5) + (e & 3);
        v = *reinterpret_cast<const uint4*>(w + static_cast<int64_t>(row) * Kp + at);
    }
    reinterpret_cast<uint4*>(f)[i] = v;
}

}  // namespace

struct EntryConv {
    Args a{};
    int device = 0, pf = 0, groups_y = 1;
    bool u8 = false, small = false;
    size_t lds = 0;
    DeviceBuffer weights;
};

namespace {

// The kernel's shape: rows of a tile, waves side by side in channels, workgroups that share a tile's channels, by the microseconds of
// a launch.  The constants are fitted to 673 shapes of 21 layers (1 - 32 images of 7 x 7 to 112 x 112, 3 - 256 channels to 8 - 512,
// one launch behind the other): over these the choice costs 1.2 % against the best shape of every layer.
struct Shape { int R, wo_shift, pf, gy; size_t lds; };

size_t lds_bytes(const Args& a, int R, int* koff_at, int* chan_at, int* tables_at) {
    const int rows = R + a.kh - 1;
    *koff_at = static_cast<int>(round_up(static_cast<int64_t>(rows) * a.PW * a.pcs + 64, 16));      // (pixels of four bytes: a row's last pieces read beyond it)
    *chan_at = static_cast<int>(round_up(*koff_at + 2 * a.steps * 4, 16));
    *tables_at = *chan_at + a.cs * 16;
    return static_cast<size_t>(*tables_at) + static_cast<size_t>((a.OC + 31) / 32) * 32 * 8;
}

Shape choose_shape(const Args& a, int images, int units) {
    Shape best{};
    double best_t = 1e30;
    const int o_tiles = (a.OC + 31) / 32;
    for (int R = 1; R <= a.H && (R == 1 || static_cast<int64_t>(R) * a.W <= 32 * kWaves * kMostFragments); ++R) {
        int k, c, t;
        const size_t lds = lds_bytes(a, R, &k, &c, &t);
        if (lds > 160 * 1024) break;
        const int64_t tiles = static_cast<int64_t>(images) * ((a.H + R - 1) / R);
        const int values = std::min(R + a.kh - 1, a.H) * a.W, frags = (R * a.W + 31) / 32, places = lds > 80 * 1024 ? 1 : 2;
        const double items = static_cast<double>((values + 63) / 64) * (a.cs / 4);
        for (int s = 0; s <= 3; ++s) {
            const int wo = 1 << s, wp = kWaves / wo, pf = (frags + wp - 1) / wp, groups = (o_tiles + wo - 1) / wo;
            if (pf > kMostFragments) continue;
            for (int gy = 1; gy <= groups; ++gy) {
                const double load = static_cast<double>(tiles * gy) / units, rounds = std::ceil(load / places), side = std::min<double>(places, std::ceil(load));
                const double stage = std::max(1.57 + 0.23 * std::ceil(items / kWaves), side * 0.0325 * items);
                const double group = a.steps * std::max(0.031, side * pf * 0.0586) + 0.21 + 0.62 * pf * side;
                const double us = rounds * (stage + (groups + gy - 1) / gy * group) + 0.46 * (rounds - 1) + 3.3;
                if (us < best_t) {
                    best_t = us;
                    best = {R, s, pf, gy, lds};
                }
            }
        }
    }
    return best;
}

template <int PF, bool BOTH>
const void* kernel_of(bool u8, bool small) {
    if (u8) return small ? reinterpret_cast<const void*>(&entry_conv_kernel<PF, true, true, BOTH>) : reinterpret_cast<const void*>(&entry_conv_kernel<PF, true, false, BOTH>);
    return small ? reinterpret_cast<const void*>(&entry_conv_kernel<PF, false, true, BOTH>) : reinterpret_cast<const void*>(&entry_conv_kernel<PF, false, false, BOTH>);
}
const void* kernel_of(const EntryConv& e, bool both) {
    if (both) return e.pf == 1 ? kernel_of<1, true>(e.u8, e.small) : kernel_of<kMostFragments, true>(e.u8, e.small);
    return e.pf == 1 ? kernel_of<1, false>(e.u8, e.small) : kernel_of<kMostFragments, false>(e.u8, e.small);
}

}  // namespace

std::shared_ptr<EntryConv> make_entry_conv(int device, const hipie_fq* fq, bool u8_in, const hipie_conv* conv, const hipie_tensor& mid, const hipie_tensor& out, int fill) {
    FqLaunch f;
    ConvLaunch l;
    hipie_tensor in = mid, to = out;
    in.data = to.data = reinterpret_cast<void*>(uintptr_t(4096));       // (only the shapes are looked at)
    if (!fq || !conv || !fq_launch_arguments(fq, mid.dtype, f) || !f.rcp || f.channels != mid.c || !conv_launch_arguments(conv, in, nullptr, to, l)) return nullptr;
    const ConvArgs& c = l.a;
    constexpr uint32_t kTakes = CF_BIAS | CF_SCALE | CF_RELU | CF_CLAMP;
    if (l.depthwise || c.koff_tile || (c.flags & ~kTakes) || out.dtype != HIPIE_F32) return nullptr;
    if (l.dil_h != 1 || l.dil_w != 1 || c.conv_sh != 1 || c.conv_sw != 1 || l.kh > 7 || l.kw > 7 || l.kh % 2 == 0 || l.kw % 2 == 0) return nullptr;
    if (l.pad_top != l.kh / 2 || l.pad_left != l.kw / 2 || out.h != mid.h || out.w != mid.w || out.n != mid.n) return nullptr;
    const int64_t cs = mid.stride_w, hw = static_cast<int64_t>(mid.h) * mid.w;
    if (mid.n < 1 || (cs != 4 && cs % 16 != 0) || cs > 1024 || mid.c > cs || mid.c * hw >= (1 << 29) || hw >= (1 << 24) || mid.stride_h >= (1ll << 31) || out.c < 1) return nullptr;
    auto e = std::make_shared<EntryConv>();
    e->device = device;
    e->u8 = u8_in;
    e->small = cs == 4;
    Args& a = e->a;
    a.tab = f.table;
    a.lm1 = f.lm1;
    a.off = f.off;
    a.lv_sn = mid.stride_n;
    a.lv_sh = static_cast<int32_t>(mid.stride_h);
    a.cs = static_cast<int32_t>(cs);
    a.corr = c.corr;
    a.bias = c.bias;
    a.scale = c.scale;
    a.C = mid.c; a.H = mid.h; a.W = mid.w; a.HW = static_cast<int32_t>(hw); a.OC = out.c;
    a.kh = l.kh; a.kw = l.kw; a.pad_h = l.pad_top; a.pad_w = l.pad_left;
    a.PW = mid.w + l.kw - 1;
    a.pcs = e->small ? 4 : static_cast<int32_t>(cs / 16 % 2 ? cs : cs + 16);      // an odd number of 16-byte pieces: neighbouring pixels in different banks
    a.pieces = static_cast<int32_t>(e->small ? static_cast<int64_t>(l.kh) * (round_up(4 * l.kw, 16) / 16) : static_cast<int64_t>(l.kh) * l.kw * cs / 16);
    a.steps = static_cast<int32_t>(round_up(ceil_div(a.pieces, 2), kAhead));
    if (16 * a.pieces > c.Kp) return nullptr;
    a.flags = c.flags;
    a.clamp_lo = c.clamp_lo;
    a.clamp_hi = c.clamp_hi;
    a.fill = (static_cast<uint32_t>(fill) & 0xffu) * 0x01010101u;
    a.inv_W = 1.0f / static_cast<float>(mid.w);
    int units = 0;
    HIPIE_CHECK_HIP(hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device));
    const Shape s = choose_shape(a, mid.n, units);
    if (s.R == 0) return nullptr;
    a.R = s.R;
    a.wo_shift = s.wo_shift;
    a.row_tiles = static_cast<int32_t>(ceil_div(a.H, a.R));
    const int64_t tiles = static_cast<int64_t>(mid.n) * a.row_tiles;
    if (tiles >= (1 << 24)) return nullptr;
    a.tiles = static_cast<int32_t>(tiles);
    a.per_xcd = static_cast<int32_t>(ceil_div(tiles, 8));
    e->lds = lds_bytes(a, a.R, &a.koff_at, &a.chan_at, &a.tables_at);
    const int64_t o_tiles = ceil_div(a.OC, 32);
    a.o_groups = static_cast<int32_t>(ceil_div(o_tiles, 1 << a.wo_shift));
    e->pf = s.pf;
    e->groups_y = s.gy;
    DeviceGuard g(device);
    for (bool both : {false, true}) HIPIE_CHECK_HIP(hipFuncSetAttribute(kernel_of(*e, both), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    const int64_t pieces = o_tiles * a.steps * 64;
    e->weights.alloc(device, static_cast<size_t>(pieces) * 16);
    hipLaunchKernelGGL(pack_entry_kernel, dim3(static_cast<uint32_t>(ceil_div(pieces, 256))), dim3(256), 0, nullptr, c.wgt, e->weights.as<int8_t>(), c.OCp, c.Kp, a.steps, pieces);
    HIPIE_CHECK_HIP(hipGetLastError());
    HIPIE_CHECK_HIP(hipStreamSynchronize(nullptr));
    a.wgt = e->weights.as<int8_t>();
    return e;
}

void run_entry_conv(const EntryConv& e, const void* in, const hipie_tensor& mid, const hipie_tensor* out, void* planes, hipStream_t s) {
    Args a = e.a;
    if (out) {
        a.tensor = static_cast<float*>(out->data);
        a.t_sn = out->stride_n;
        a.t_sh = out->stride_h;
        a.t_sw = static_cast<int32_t>(out->stride_w);
    }
    a.x = in;
    a.levels = static_cast<uint8_t*>(mid.data);
    a.out = static_cast<float*>(planes);
    void* args[] = {&a};
    HIPIE_CHECK_HIP(hipLaunchKernel(kernel_of(e, out != nullptr), dim3(8u * static_cast<uint32_t>(a.per_xcd), static_cast<uint32_t>(e.groups_y)), dim3(kThreads), args, e.lds, s));
}

}  // namespace hipie
