// A convolution of at most 192 K bytes a pixel (1 x 1, or the few channels of an image) and the depthwise 3 x 3 convolution that
// alone reads it, the first two layers of an inverted residual block, in one launch: the expanded tensor lives in LDS only.
//
// Reference semantics: reference::convolution / group_convolution on widened inputs
// (ngraph/core/reference/.../convolution.hpp:63-146) and the elementwise chain behind each, as the layers' own kernels evaluate
// them: the same integers, the same f32 operations in the same order, the same bytes.
//
// A workgroup of four waves computes 16 T channels of the input rows under a band of R output rows - whole rows, so that the
// only values computed twice are the 3 - S rows between two bands - requantises them into an LDS patch whose border holds the
// level of the padding, and runs the depthwise layer from there, two rows of four pixels x four channels a lane.
//   first half:  v_mfma_i32_16x16x64_i8 with the channels as rows: a lane receives four consecutive channels of one pixel, one
//                LDS dword.  The channel tile's weights and the lane's constants stay in registers, the pixels' 64-byte slices
//                are requested two fragments ahead.  A patch pixel is 16 T + 4 bytes: both halves' dword accesses then meet
//                the minimum of two lanes a bank.
//   second half: the window in registers, v_dot4 on transposed dwords as dwconv3x3_lds_kernel.
// What bounds it: the vector pipe on large maps (the exact chain and a lane's way to its next pixel, 10 + 15 instructions a value:
// 16 -> 96 channels at 112 x 112, stride 2, batch 64 took 42 us alone with 39 of vector issue when the way was two divisions and
// the sums came through accumulation registers, 34.2 -> 30.0 us a launch in flight without), the launch on small ones.
// Small images share a workgroup: a 7 x 7 image alone gives the second half 64 of 256 lanes something to do.
// Measured per launch with three requests in flight, the two layers' own kernels / this one: 16 -> 96 channels at 112 x 112,
// stride 2, batch 64: 55.8 / 30.0 us; 24 -> 144 at 56 x 56 29.1 / 19.5; 64 -> 384 at 14 x 14 7.1 / 6.4; 160 -> 960 at 7 x 7
// 7.2 / 9.7 with one image a workgroup, 4.5 with several.  At batch 8 all of them 5.5 - 8 / 2.7 - 4.7.
#include "conv_dispatch.h"
#include "conv.h"

#include <algorithm>

namespace hipie {

namespace {

typedef int32_t v4i __attribute__((ext_vector_type(4)));
typedef int32_t unaligned_v4i __attribute__((ext_vector_type(4), aligned(4)));      // (an image's pixels are 4 bytes)
typedef __attribute__((address_space(3))) int8_t* lds_bytes;
typedef __attribute__((address_space(3))) uint32_t* lds_dwords;
typedef __attribute__((address_space(3))) v4i* lds_quads;

struct ExpandLayer {
    const int32_t* corr;
    const float *bias, *scale, *ih, *r, *r2;
    float lm1, lo, hi;
    uint32_t xmask;
    int32_t OCp;
};

struct ExpandArgs {
    ExpandLayer l1, l2;
    const int8_t *in, *wgt, *wgt2;
    const int32_t* koff;
    int8_t* out;
    int32_t in_sn, in_sh, in_sw, Kp;
    int32_t out_sn, out_sh, out_sw;
    int32_t W, H, OW, OH, pad_t, pad_l;
    int32_t R, PW, slabs, bands, units, per_xcd;
    int32_t images, N;                     // images a workgroup takes one behind the other (1 where an image has several bands)
    int32_t image_pixels, image_bytes, image_items;   // where it takes several: of one image's patch
    float inv_image_pixels, inv_image_items;
    // 64 pixels on: columns, and what that adds to the offsets in the input and in the patch; into the next row and the next image
    int32_t step_col, step_row, image_rows, nowhere;
    uint32_t step_in, step_lds, row_in, row_lds, image_in, image_lds;
    int32_t quads, channel_groups;         // groups of four output pixels in a row, of four channels that the output holds
    int32_t patch_pieces;                  // 16-byte pieces of the patch
    uint32_t fill;
    float inv_W, inv_quads;
};

template <uint32_t F, int N>
struct ExpandConstants {
    int32_t corr[N];
    float bias[N], scale[N], ih[N], r[N], r2[N];
};

// constants of four consecutive channels into place j of the lane's
template <uint32_t F, int N>
__device__ __forceinline__ void load_constants(const ExpandLayer& l, int oc, int j, ExpandConstants<F, N>& k) {
    const int at = min(oc, l.OCp - 4);     // (channels that do not exist are computed with the last ones' constants and stored nowhere)
    const int4 c = *reinterpret_cast<const int4*>(l.corr + at);
    k.corr[j] = c.x; k.corr[j + 1] = c.y; k.corr[j + 2] = c.z; k.corr[j + 3] = c.w;
    auto four = [&](const float* from, float* to) {
        const float4 v = ld4f(from + at);
        to[0] = v.x; to[1] = v.y; to[2] = v.z; to[3] = v.w;
    };
    four(l.bias, k.bias + j);
    if (F & CF_SCALE) four(l.scale, k.scale + j);
    four(l.ih, k.ih + j);
    four(l.r, k.r + j);
    four(l.r2, k.r2 + j);
}

// the level of one accumulator, in its byte of `packed`
template <uint32_t F, int N>
__device__ __forceinline__ uint32_t level_into(const ExpandLayer& l, const ExpandConstants<F, N>& k, int j, int32_t sum, int byte, uint32_t packed) {
    float x = static_cast<float>(sum);
    x = x + k.bias[j];
    if (F & CF_SCALE) x = x * k.scale[j];
    if (F & CF_CLAMP) x = __builtin_amdgcn_fmed3f(x, l.lo, l.hi);
    return __builtin_amdgcn_cvt_pk_u8_f32(fq_level_fast<2, true, true>(x, 0.f, k.ih[j], k.ih[j], k.r[j], k.r2[j], l.lm1), byte, packed);
}

constexpr int kRows = 2;       // output rows a lane of the depthwise half computes at a time

template <uint32_t F, int S, int NK, int T>
__global__ __launch_bounds__(256, T == 2 ? 4 : 3) void expand_dw_kernel(const ExpandArgs e) {
    extern __shared__ __attribute__((aligned(16))) int8_t patch_memory[];
    const lds_bytes patch = (lds_bytes)patch_memory;
    constexpr int PS = 16 * T + 4, G = 4 * T, SLOTS = 256 / G;
    const int unit = e.per_xcd > 0 ? static_cast<int>(blockIdx.x & 7) * e.per_xcd + static_cast<int>(blockIdx.x >> 3) : static_cast<int>(blockIdx.x);
    if (unit >= e.units) return;                      // whole workgroup, before the barriers
    const int slab = unit % e.slabs, nb = unit / e.slabs, band = nb % e.bands, n = nb / e.bands * e.images, images = min(e.images, e.N - n);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane16 = lane & 15, quad = lane >> 4;
    const int oy0 = band * e.R, rows = min(e.R, e.OH - oy0), iy0 = oy0 * S - e.pad_t;
    const int y0 = max(iy0, 0), y1 = min(iy0 + (rows - 1) * S + 3, e.H), count = (y1 - y0) * e.W * images, frags = (count + 15) >> 4;
    const int c0 = slab * (16 * T);

    // ---- first half: what a lane keeps
    v4i wt[NK][T];
    int32_t ko[NK];
#pragma unroll
    for (int k = 0; k < NK; ++k) ko[k] = e.koff[4 * k + quad];
    const int8_t* const image = e.in + static_cast<int64_t>(n) * e.in_sn + static_cast<int64_t>(y0) * e.in_sh;
    // the lane's pixel of the next fragment to request, 64 pixels behind the one before: in mixed radix (image, row, column), as
    // two divisions and their products a fragment cost as much as half of the chain on its values
    int j = 16 * wave + lane16, col, row = 0, m = 0;
    if (images > 1) {
        fast_divmod(j, e.image_pixels, e.inv_image_pixels, m, row);
        fast_divmod(row, e.W, e.inv_W, row, col);
    } else {
        fast_divmod(j, e.W, e.inv_W, row, col);
    }
    uint32_t from = static_cast<uint32_t>(m * e.in_sn + row * e.in_sh + col * e.in_sw);
    uint32_t to_lds = static_cast<uint32_t>(m * e.image_bytes + ((y0 - iy0 + row) * e.PW + col + e.pad_l) * PS + 4 * quad);
    auto request = [&](v4i (&to)[NK], lds_bytes& at) {       // (pixels behind the last one: the first one's bytes, to where nobody reads)
        const bool on = j < count;
        const uint32_t off = on ? from : 0u;
#pragma unroll
        for (int k = 0; k < NK; ++k) to[k] = *reinterpret_cast<const unaligned_v4i*>(image + (off + static_cast<uint32_t>(ko[k])));
        at = patch + (on ? to_lds : static_cast<uint32_t>(e.nowhere));
        j += 64;
        col += e.step_col;
        from += e.step_in;
        to_lds += e.step_lds;
        const bool next_row = col >= e.W;
        col -= next_row ? e.W : 0;
        from += next_row ? e.row_in : 0u;
        to_lds += next_row ? e.row_lds : 0u;
        if (images > 1) {
            row += e.step_row + (next_row ? 1 : 0);
            const bool next_image = row >= e.image_rows;
            row -= next_image ? e.image_rows : 0;
            from += next_image ? e.image_in : 0u;
            to_lds += next_image ? e.image_lds : 0u;
        }
    };
    v4i p0[NK], p1[NK];
    lds_bytes at0, at1;
    request(p0, at0);
#pragma unroll
    for (int t = 0; t < T; ++t) {
        // row of the packed weights that holds the channel (conv_kernel.h)
        const int ch = min(c0 + 16 * t + lane16, e.l1.OCp - 1), r = ch & 63;
        const int64_t row = (ch & ~63) + 32 * ((r >> 4) & 1) + 8 * ((r >> 2) & 3) + 4 * (r >> 5) + (r & 3);
#pragma unroll
        for (int k = 0; k < NK; ++k) wt[k][t] = *reinterpret_cast<const v4i*>(e.wgt + row * e.Kp + 64 * k + 16 * quad);
    }
    ExpandConstants<F, 4 * T> k1;
#pragma unroll
    for (int t = 0; t < T; ++t) load_constants(e.l1, c0 + 16 * t + 4 * quad, 4 * t, k1);
    request(p1, at1);
    for (int i = tid; i < e.patch_pieces; i += 256) {
        const int b = static_cast<int>(e.fill);
        ((lds_quads)patch)[i] = v4i{b, b, b, b};
    }
    __syncthreads();
    auto fragment = [&](const v4i (&p)[NK], lds_bytes at) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            v4i acc = v4i{k1.corr[4 * t], k1.corr[4 * t + 1], k1.corr[4 * t + 2], k1.corr[4 * t + 3]};
#pragma unroll
            for (int k = 0; k < NK; ++k) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wt[k][t], p[k], acc, 0, 0, 0);
            uint32_t packed = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) packed = level_into(e.l1, k1, 4 * t + j, acc[j], j, packed);
            *(lds_dwords)(at + 16 * t) = packed ^ e.l1.xmask;
        }
    };
    for (int f = wave; f < frags; f += 8) {
        fragment(p0, at0);
        request(p0, at0);
        if (f + 4 < frags) fragment(p1, at1);
        request(p1, at1);
    }

    // ---- second half
    const int cg = tid % G, slot = tid / G, oc = c0 + 4 * cg;
    uint32_t w[3][4], ws[3][4];                       // (w0, w1, w2, 0) of a filter row and the same one byte up
    const int oc_w = min(oc, e.l2.OCp - 4);
#pragma unroll
    for (int kh = 0; kh < 3; ++kh) {
        const uint4 q = *reinterpret_cast<const uint4*>(e.wgt2 + (static_cast<int64_t>(kh) * e.l2.OCp + oc_w) * 4);
        w[kh][0] = q.x; w[kh][1] = q.y; w[kh][2] = q.z; w[kh][3] = q.w;
#pragma unroll
        for (int c = 0; c < 4; ++c) ws[kh][c] = w[kh][c] << 8;
    }
    ExpandConstants<F, 4> k2;
    load_constants(e.l2, oc, 0, k2);
    __syncthreads();
    if (slot >= SLOTS || c0 / 4 + cg >= e.channel_groups) return;
    auto transpose4 = [](uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t (&o)[4]) {
        const uint32_t lo01 = __builtin_amdgcn_perm(b, a, 0x05010400u), hi01 = __builtin_amdgcn_perm(b, a, 0x07030602u);
        const uint32_t lo23 = __builtin_amdgcn_perm(d, c, 0x05010400u), hi23 = __builtin_amdgcn_perm(d, c, 0x07030602u);
        o[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
        o[1] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
        o[2] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
        o[3] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
    };
    constexpr int ROWS_IN = (kRows - 1) * S + 3, NPX = 3 * S + 3;
    const int items = (rows + kRows - 1) / kRows * e.quads * images;
    int8_t* const out = e.out + static_cast<int64_t>(n) * e.out_sn + oc;
    for (int item = slot; item < items; item += SLOTS) {
        int rg, px0, m = 0, j = item;
        if (images > 1) fast_divmod(j, e.image_items, e.inv_image_items, m, j);
        fast_divmod(j, e.quads, e.inv_quads, rg, px0);
        px0 *= 4;
        const lds_bytes from = patch + m * e.image_bytes + (rg * kRows * S * e.PW + px0 * S) * PS + 4 * cg;
        int32_t acc[kRows][4][4];
#pragma unroll
        for (int v = 0; v < kRows; ++v)
#pragma unroll
            for (int px = 0; px < 4; ++px)
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[v][px][c] = k2.corr[c];
#pragma unroll
        for (int i = 0; i < ROWS_IN; ++i) {
            uint32_t p[NPX];
#pragma unroll
            for (int j = 0; j < NPX; ++j) p[j] = *(lds_dwords)(from + (i * e.PW + j) * PS);
            uint32_t x[S == 1 ? 2 : 4][4];            // a channel's four pixels under an output pixel pair / pixel
            transpose4(p[0], p[1], p[2], p[3], x[0]);
            transpose4(p[2], p[3], p[4], p[5], x[1]);
            if constexpr (S == 2) {
                transpose4(p[4], p[5], p[6], p[7], x[2]);
                transpose4(p[6], p[7], p[8], p[8], x[3]);
            }
#pragma unroll
            for (int kh = 0; kh < 3; ++kh) {
                if ((i - kh) % S != 0 || i - kh < 0 || (i - kh) / S >= kRows) continue;
                const int v = (i - kh) / S;
#pragma unroll
                for (int px = 0; px < 4; ++px)
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const uint32_t in4 = S == 1 ? x[px >> 1][c] : x[px][c], w4 = (S == 1 && (px & 1)) ? ws[kh][c] : w[kh][c];
                        acc[v][px][c] = __builtin_amdgcn_sdot4(static_cast<int>(in4), static_cast<int>(w4), acc[v][px][c], false);
                    }
            }
        }
#pragma unroll
        for (int v = 0; v < kRows; ++v) {
            const int row = rg * kRows + v;
            uint32_t packed[4];
#pragma unroll
            for (int px = 0; px < 4; ++px) {
                packed[px] = 0;
#pragma unroll
                for (int c = 0; c < 4; ++c) packed[px] = level_into(e.l2, k2, c, acc[v][px][c], c, packed[px]);
            }
            if (row < rows) {
                int8_t* const o = out + static_cast<int64_t>(m) * e.out_sn + static_cast<int64_t>(oy0 + row) * e.out_sh + static_cast<int64_t>(px0) * e.out_sw;
#pragma unroll
                for (int px = 0; px < 4; ++px)
                    if (px0 + px < e.OW) *reinterpret_cast<uint32_t*>(o + px * e.out_sw) = packed[px] ^ e.l2.xmask;
            }
        }
    }
}

ExpandLayer expand_layer(const ConvArgs& a) {
    return {a.corr, a.bias, a.scale, a.fq_ih, a.fq_r, a.fq_r2, a.lm1, a.clamp_lo, a.clamp_hi, (a.flags & CF_OUT_XOR) ? 0x80808080u : 0u, a.OCp};
}

template <uint32_t F, int S, int NK, int T>
void launch(const ExpandArgs& e, uint32_t blocks, size_t lds, hipStream_t s) {
    hipLaunchKernelGGL((expand_dw_kernel<F, S, NK, T>), dim3(blocks), dim3(256), lds, s, e);
}

template <uint32_t F, int S>
void launch_form(const ExpandArgs& e, int nk, int tiles, uint32_t blocks, size_t lds, hipStream_t s) {
    if (tiles == 2) {
        if (nk == 1) launch<F, S, 1, 2>(e, blocks, lds, s);
        else if (nk == 2) launch<F, S, 2, 2>(e, blocks, lds, s);
        else launch<F, S, 3, 2>(e, blocks, lds, s);
    } else {
        if (nk == 1) launch<F, S, 1, 3>(e, blocks, lds, s);
        else if (nk == 2) launch<F, S, 2, 3>(e, blocks, lds, s);
        else launch<F, S, 3, 3>(e, blocks, lds, s);
    }
}

// LDS of a workgroup at most, so that a compute unit holds three or more
constexpr int64_t kMostLds = 48 * 1024;

}  // namespace

bool expand_dw_epilogues_fit(uint32_t flags1, uint32_t flags2) {
    const uint32_t c1 = flags1 & ~CF_OUT_XOR, c2 = flags2 & ~CF_OUT_XOR;
    return c1 == c2 && (c1 == E_PLAIN0 || c1 == E_CLAMPFQ || c1 == E_SCALEFQ0);
}

ExpandGeometry expand_dw_geometry(int channels, int images, int h, int w, int oh, int ow, int stride, int pad_top, int pad_left, int form) {
    ExpandGeometry g{};
    if (images <= 0 || oh <= 0 || ow <= 0 || pad_top > 2 || (oh - 1) * stride - pad_top >= h) return g;      // (every band has an input row)
    g.tiles = form == 2 ? 3 : 2;
    g.quads = (ow + 3) / 4;
    g.patch_w = std::max((4 * g.quads - 1) * stride + 3, w + pad_left);
    g.slabs = static_cast<int>(ceil_div(channels, 16 * g.tiles));
    const int64_t row_bytes = static_cast<int64_t>(g.patch_w) * (16 * g.tiles + 4), most = form == 1 ? kMostLds / 2 : kMostLds;
    // bands of an even number of rows (a lane computes two), as high as the patch fits and as gives four workgroups to a
    // compute unit, all bands of nearly one height
    const int64_t fit = (most / row_bytes - 3) / stride + 1;
    if (fit < kRows) return g;
    int64_t bands = ceil_div(oh, std::min<int64_t>(fit / kRows * kRows, round_up(oh, kRows)));
    while (form != 3 && bands * images * g.slabs < 1024 && ceil_div(oh, bands) > kRows * 2) ++bands;
    g.rows = static_cast<int>(round_up(ceil_div(oh, bands), kRows));
    g.bands = static_cast<int>(ceil_div(oh, g.rows));
    const int64_t patch = ((g.rows - 1) * stride + 3) * row_bytes;
    g.images = 1;
    if (form == 3) {
        // as many small images as give the depthwise half's lanes an item each (a 7 x 7 image has 8 for the 32 slots)
        const int items = (oh + kRows - 1) / kRows * g.quads, slots = 256 / (4 * g.tiles);
        if (g.bands > 1 || 2 * items > slots) return g;
        g.images = static_cast<int>(std::min<int64_t>({slots / items, images, most / patch}));
        while (g.images > 1 && g.slabs * ceil_div(images, g.images) < 256) --g.images;
        if (g.images < 2) return g;
    }
    g.lds = static_cast<size_t>(round_up(patch * g.images, 16) + round_up(16 * g.tiles + 4, 16));      // (and a pixel nobody reads)
    const int64_t units = static_cast<int64_t>(g.slabs) * g.bands * ceil_div(images, g.images);
    g.ok = units < (1 << 24) && static_cast<int64_t>(h) * w < (1 << 24);
    return g;
}

void launch_expand_dw(const ConvLaunch& first, const ConvLaunch& second, int images, int h, int w, int fill, int form, hipStream_t s) {
    const ConvArgs &a = first.a, &b = second.a;
    const int OH = b.OHOW / b.OW, S = b.conv_sh, channels = std::min(a.out_sw, b.out_sw);
    const ExpandGeometry g = expand_dw_geometry(channels, images, h, w, OH, b.OW, S, second.pad_top, second.pad_left, form);
    HIPIE_REQUIRE(g.ok && a.nk >= 1 && a.nk <= 3 && b.wgt2 && S == b.conv_sw && (S == 1 || S == 2), HIPIE_GENERAL_ERROR,
                  "expansion and depthwise layer in one launch: %d x %d, %d K steps", h, w, a.nk);
    ExpandArgs e{};
    e.l1 = expand_layer(a);
    e.l2 = expand_layer(b);
    e.in = a.in + a.in_origin;
    e.wgt = a.wgt;
    e.wgt2 = b.wgt2;
    e.koff = a.koff;
    e.out = static_cast<int8_t*>(b.out);
    e.in_sn = a.in_sn; e.in_sh = a.in_sh * a.conv_sh; e.in_sw = a.in_sw * a.conv_sw; e.Kp = a.Kp;
    e.out_sn = b.out_sn; e.out_sh = b.out_sh; e.out_sw = b.out_sw;
    e.W = w; e.H = h; e.OW = b.OW; e.OH = OH; e.pad_t = second.pad_top; e.pad_l = second.pad_left;
    e.R = g.rows; e.PW = g.patch_w; e.slabs = g.slabs; e.bands = g.bands; e.units = static_cast<int32_t>(g.slabs * g.bands * ceil_div(images, g.images));
    e.images = g.images; e.N = images;
    // (an image in one band: its patch holds all of the rows that it reads)
    e.image_rows = std::min((OH - 1) * S + 3 - second.pad_top, h);
    e.image_pixels = e.image_rows * w;
    e.image_bytes = ((g.rows - 1) * S + 3) * g.patch_w * (16 * g.tiles + 4);
    e.image_items = (OH + kRows - 1) / kRows * g.quads;
    const int PS = 16 * g.tiles + 4, per_image = g.images > 1 ? e.image_pixels : 1 << 30, step_images = 64 / per_image, rest = 64 % per_image;
    e.step_row = rest / w;
    e.step_col = rest % w;
    e.step_in = static_cast<uint32_t>(step_images * e.in_sn + e.step_row * e.in_sh + e.step_col * e.in_sw);
    e.step_lds = static_cast<uint32_t>(step_images * e.image_bytes + (e.step_row * g.patch_w + e.step_col) * PS);
    e.row_in = static_cast<uint32_t>(e.in_sh - w * e.in_sw);
    e.row_lds = static_cast<uint32_t>((g.patch_w - w) * PS);
    e.image_in = static_cast<uint32_t>(e.in_sn - e.image_rows * e.in_sh);
    e.image_lds = static_cast<uint32_t>(e.image_bytes - e.image_rows * g.patch_w * PS);
    e.nowhere = static_cast<int32_t>(g.lds - round_up(PS, 16));
    e.inv_image_pixels = 1.0f / static_cast<float>(e.image_pixels);
    e.inv_image_items = 1.0f / static_cast<float>(e.image_items);
    e.quads = g.quads;
    e.channel_groups = channels / 4;
    e.patch_pieces = static_cast<int32_t>(g.lds / 16);
    e.fill = (static_cast<uint32_t>(fill) & 0xffu) * 0x01010101u;
    e.inv_W = 1.0f / static_cast<float>(w);
    e.inv_quads = 1.0f / static_cast<float>(g.quads);
    // the slabs of a band read the same pixels and write parts of the same cache lines: on one XCD
    e.per_xcd = e.units >= 64 ? static_cast<int32_t>(ceil_div(e.units, 8)) : 0;
    const uint32_t blocks = static_cast<uint32_t>(e.per_xcd > 0 ? 8 * e.per_xcd : e.units);
    const uint32_t core = a.flags & ~CF_OUT_XOR;
    if (core == E_PLAIN0) {
        if (S == 1) launch_form<E_PLAIN0, 1>(e, a.nk, g.tiles, blocks, g.lds, s); else launch_form<E_PLAIN0, 2>(e, a.nk, g.tiles, blocks, g.lds, s);
    } else if (core == E_SCALEFQ0) {
        if (S == 1) launch_form<E_SCALEFQ0, 1>(e, a.nk, g.tiles, blocks, g.lds, s); else launch_form<E_SCALEFQ0, 2>(e, a.nk, g.tiles, blocks, g.lds, s);
    } else {
        if (S == 1) launch_form<E_CLAMPFQ, 1>(e, a.nk, g.tiles, blocks, g.lds, s); else launch_form<E_CLAMPFQ, 2>(e, a.nk, g.tiles, blocks, g.lds, s);
    }
}

}  // namespace hipie
