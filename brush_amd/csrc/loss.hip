// loss.hip — fused L1 + SSIM image loss and its VJP for gfx950.
//
// Restates the image-loss kernels of crates/brush-loss/src/lib.rs:
//   image_l1_forward_kernel / image_loss_forward_kernel   (lib.rs:228-555)
//   image_l1_backward_kernel / image_loss_backward_kernel  (lib.rs:280-893)
// The loss map is l1_w * |pred - gt_eff| + ssim_w * SSIM(pred, gt_eff) per
// colour channel, with SSIM over an 11x11 Gaussian window (sigma 1.5) and
// zero padding outside the image; a 4th (alpha) channel gets |pred.a - gt.a|.
// GT stays packed RGBA8 ([H, W] u32, r in the low byte).  Optional compositing
// gt_eff = gt + (1 - gt.a) * bg and masking by gt.a as in the reference.
//
// Layout differs from the reference on purpose: the reference permutes the
// render to [C, H, W] before its kernels; here `pred` is read in the render's
// own [H, W, stride] layout (stride 4 reads RGB out of an RGBA image) and the
// gradient is written in that layout, zeros in the channels the loss does
// not see, so a training step hands the render's gradient straight to the
// rasterizer's backward.
//
// SSIM: a wave owns one colour channel of a strip of 64 columns and marches
// down its rows; a workgroup holds a wave per channel.  Per row, the wave
// stages 74 pixels in LDS (its own, no barrier), each lane forms the
// horizontal sums of its column, and a ring of the last eleven rows' sums, in
// registers, gives the vertical ones: no vertical halo but the ten rows a
// strip starts with, and no LDS traffic for the second direction.  The VJP is
// two such kernels: the first writes each pixel's three partials times the
// chain to a workspace (36 bytes a pixel), the second blurs those.
//
// What bounds them: VALU issue (the two blurs of five moments are 170
// operations a pixel and channel without contraction, which the bits of the
// map depend on; 26M, 31M and 17M wave instructions at 1919x1081, 43, 51 and
// 27 us), with the memory latency of the rows read ahead on top in the last.
// Tiles of 16x16 with a 10-pixel halo recomputed the first blur 3.7 times and
// read each tap from LDS.  At 1919x1081, three channels: forward 74 -> 57 us,
// VJP 275 (with a fill) -> 112 us.
//
// A forward whose VJP follows (autograd, the training step) leaves the partials
// that it has at hand anyway (36 bytes a pixel), and the VJP is the second kernel
// alone, which takes the chain in as it reads them.  image_loss_partials_kernel
// repeats the forward's two blurs, for a VJP called by itself.  At 1919x1081
// forward and VJP 205 -> 156 us with the autograd node's copies, a training step
// at 1600x1064 951 -> 915 us.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bh_internal.h"
#include "bh_tile_walk.h"

namespace bh {

constexpr int kHalo = 5;
constexpr int kTaps = 2 * kHalo + 1;
// the tiles of the VJP without a workspace
constexpr int kLTile = 16;
constexpr int kShared = kLTile + 2 * kHalo;    // 26
constexpr int kExtended = kLTile + 4 * kHalo;  // 36

constexpr uint32_t kStrip = 64;                   // output columns of a wave
constexpr uint32_t kStripIn = kStrip + 2 * kHalo;  // 74

struct LossParams {
    uint32_t w, h, stride, channels;
    float l1_w, ssim_w, bg[3];
    uint32_t composite, mask;
    uint32_t rows;  // output rows of a strip
    float taps[6];  // taps[5 - d] is the weight at distance d (taps[5] the centre)
};

constexpr float kC1 = 0.01f * 0.01f;
constexpr float kC2 = 0.03f * 0.03f;
constexpr float kInv255 = 1.0f / 255.0f;

// One packed GT byte as the reference's read_gt (lib.rs:140-159): colour byte c
// and alpha, both * 1/255.
__device__ __forceinline__ void gt_bytes(uint32_t v, uint32_t c, float& gc, float& ga) {
    gc = (float)((v >> (c * 8u)) & 0xFFu) * kInv255;
    ga = (float)((v >> 24u) & 0xFFu) * kInv255;
}

__device__ __forceinline__ float gt_effective(const LossParams& p, uint32_t v, uint32_t c, float& ga) {
    float gc;
    gt_bytes(v, c, gc, ga);
    return p.composite ? gc + (1.0f - ga) * p.bg[c] : gc;
}

// SSIM value and its partials from the five blurred moments (lib.rs:192-209,
// 502-520): returns the clamped SSIM; dmu1, dsigma1, dsigma12 zero when the
// raw value was clamped.
__device__ __forceinline__ float ssim_from_moments(float o0, float o1, float o2, float o3, float o4, float& dmu1,
                                                   float& dsigma1, float& dsigma12) {
    const float mu1 = o0, mu2 = o2;
    const float mu1_sq = mu1 * mu1, mu2_sq = mu2 * mu2;
    const float sigma1_sq = fmaxf(0.0f, o1 - mu1_sq);
    const float sigma2_sq = fmaxf(0.0f, o3 - mu2_sq);
    const float sigma12 = o4 - mu1 * mu2;
    const float a = mu1_sq + mu2_sq + kC1;
    const float b = sigma1_sq + sigma2_sq + kC2;
    const float c_top = 2.0f * mu1 * mu2 + kC1;
    const float d_top = 2.0f * sigma12 + kC2;
    const float inv_ab = 1.0f / (a * b);
    const float cd = c_top * d_top * inv_ab;
    const bool clamped = cd < -1.0f || cd > 1.0f;
    dmu1 = clamped ? 0.0f : 2.0f * mu2 * inv_ab * (d_top - c_top) - 2.0f * mu1 * cd * (1.0f / a - 1.0f / b);
    dsigma1 = clamped ? 0.0f : -cd / b;
    dsigma12 = clamped ? 0.0f : 2.0f * c_top * inv_ab;
    const float raw = (c_top * d_top) / (a * b);
    return fminf(fmaxf(raw, -1.0f), 1.0f);
}

__device__ __forceinline__ float l1_sign(float diff) { return diff > 0.0f ? 1.0f : (diff < 0.0f ? -1.0f : 0.0f); }

// ---- strips ---------------------------------------------------------------------------

// The five moments (x, x^2, y, y^2, x y) of the pixels of one input row, in a
// wave's LDS, and their horizontal sums at column col + 5, in the reference's
// order: the taps from the nearest pair outwards, then the centre.  The
// products are formed once a pixel instead of once a tap.
struct MomentRow {
    float2 xy[kStripIn];
    float3 q[kStripIn];  // x^2, y^2, x y
};
struct Moments {
    float v[5];
};
__device__ __forceinline__ void put_moments(MomentRow& row, uint32_t col, float2 xy) {
    row.xy[col] = xy;
    row.q[col] = make_float3(xy.x * xy.x, xy.y * xy.y, xy.x * xy.y);
}
__device__ __forceinline__ Moments blur_row(const MomentRow& row, uint32_t col, const float* taps) {
    Moments m = {{0.0f, 0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int d = 1; d <= kHalo; d++) {
        const float wd = taps[kHalo - d];
        const float2 l = row.xy[col + kHalo - d], r = row.xy[col + kHalo + d];
        const float3 lq = row.q[col + kHalo - d], rq = row.q[col + kHalo + d];
        m.v[0] += (l.x + r.x) * wd;
        m.v[1] += (lq.x + rq.x) * wd;
        m.v[2] += (l.y + r.y) * wd;
        m.v[3] += (lq.y + rq.y) * wd;
        m.v[4] += (lq.z + rq.z) * wd;
    }
    const float2 c = row.xy[col + kHalo];
    const float3 cq = row.q[col + kHalo];
    const float wc = taps[kHalo];
    m.v[0] += c.x * wc;
    m.v[1] += cq.x * wc;
    m.v[2] += c.y * wc;
    m.v[3] += cq.y * wc;
    m.v[4] += cq.z * wc;
    return m;
}

// This workgroup's strip: its first output column and row, and the end of its
// output rows.
struct Strip {
    uint32_t x0, y0, y1;
};
__device__ __forceinline__ Strip strip_of(const LossParams& p) {
    const uint32_t y0 = blockIdx.y * p.rows;
    return Strip{blockIdx.x * kStrip, y0, min(p.h, y0 + p.rows)};
}

// The channel that a wave of the workgroup owns.
__device__ __forceinline__ uint32_t wave_channel() {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

// The SSIM moments of every output pixel of channel c of the strip, in row
// order: use(column, row, x, y, five moments), called by the whole wave (the
// column may lie past the image).  ahead(row) is called one output row before
// use, to start the loads that it needs (rows past the strip's end are its
// last).  `rows` is the wave's two rows of LDS.
template <typename A, typename F>
__device__ __forceinline__ void march_moments(const LossParams& p, const Strip& st, uint32_t c,
                                              const float* __restrict__ pred, const uint32_t* __restrict__ gt,
                                              MomentRow* rows, A ahead, F use) {
    const uint32_t lane = threadIdx.x & 63u;
    // this lane's input columns: x0 - 5 + lane, and for the first ten lanes
    // x0 + 59 + lane (clamped addresses; what lies outside reads as zero)
    const int ca = (int)(st.x0 + lane) - kHalo, cb = ca + (int)kStrip;
    const bool in_a = ca >= 0 && ca < (int)p.w, in_b = lane < 2u * kHalo && cb < (int)p.w;
    const uint32_t xa = in_a ? (uint32_t)ca : 0u, xb = in_b ? (uint32_t)cb : 0u;
    // the next row's pixels, unconverted until they are staged
    float va = 0.0f, vb = 0.0f;
    uint32_t ga = 0u, gb = 0u;
    bool in_next = false;
    auto load = [&](uint32_t r) {
        const int y = (int)(st.y0 + r) - kHalo;
        in_next = y >= 0 && y < (int)p.h;  // uniform
        const size_t at = (size_t)(in_next ? y : 0) * p.w;
        const float* pr = pred + at * p.stride + c;
        const uint32_t* gr = gt + at;
        va = pr[(size_t)xa * p.stride], vb = pr[(size_t)xb * p.stride];
        ga = gr[xa], gb = gr[xb];
    };
    load(0u);
    Moments ring[kTaps];
    float2 centre[kTaps];
    for (uint32_t r0 = 0;; r0 += kTaps) {
#pragma unroll
        for (int k = 0; k < kTaps; k++) {
            const uint32_t r = r0 + (uint32_t)k;
            MomentRow& row = rows[k & 1];
            // (a row is written again two rows later: the reads of the one
            // between come before it in the wave's order)
            if (k == 0) wave_lds_fence();
            float alpha;
            const float wa = gt_effective(p, ga, c, alpha), wb = gt_effective(p, gb, c, alpha);
            put_moments(row, lane, in_next && in_a ? make_float2(va, wa) : make_float2(0.0f, 0.0f));
            if (lane < 2u * kHalo)
                put_moments(row, kStrip + lane, in_next && in_b ? make_float2(vb, wb) : make_float2(0.0f, 0.0f));
            load(r + 1u);
            if (k >= kTaps - 2 || r0 > 0u) ahead(min(st.y0 + r + 1u - 2u * kHalo, st.y1 - 1u));
            wave_lds_fence();
            ring[k] = blur_row(row, lane, p.taps);
            centre[k] = row.xy[lane + kHalo];
            if (k == kTaps - 1 || r0 > 0u) {  // row r - 10 of the strip is complete
                const uint32_t y = st.y0 + r - 2u * kHalo;
                if (y >= st.y1) return;
                constexpr int C = kHalo + 1;  // ring slot of input row r - 5: (k + 6) mod 11
                Moments o = {{0.0f, 0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
                for (int d = 1; d <= kHalo; d++) {
                    const float wd = p.taps[kHalo - d];
                    const Moments &t = ring[(k + C - d + kTaps) % kTaps], &b = ring[(k + C + d) % kTaps];
#pragma unroll
                    for (int q = 0; q < 5; q++) o.v[q] += (t.v[q] + b.v[q]) * wd;
                }
                const Moments& m = ring[(k + C) % kTaps];
#pragma unroll
                for (int q = 0; q < 5; q++) o.v[q] += m.v[q] * p.taps[kHalo];
                const float2 xy = centre[(k + C) % kTaps];
                use(st.x0 + lane, y, xy.x, xy.y, o);
            }
        }
    }
}

// ---- forward ----------------------------------------------------------------------

// The L1 map (ssim_weight 0), one thread per pixel.
__global__ __launch_bounds__(256) void image_l1_forward_kernel(LossParams p, const float* __restrict__ pred,
                                                                const uint32_t* __restrict__ gt,
                                                                float* __restrict__ map) {
    const uint64_t pix = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (pix >= (uint64_t)p.w * p.h) return;
    const uint32_t v = gt[pix];
    const float* x = pred + pix * p.stride;
    float* o = map + pix * p.channels;
    float ga;
#pragma unroll
    for (uint32_t c = 0; c < 3u; c++) {
        float l = p.l1_w * fabsf(x[c] - gt_effective(p, v, c, ga));
        if (p.mask) l = l * ga;
        o[c] = l;
    }
    if (p.channels == 4u) {
        gt_bytes(v, 0u, ga, ga);
        float l = 1.0f * fabsf(x[3] - ga);
        if (p.mask) l = l * ga;
        o[3] = l;
    }
}

// With PARTIALS, the SSIM partials of each pixel go out beside the map, for a
// VJP that follows (partials[(c H + y) W + x]).
template <bool PARTIALS>
__global__ __launch_bounds__(256) void image_loss_forward_kernel(LossParams p, const float* __restrict__ pred,
                                                                  const uint32_t* __restrict__ gt,
                                                                  float* __restrict__ map,
                                                                  float3* __restrict__ partials) {
    __shared__ MomentRow s_rows[3][2];
    const Strip st = strip_of(p);
    const uint32_t c = wave_channel(), lane = threadIdx.x & 63u;
    if (c == 3u) {  // the alpha match, per pixel
        const uint32_t x = st.x0 + lane, y1 = st.y1;
        for (uint32_t y = st.y0; y < y1 && x < p.w; y++) {
            const size_t pix = (size_t)y * p.w + x;
            float gc, ga;
            gt_bytes(gt[pix], 0u, gc, ga);
            float v = 1.0f * fabsf(pred[pix * p.stride + 3u] - ga);
            if (p.mask) v = v * ga;
            map[pix * p.channels + 3u] = v;
        }
        return;
    }
    float3* plane = PARTIALS ? partials + (size_t)c * p.h * p.w : nullptr;
    march_moments(p, st, c, pred, gt, s_rows[c], [](uint32_t) {},
                  [&](uint32_t x, uint32_t y, float pv, float gv, const Moments& o) {
        float dm, ds, dsc;
        const float ssim = ssim_from_moments(o.v[0], o.v[1], o.v[2], o.v[3], o.v[4], dm, ds, dsc);
        float v = p.l1_w * fabsf(pv - gv) + p.ssim_w * ssim;
        if (x < p.w) {
            const size_t pix = (size_t)y * p.w + x;
            if (p.mask) {
                float gc, ga;
                gt_bytes(gt[pix], c, gc, ga);
                v = v * ga;
            }
            map[pix * p.channels + c] = v;
            if (PARTIALS) plane[pix] = make_float3(dm, ds, dsc);
        }
    });
}

// ---- backward ------------------------------------------------------------------------

// dl_dpred has the layout of pred ([H, W, stride]); the channels past the
// loss's are zero.
__global__ __launch_bounds__(256) void image_l1_backward_kernel(LossParams p, const float* __restrict__ pred,
                                                                 const uint32_t* __restrict__ gt,
                                                                 const float* __restrict__ dl_dmap,
                                                                 float* __restrict__ dl_dpred) {
    const uint64_t pix = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (pix >= (uint64_t)p.w * p.h) return;
    const uint32_t v = gt[pix];
    const float* x = pred + pix * p.stride;
    const float* ch = dl_dmap + pix * p.channels;
    float* o = dl_dpred + pix * p.stride;
    float ga;
#pragma unroll
    for (uint32_t c = 0; c < 3u; c++) {
        const float g = gt_effective(p, v, c, ga);
        float chain = ch[c];
        if (p.mask) chain = chain * ga;
        o[c] = p.l1_w * l1_sign(x[c] - g) * chain;
    }
    if (p.channels == 4u) {
        gt_bytes(v, 0u, ga, ga);
        float chain = ch[3];
        if (p.mask) chain = chain * ga;
        o[3] = 1.0f * l1_sign(x[3] - ga) * chain;
    }
    for (uint32_t c = p.channels; c < p.stride; c++) o[c] = 0.0f;
}

// The SSIM partials of channel c times the chain, three floats a pixel:
// partials[(c H + y) W + x].
__global__ __launch_bounds__(192) void image_loss_partials_kernel(LossParams p, const float* __restrict__ pred,
                                                                   const uint32_t* __restrict__ gt,
                                                                   const float* __restrict__ dl_dmap,
                                                                   float3* __restrict__ partials) {
    __shared__ MomentRow s_rows[3][2];
    const Strip st = strip_of(p);
    const uint32_t c = wave_channel();
    float3* plane = partials + (size_t)c * p.h * p.w;
    const uint32_t xc = min(st.x0 + (threadIdx.x & 63u), p.w - 1u);
    float chain = 0.0f, chain_n = 0.0f;
    uint32_t gt_n = 0u, gt_v = 0u;
    march_moments(
        p, st, c, pred, gt, s_rows[c],
        [&](uint32_t y) {
            const size_t pix = (size_t)y * p.w + xc;
            chain = chain_n, gt_v = gt_n;
            chain_n = dl_dmap[pix * p.channels + c];
            if (p.mask) gt_n = gt[pix];
        },
        [&](uint32_t x, uint32_t y, float, float, const Moments& o) {
            float ch = chain;
            if (p.mask) {
                float gc, ga;
                gt_bytes(gt_v, c, gc, ga);
                ch = ch * ga;
            }
            float dm, ds, dsc;
            (void)ssim_from_moments(o.v[0], o.v[1], o.v[2], o.v[3], o.v[4], dm, ds, dsc);
            if (x < p.w) plane[(size_t)y * p.w + x] = make_float3(dm * ch, ds * ch, dsc * ch);
        });
}

// The second blur, of the partials times the chain, and the gradient.  (Outside
// the image the products are zero: the chain is.)  CHAINED partials are the
// products already (image_loss_partials_kernel); the forward's are multiplied
// as they are read, rounded the same.
template <bool CHAINED>
__global__ __launch_bounds__(256) void image_loss_backward_kernel(LossParams p, const float* __restrict__ pred,
                                                                   const uint32_t* __restrict__ gt,
                                                                   const float* __restrict__ dl_dmap,
                                                                   const float3* __restrict__ partials,
                                                                   float* __restrict__ dl_dpred) {
    __shared__ float3 s_rows[3][2][kStripIn];
    const Strip st = strip_of(p);
    const uint32_t c = wave_channel(), lane = threadIdx.x & 63u;
    const uint32_t x = st.x0 + lane;
    const uint32_t xc = min(x, p.w - 1u);
    if (c == 3u) {  // the alpha match, per pixel
        const uint32_t y1 = st.y1;
        for (uint32_t y = st.y0; y < y1 && x < p.w; y++) {
            const size_t pix = (size_t)y * p.w + x;
            float gc, ga;
            gt_bytes(gt[pix], 0u, gc, ga);
            float chain = dl_dmap[pix * p.channels + 3u];
            if (p.mask) chain = chain * ga;
            dl_dpred[pix * p.stride + 3u] = 1.0f * l1_sign(pred[pix * p.stride + 3u] - ga) * chain;
        }
        return;
    }
    const float3* plane = partials + (size_t)c * p.h * p.w;
    float3(*rows)[kStripIn] = s_rows[c];
    const int ca = (int)(st.x0 + lane) - kHalo, cb = ca + (int)kStrip;
    const bool in_a = ca >= 0 && ca < (int)p.w, in_b = lane < 2u * kHalo && cb < (int)p.w;
    const uint32_t xa = in_a ? (uint32_t)ca : 0u, xb = in_b ? (uint32_t)cb : 0u;
    // the next row's partials and chains, untouched until they are staged
    float3 va, vb;
    float cha = 0.0f, chb = 0.0f;
    uint32_t gta = 0u, gtb = 0u;
    bool in_next = false;
    auto load = [&](uint32_t r) {
        const int y = (int)(st.y0 + r) - kHalo;
        in_next = y >= 0 && y < (int)p.h;  // uniform
        const size_t at = (size_t)(in_next ? y : 0) * p.w;
        va = plane[at + xa], vb = plane[at + xb];
        if (!CHAINED) {
            cha = dl_dmap[(at + xa) * p.channels + c], chb = dl_dmap[(at + xb) * p.channels + c];
            if (p.mask) gta = gt[at + xa], gtb = gt[at + xb];
        }
    };
    auto staged = [&](bool in, float3 v, float ch, uint32_t g) {
        if (!CHAINED) {
            if (p.mask) {
                float gc, ga;
                gt_bytes(g, c, gc, ga);
                ch = ch * ga;
            }
            v = make_float3(v.x * ch, v.y * ch, v.z * ch);
        }
        return in_next && in ? v : make_float3(0.0f, 0.0f, 0.0f);
    };
    load(0u);
    float p1_n = 0.0f, chain_n = 0.0f;
    uint32_t gt_n = 0u;
    float3 ring[kTaps];
    for (uint32_t r0 = 0;; r0 += kTaps) {
#pragma unroll
        for (int k = 0; k < kTaps; k++) {
            const uint32_t r = r0 + (uint32_t)k;
            float3* row = rows[k & 1];
            if (k == 0) wave_lds_fence();
            row[lane] = staged(in_a, va, cha, gta);
            if (lane < 2u * kHalo) row[kStrip + lane] = staged(in_b, vb, chb, gtb);
            load(r + 1u);
            // the output row's own inputs, read one row ahead
            const bool out = k == kTaps - 1 || r0 > 0u;
            const uint32_t y = out ? st.y0 + r - 2u * kHalo : st.y0;
            if (y >= st.y1) return;
            const float p1 = p1_n, chain_v = chain_n;
            const uint32_t gt_v = gt_n;
            if (k >= kTaps - 2 || r0 > 0u) {
                const size_t at = (size_t)min(st.y0 + r + 1u - 2u * kHalo, st.y1 - 1u) * p.w + xc;
                p1_n = pred[at * p.stride + c];
                chain_n = dl_dmap[at * p.channels + c];
                gt_n = gt[at];
            }
            wave_lds_fence();
            float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
#pragma unroll
            for (int d = 1; d <= kHalo; d++) {
                const float wd = p.taps[kHalo - d];
                const float3 l = row[lane + kHalo - d], q = row[lane + kHalo + d];
                a0 += (l.x + q.x) * wd;
                a1 += (l.y + q.y) * wd;
                a2 += (l.z + q.z) * wd;
            }
            const float wc = p.taps[kHalo];
            const float3 m = row[lane + kHalo];
            a0 += m.x * wc;
            a1 += m.y * wc;
            a2 += m.z * wc;
            ring[k] = make_float3(a0, a1, a2);
            if (out) {
                constexpr int C = kHalo + 1;
                float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
#pragma unroll
                for (int d = 1; d <= kHalo; d++) {
                    const float wd = p.taps[kHalo - d];
                    const float3 t = ring[(k + C - d + kTaps) % kTaps], b = ring[(k + C + d) % kTaps];
                    s0 += (t.x + b.x) * wd;
                    s1 += (t.y + b.y) * wd;
                    s2 += (t.z + b.z) * wd;
                }
                const float3 v = ring[(k + C) % kTaps];
                s0 += v.x * wc;
                s1 += v.y * wc;
                s2 += v.z * wc;
                float ga;
                const float gv = gt_effective(p, gt_v, c, ga);
                const float chain = p.mask ? chain_v * ga : chain_v;
                const float ssim_grad = s0 + (2.0f * p1) * s1 + gv * s2;
                if (x < p.w) {
                    float* o = dl_dpred + ((size_t)y * p.w + x) * p.stride;
                    o[c] = p.ssim_w * ssim_grad + p.l1_w * l1_sign(p1 - gv) * chain;
                    if (c == 0u)
                        for (uint32_t q = p.channels; q < p.stride; q++) o[q] = 0.0f;
                }
            }
        }
    }
}

// The VJP without a workspace, for calls that cannot have one (a stream under
// capture, no device memory left): one workgroup per 16x16 tile and channel,
// both blurs through LDS with a 10-pixel halo.  The zero channels are written
// by the launcher's fill.
__global__ __launch_bounds__(256) void image_loss_backward_tiled_kernel(LossParams p, const float* __restrict__ pred,
                                                                   const uint32_t* __restrict__ gt,
                                                                   const float* __restrict__ dl_dmap,
                                                                   float* __restrict__ dl_dpred) {
    // buf_a: the (pred, gt_eff) tile with a 10-pixel halo, later the chained
    // partials on the 26x26 ring; buf_b: first-blur sums, later the second
    // horizontal blur (lib.rs:612-626 reuses its scratch the same way)
    __shared__ float buf_a[kExtended * kExtended * 2];
    __shared__ float buf_b[kExtended * kShared * 5];
    const uint32_t c = blockIdx.z;
    const uint32_t tx = threadIdx.x & 15u, ty = threadIdx.x >> 4;
    const uint32_t x0 = blockIdx.x * kLTile, y0 = blockIdx.y * kLTile;
    const uint32_t px = x0 + tx, py = y0 + ty;
    const bool inside = px < p.w && py < p.h;
    if (c == 3u) {
        if (!inside) return;
        const size_t pix = (size_t)py * p.w + px;
        float ga;
        gt_bytes(gt[pix], 0u, ga, ga);
        float chain = dl_dmap[pix * p.channels + c];
        if (p.mask) chain = chain * ga;
        dl_dpred[pix * p.stride + c] = 1.0f * l1_sign(pred[pix * p.stride + c] - ga) * chain;
        return;
    }
    for (uint32_t i = threadIdx.x; i < (uint32_t)(kExtended * kExtended); i += 256u) {
        const uint32_t ly = i / kExtended, lx = i % kExtended;
        const int gy = (int)(y0 + ly) - 2 * kHalo, gx = (int)(x0 + lx) - 2 * kHalo;
        float pv = 0.0f, gv = 0.0f;
        if (gy >= 0 && gx >= 0 && gy < (int)p.h && gx < (int)p.w) {
            const size_t pix = (size_t)gy * p.w + gx;
            float ga;
            pv = pred[pix * p.stride + c];
            gv = gt_effective(p, gt[pix], c, ga);
        }
        buf_a[2 * i] = pv;
        buf_a[2 * i + 1] = gv;
    }
    __syncthreads();
    // first horizontal blur over the 36 rows x 26 columns of the ring
    for (uint32_t i = threadIdx.x; i < (uint32_t)(kExtended * kShared); i += 256u) {
        const uint32_t row = i / kShared, col = i % kShared, centre = col + kHalo;
        float sx = 0.0f, sx2 = 0.0f, sy = 0.0f, sy2 = 0.0f, sxy = 0.0f;
#pragma unroll
        for (int d = 1; d <= kHalo; d++) {
            const float wd = p.taps[kHalo - d];
            const uint32_t il = row * kExtended + centre - d, ir = row * kExtended + centre + d;
            const float xl = buf_a[2 * il], yl = buf_a[2 * il + 1], xr = buf_a[2 * ir], yr = buf_a[2 * ir + 1];
            sx += (xl + xr) * wd;
            sx2 += (xl * xl + xr * xr) * wd;
            sy += (yl + yr) * wd;
            sy2 += (yl * yl + yr * yr) * wd;
            sxy += (xl * yl + xr * yr) * wd;
        }
        const uint32_t ic = row * kExtended + centre;
        const float xc = buf_a[2 * ic], yc = buf_a[2 * ic + 1], wc = p.taps[kHalo];
        sx += xc * wc;
        sx2 += xc * xc * wc;
        sy += yc * wc;
        sy2 += yc * yc * wc;
        sxy += xc * yc * wc;
        float* o = buf_b + (row * kShared + col) * 5;
        o[0] = sx;
        o[1] = sx2;
        o[2] = sy;
        o[3] = sy2;
        o[4] = sxy;
    }
    __syncthreads();
    // vertical blur on the 26x26 ring, SSIM partials times the chain (zero
    // outside the image)
    for (uint32_t i = threadIdx.x; i < (uint32_t)(kShared * kShared); i += 256u) {
        const uint32_t py2 = i / kShared, px2 = i % kShared, centre = py2 + kHalo;
        float out[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int d = 1; d <= kHalo; d++) {
            const float wd = p.taps[kHalo - d];
            const float* t = buf_b + ((centre - d) * kShared + px2) * 5;
            const float* b = buf_b + ((centre + d) * kShared + px2) * 5;
#pragma unroll
            for (int k = 0; k < 5; k++) out[k] += (t[k] + b[k]) * wd;
        }
        {
            const float* m = buf_b + (centre * kShared + px2) * 5;
#pragma unroll
            for (int k = 0; k < 5; k++) out[k] += m[k] * p.taps[kHalo];
        }
        float dm, ds, dsc;
        (void)ssim_from_moments(out[0], out[1], out[2], out[3], out[4], dm, ds, dsc);
        const int gy = (int)(y0 + py2) - kHalo, gx = (int)(x0 + px2) - kHalo;
        float chain = 0.0f;
        if (gy >= 0 && gx >= 0 && gy < (int)p.h && gx < (int)p.w) {
            const size_t pix = (size_t)gy * p.w + gx;
            chain = dl_dmap[pix * p.channels + c];
            if (p.mask) {
                float gc, ga;
                gt_bytes(gt[pix], c, gc, ga);
                chain = chain * ga;
            }
        }
        // buf_a's image tile is dead once buf_b holds the first blur
        float* o = buf_a + i * 3;
        o[0] = dm * chain;
        o[1] = ds * chain;
        o[2] = dsc * chain;
    }
    __syncthreads();
    // second horizontal blur: 26 rows x 16 columns into buf_b
    for (uint32_t i = threadIdx.x; i < (uint32_t)(kShared * kLTile); i += 256u) {
        const uint32_t row = i / kLTile, col = i % kLTile, centre = col + kHalo;
        float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
#pragma unroll
        for (int d = 1; d <= kHalo; d++) {
            const float wd = p.taps[kHalo - d];
            const float* l = buf_a + (row * kShared + centre - d) * 3;
            const float* r = buf_a + (row * kShared + centre + d) * 3;
            a0 += (l[0] + r[0]) * wd;
            a1 += (l[1] + r[1]) * wd;
            a2 += (l[2] + r[2]) * wd;
        }
        const float* m = buf_a + (row * kShared + centre) * 3;
        const float wc = p.taps[kHalo];
        a0 += m[0] * wc;
        a1 += m[1] * wc;
        a2 += m[2] * wc;
        float* o = buf_b + (row * kLTile + col) * 3;
        o[0] = a0;
        o[1] = a1;
        o[2] = a2;
    }
    __syncthreads();
    if (!inside) return;
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
    const uint32_t ly = ty + kHalo;
#pragma unroll
    for (int d = 1; d <= kHalo; d++) {
        const float wd = p.taps[kHalo - d];
        const float* t = buf_b + ((ly - d) * kLTile + tx) * 3;
        const float* b = buf_b + ((ly + d) * kLTile + tx) * 3;
        s0 += (t[0] + b[0]) * wd;
        s1 += (t[1] + b[1]) * wd;
        s2 += (t[2] + b[2]) * wd;
    }
    {
        const float* m = buf_b + (ly * kLTile + tx) * 3;
        const float wc = p.taps[kHalo];
        s0 += m[0] * wc;
        s1 += m[1] * wc;
        s2 += m[2] * wc;
    }
    const size_t pix = (size_t)py * p.w + px;
    const float p1 = pred[pix * p.stride + c];
    float ga;
    const float g = gt_effective(p, gt[pix], c, ga);
    const float ssim_grad = s0 + (2.0f * p1) * s1 + g * s2;
    float chain = dl_dmap[pix * p.channels + c];
    if (p.mask) chain = chain * ga;
    dl_dpred[pix * p.stride + c] = p.ssim_w * ssim_grad + p.l1_w * l1_sign(p1 - g) * chain;
}

// 11-tap Gaussian at sigma 1.5 normalised to sum 1, in f32 with the same
// operations as the reference's gauss_taps (lib.rs:86-100).
static void gauss_taps(float* taps6) {
    const float sigma = 1.5f;
    float w[11];
    float sum = 0.0f;
    for (int i = 0; i < 11; i++) {
        const float x = (float)i - 5.0f;
        w[i] = expf(-x * x / (2.0f * sigma * sigma));
        sum += w[i];
    }
    for (int i = 0; i < 11; i++) w[i] /= sum;
    for (int i = 0; i < 6; i++) taps6[i] = w[i];  // taps[5 - d] = weight at distance d
}

static LossParams loss_params(const bh_image_loss_config& cfg, uint32_t w, uint32_t h, uint32_t stride,
                              uint32_t channels) {
    LossParams p;
    p.w = w;
    p.h = h;
    p.stride = stride;
    p.channels = channels;
    p.l1_w = cfg.l1_weight;
    p.ssim_w = cfg.ssim_weight;
    p.composite = cfg.composite ? 1u : 0u;
    p.mask = cfg.mask ? 1u : 0u;
    for (int i = 0; i < 3; i++) p.bg[i] = cfg.composite ? cfg.background[i] : 0.0f;
    gauss_taps(p.taps);
    return p;
}

// Output rows of a strip: about 1,024 workgroups, four on each of the 256 CUs
// (three waves of up to 134 registers each: what a CU holds at once), of 2 to
// 32 rows.  Fewer rows repeat more of the ten a strip starts with, more leave
// CUs idle or uneven: forward + partials + backward at 1919x1081 take 250 us
// with strips of 6 rows, 191 of 16, 169 of 32 (1,020 workgroups), 182 of 36;
// at 3840x2160 712, 674 (32) and 679 us (44); at 640x360 61 us with 4 rows (900
// workgroups), 64 with 8 and 82 with 16.
static void set_rows(LossParams& p) {
    const uint32_t n = std::max(1u, 1024u / div_up(p.w, kStrip));
    p.rows = std::min(std::max(div_up(p.h, n), 2u), 32u);
}

static dim3 strip_grid(const LossParams& p) { return dim3(div_up(p.w, kStrip), div_up(p.h, p.rows)); }

size_t image_loss_workspace_bytes(uint32_t w, uint32_t h, const bh_image_loss_config& cfg) {
    return cfg.ssim_weight != 0.0f ? (size_t)w * h * 3u * sizeof(float3) : 0u;
}

void launch_image_loss_forward(bh_ctx* ctx, const float* pred, uint32_t stride, uint32_t channels,
                               const uint32_t* gt, uint32_t w, uint32_t h, const bh_image_loss_config& cfg,
                               float* map, float* partials) {
    LossParams p = loss_params(cfg, w, h, stride, channels);
    set_rows(p);
    KernelTimer t(ctx, "image_loss_forward");
    float3* p3 = reinterpret_cast<float3*>(partials);
    if (cfg.ssim_weight == 0.0f)
        launch(ctx, image_l1_forward_kernel, dim3(div_up((uint64_t)w * h, 256)), dim3(256), 0u, p, pred, gt, map);
    else if (p3)
        launch(ctx, image_loss_forward_kernel<true>, strip_grid(p), dim3(64u * channels), 0u, p, pred, gt, map, p3);
    else
        launch(ctx, image_loss_forward_kernel<false>, strip_grid(p), dim3(64u * channels), 0u, p, pred, gt, map, p3);
}

void launch_image_loss_backward(bh_ctx* ctx, const float* pred, uint32_t stride, uint32_t channels,
                                const uint32_t* gt, uint32_t w, uint32_t h, const bh_image_loss_config& cfg,
                                const float* dl_dmap, const float* forward_partials, void* workspace,
                                float* dl_dpred) {
    LossParams p = loss_params(cfg, w, h, stride, channels);
    set_rows(p);
    if (cfg.ssim_weight == 0.0f) {
        KernelTimer t(ctx, "image_loss_backward");
        launch(ctx, image_l1_backward_kernel, dim3(div_up((uint64_t)w * h, 256)), dim3(256), 0u, p, pred, gt, dl_dmap,
               dl_dpred);
        return;
    }
    if (forward_partials) {
        KernelTimer t(ctx, "image_loss_backward");
        launch(ctx, image_loss_backward_kernel<false>, strip_grid(p), dim3(64u * channels), 0u, p, pred, gt, dl_dmap,
               reinterpret_cast<const float3*>(forward_partials), dl_dpred);
        return;
    }
    if (!workspace) {
        if (stride > channels) launch_fill_u32(ctx, (uint32_t*)dl_dpred, 0u, (uint64_t)w * h * stride);
        KernelTimer t(ctx, "image_loss_backward");
        launch(ctx, image_loss_backward_tiled_kernel, dim3(div_up(w, kLTile), div_up(h, kLTile), channels), dim3(256), 0u,
               p, pred, gt, dl_dmap, dl_dpred);
        return;
    }
    float3* partials = static_cast<float3*>(workspace);
    {
        KernelTimer t(ctx, "image_loss_partials");
        launch(ctx, image_loss_partials_kernel, strip_grid(p), dim3(192), 0u, p, pred, gt, dl_dmap, partials);
    }
    KernelTimer t(ctx, "image_loss_backward");
    launch(ctx, image_loss_backward_kernel<true>, strip_grid(p), dim3(64u * channels), 0u, p, pred, gt, dl_dmap,
           (const float3*)partials, dl_dpred);
}

}  // namespace bh
