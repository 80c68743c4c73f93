// bh_tile_walk.h — wave-cooperative walk over the tile bounding boxes of 64 splats.
//
// The reference tests a splat's bounding-box tiles in a loop run by the
// splat's own thread (project_forward.rs:105-118, map_gaussians.rs:56-79), so
// a wave waits for its largest splat while most lanes idle.  Here a wave
// flattens the (splat, bbox tile) items of its 64 splats into one list, in
// splat order and, within a splat, in the reference's row-major tile order,
// and tests 64 items per step.  Per step, every lane finds the splat that owns
// its item (the splats that start within the step as bits of one LDS word, of
// which a lane counts those below it), fetches that splat's record from LDS and
// evaluates the same tile predicate.  The lane holding a splat's last item
// records the wave's running count of passing items through it, and a splat's
// hits are the difference of two such prefixes.  Passing items come out in
// exactly the order the per-splat loops would emit them, so the map kernel
// writes them contiguously.
//
// What bounds it: VALU issue, 93 instructions a step of the runs' walk.  The
// owner by a max-scan over 64 words of LDS, and the predicate's divisors and
// numerators scaled by the tile's width in every lane, made it 110 and eleven
// waits: 6M splats at 3840x2160, project_forward 526 -> 481 us and map_runs 504
// -> 451 us; 1M at 1920x1080, 73 -> 71 and 53 -> 50 us.
#pragma once

#include "bh_splat_math.h"
#include "bh_wave.h"

namespace bh {

// The walk record in LDS (64 bytes, four reads) of a splat that has items; the
// wave's records lie next to each other in lane order.
struct WalkRec {
    float4 a;  // mean x, mean y, conic c00, conic c01
    float4 b;  // conic c11, power threshold, 1 / bbox width, end item index (kWalkRuns: lane; bits)
    uint4 c;   // bbox min_x, bbox min_y, bbox width, first item index
    float4 d;  // the predicate's divisors' reciprocals 1 / (16 c00), 1 / (TH c11), then
               // the divisors (kWalkPairs: lane, bits)
};

// RN(num / den) from y = RN(1 / den) for den > 0 and num < den (quotient
// below 1, so nothing overflows): q0 = RN(num y) is within an ulp of the
// quotient, the residual num - den q0 is exact in one fma, and RN(q0 + r y)
// is the correctly rounded quotient (Markstein's theorem for a correctly
// rounded reciprocal and a faithful first quotient; the quotient's
// correctly rounded value is what the reference's division gives).  Below the
// normal range the result can differ from the division in the last place of
// a subnormal, which the predicate then adds to a tile edge that absorbs it.
__device__ __forceinline__ float div_by_recip(float num, float den, float y) {
    const float q0 = num * y;
    const float r = __builtin_fmaf(-den, q0, num);
    return __builtin_fmaf(r, y, q0);
}

// Orders this wave's LDS writes before its later LDS reads as seen by the
// compiler: without it, a lane's read of a slot it wrote itself may be
// forwarded from its own store even when another lane of the wave overwrote
// the slot in between.  Wavefront scope: no instruction is emitted.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// The power will_contribute (bh_splat_math.h) compares with the threshold,
// evaluated without branches: both edge quotients and the power at the
// clamped edge point are computed for every lane and the predicate's selects
// pick them, so `power <= pt` is the predicate's decision bit for bit (a splat
// whose mean lies in the tile gets -1, which passes).  Tile widths 16 and TH
// are exact differences of the tile's float edges for tile columns < 2^20.
//
// The reference's quotients are (dxf c00 dx + dxf c01 dy) / (dxf c00 dxf) with
// dxf = +-16 (and +-TH in y).  A product by a power of two is exact (short of
// over- and underflow, which a conic of pixels^-2 that contributes does not
// come near), so each is +-(c00 dx + c01 dy) / (16 c00), rounded the same, and
// den_x = 16 c00, den_y = TH c11 and their reciprocals rx, ry are the splat's.
template <int TH>
__device__ __forceinline__ float tile_power(uint32_t tx, uint32_t ty, V2 m, const S2& c, float den_x, float den_y,
                                            float rx, float ry) {
    const float min_x = (float)(tx * 16u), min_y = (float)(ty * (uint32_t)TH);
    const float max_x = min_x + 16.0f, max_y = min_y + (float)TH;
    const bool x_left = m.x < min_x, x_right = m.x > max_x;
    const bool in_x = !(x_left || x_right);
    const bool y_above = m.y < min_y, y_below = m.y > max_y;
    const bool in_y = !(y_above || y_below);
    const float corner_x = x_left ? min_x : max_x;
    const float corner_y = y_above ? min_y : max_y;
    const float dxf = x_left ? 16.0f : -16.0f;
    const float dyf = y_above ? (float)TH : -(float)TH;
    const float diff_x = m.x - corner_x;
    const float diff_y = m.y - corner_y;
    // a quotient at or above 1 clamps to 1
    const float gx = c.c00 * diff_x + c.c01 * diff_y, gy = c.c01 * diff_x + c.c11 * diff_y;
    const float nx = x_left ? gx : -gx, ny = y_above ? gy : -gy;
    const float qx = nx >= den_x ? 1.0f : bh_maxf(div_by_recip(nx, den_x, rx), 0.0f);
    const float qy = ny >= den_y ? 1.0f : bh_maxf(div_by_recip(ny, den_y, ry), 0.0f);
    const float tt_x = in_y ? 0.0f : qx;
    const float tt_y = in_x ? 0.0f : qy;
    const float px = corner_x + tt_x * dxf;
    const float py = corner_y + tt_y * dyf;
    const float power = calc_sigma(px, py, c, m.x, m.y);
    return (in_x && in_y) ? -1.0f : power;
}

// Items (bbox tiles) of a splat whose box is bb; zero for an empty box.
__device__ __forceinline__ uint32_t bbox_items(const TileBox& bb) {
    return (bb.max_x > bb.min_x && bb.max_y > bb.min_y) ? (bb.max_x - bb.min_x) * (bb.max_y - bb.min_y) : 0u;
}

// Cooperative walk of one wave over 16 x TH tiles.  Every lane of the wave must call it (it uses
// wave-wide DPP and ballots).  `items` is this lane's bbox tile count (0 for a
// culled or absent splat); m, conic, pt, bb describe its splat.  `rec`
// and `ends` are this wave's 64-entry LDS arrays (kWalkRuns: no `ends`),
// `starts_word` its word of LDS.
//
// Returns the number of passing tiles of this lane's splat (with kWalkRuns 0).
//
// With OUT == kWalkPairs, the passing items are stored at out_base + (passing
// items before it in walk order): tile id tx + ty * tile_bw into tile_ids (as
// TileT) and id_base + owner lane into ids, skipping positions >= out_end.
//
// With OUT == kWalkRuns, runs of passing items next to each other in a row are
// stored instead, in walk order from out_base: ty << 16 | tx << 8 | length - 1
// into tile_ids (as uint32_t; tile coordinates below 256) and the id into ids;
// a run ends with its step of 64 items at the latest.  Each adds one to
// row_hist[ty] (LDS), and *runs receives their number (the same in every lane).
constexpr int kWalkCount = 0, kWalkPairs = 1, kWalkRuns = 2;
template <int OUT, int TH, typename TileT>
__device__ uint32_t wave_tile_walk(uint32_t lane, uint32_t items, V2 m, const S2& conic, float pt,
                                   const TileBox& bb, WalkRec* rec, unsigned long long* starts_word, uint32_t* ends,
                                   uint32_t tile_bw, uint32_t out_base, uint32_t out_end, uint32_t id_base,
                                   TileT* __restrict__ tile_ids, uint32_t* __restrict__ ids,
                                   uint32_t* row_hist = nullptr, uint32_t* runs = nullptr) {
    const uint32_t incl = wave_incl_add_u32(items);
    const uint32_t start = incl - items;
    const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
    const uint32_t bw = bb.max_x - bb.min_x;
    const uint32_t rank = lanes_below(__builtin_amdgcn_ballot_w64(items != 0u));
    if (items != 0u) {
        const float den_x = 16.0f * conic.c00, den_y = (float)TH * conic.c11;
        rec[rank].a = make_float4(m.x, m.y, conic.c00, conic.c01);
        rec[rank].b = make_float4(conic.c11, pt, 1.0f / (float)bw, __uint_as_float(OUT == kWalkRuns ? lane : incl));
        rec[rank].c = make_uint4(bb.min_x, bb.min_y, bw, start);
        rec[rank].d = make_float4(1.0f / den_x, 1.0f / den_y, OUT == kWalkPairs ? __uint_as_float(lane) : den_x, den_y);
    }
    // the first item of a splat that has any
    const uint32_t key = items != 0u ? start : 0xFFFFFFFFu;
    uint32_t written = 0;  // passing items of earlier steps (wave uniform)
    uint32_t run_count = 0;
    for (uint32_t base = 0; base < total; base += 64u) {
        // the owner of item base + lane: the last splat that starts at or
        // before it.  Bit k of the word: one starts at item base + 1 + k.
        *starts_word = 0ull;
        wave_lds_fence();
        const uint32_t ahead = key - base - 1u;
        if (ahead < 63u)
            __hip_atomic_fetch_or(starts_word, 1ull << ahead, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        wave_lds_fence();
        const uint32_t first = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(key <= base)) - 1u;
        const uint32_t owner = first + lanes_below(*starts_word);
        const uint32_t item = base + lane;
        const bool valid = item < total;
        const WalkRec r = rec[owner];
        // the owner's item prefix, read with the rest of its record (left to
        // itself the compiler reads it again inside the branch below: one
        // more LDS round trip per step)
        uint32_t r_incl = __float_as_uint(r.b.w);  // kWalkRuns: the lane
        __asm__ volatile("" : "+v"(r_incl));
        const uint32_t local = item - r.c.w;
        // row = local / width, exactly, through the float reciprocal: with
        // w = width and 1/w rounded, (local + 0.5) / w lies at least 0.5 / w
        // from an integer and the two roundings move it by less than
        // (row + 1) 2^-23, below 0.5 / w while (row + 1) w < 2^22 (a box
        // holds at most tile_bw * tile_bh < 2^21 tiles: bh_render_forward
        // rejects larger images)
        const uint32_t row = (uint32_t)(((float)local + 0.5f) * r.b.z);
        const uint32_t col = local - __umul24(row, r.c.z);  // both factors and the product < 2^21
        const uint32_t tx = r.c.x + col, ty = r.c.y + row;
        // will_contribute as one comparison; the lane conditions stay wave masks
        const float den_x = OUT == kWalkPairs ? 16.0f * r.a.z : r.d.z;
        const float power =
            tile_power<TH>(tx, ty, v2(r.a.x, r.a.y), S2{r.a.z, r.a.w, r.b.x}, den_x, r.d.w, r.d.x, r.d.y);
        const uint64_t pmask = __builtin_amdgcn_ballot_w64(power <= r.b.y) & __builtin_amdgcn_ballot_w64(valid);
        const bool pass = __builtin_amdgcn_inverse_ballot_w64(pmask);
        // the wave's passing items up to and including this one, kept at a
        // splat's last item
        const uint32_t below = lanes_below(pmask);
        if (OUT != kWalkRuns && valid && item + 1u == r_incl) ends[owner] = written + below + (pass ? 1u : 0u);
        if (OUT == kWalkRuns) {
            // a run starts at a passing item that opens a row of its box or
            // follows one that fails, and ends likewise
            const uint64_t opens = __builtin_amdgcn_ballot_w64(col == 0u);
            const uint64_t starts = pmask & (~(pmask << 1) | opens);
            const uint64_t stops = pmask & (~(pmask >> 1) | (opens >> 1));
            if (__builtin_amdgcn_inverse_ballot_w64(starts)) {
                const uint32_t more = (uint32_t)__builtin_ctzll(stops >> lane);
                const uint32_t pos = out_base + run_count + lanes_below(starts);
                if (pos < out_end) {
                    tile_ids[pos] = (TileT)(ty << 16 | tx << 8 | more);
                    ids[pos] = id_base + r_incl;
                }
                atomicAdd(&row_hist[ty], 1u);
            }
            run_count += (uint32_t)__popcll(starts);
        }
        if (OUT == kWalkPairs && pass) {
            const uint32_t pos = out_base + written + below;
            if (pos < out_end) {
                tile_ids[pos] = (TileT)(tx + __umul24(ty, tile_bw));  // a tile id < 2^21
                ids[pos] = id_base + __float_as_uint(r.d.z);
            }
        }
        written += (uint32_t)__popcll(pmask);
        wave_lds_fence();
    }
    if (OUT == kWalkRuns) {
        *runs = run_count;
        return 0u;
    }
    if (items == 0u) return 0u;
    return ends[rank] - (rank ? ends[rank - 1u] : 0u);
}

}  // namespace bh
