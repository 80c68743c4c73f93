// tile_runs.hip — the tile sort by runs of tiles, for gfx950.
//
// The tiles a splat touches in one tile row are next to each other (its ellipse
// is convex; a row with a gap gives two runs), so the pairs that the reference
// sorts one by one (render.rs:373-400) come in runs: about five pairs each where
// splats cover thirty tiles.  The sort moves runs and forms the pairs once, in
// their final order:
//
//   map_runs     (project.hip) a splat's runs in depth order, and the number of
//                runs per tile row of every 256 splats
//   radix_scan   (sort.hip) those counts into offsets
//   scatter_runs the runs by tile row, stably
//   count_runs   how many pairs each chunk of 1024 runs of a row has in each
//                column (one LDS add where a run starts, one where it ends)
//   scan_tiles   the first pair of every tile: the tile offsets
//   expand_runs  a chunk's pairs, tile by tile and in depth order inside a tile,
//                written with the sorted tile ids
//
// The result is the stable sort of the depth-ordered pairs by tile id, bit for
// bit what a radix sort of the pairs gives.  Per pair the radix sort moved 36
// bytes (the map's pairs, two digit passes with their upsweeps over 16-bit ids)
// and tile_offsets read 4; here a pair is written once (8 bytes), and a run
// moves 8 + 8 + 6 + 8 bytes.  3M splats at 3840x2160 (one rocprofv3 trace, us):
// the radix passes, scans, upsweeps and tile_offsets took about 1770, radix_scan
// and these kernels take 900; 1M splats at 1920x1080: 125 and 102.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bh_block.h"
#include "bh_internal.h"
#include "bh_tile_walk.h"
#include "bh_wave.h"

namespace bh {

constexpr uint32_t kCols = 256;        // columns of the per-row tables
constexpr uint32_t kChunk = 1024;      // runs per chunk (16 groups of 64)
constexpr uint32_t kChunkWords = kChunk / 64;
constexpr uint32_t kExpandThreads = 512;
constexpr uint32_t kExpandPairs = 6912;  // pairs staged in LDS at a time (two workgroups fit a CU)

// ---- by row ---------------------------------------------------------------------------

// One workgroup per partition of the map (256 splats): its runs, in four
// segments (one per wave of the map), to offs[part][row] + their rank among the
// partition's runs of that row.  A wave ranks 64 runs by their row's bits
// (ballots); the runs go through LDS in row order, so that a row's leave
// together.  Bound by those scattered groups (about four runs each at 1080p):
// 25 us there, 151 us at 3840x2160.
__global__ __launch_bounds__(256) void scatter_runs_kernel(TileRuns r, const uint32_t* __restrict__ cum,
                                                            uint32_t num_visible, const uint32_t* __restrict__ dev,
                                                            uint32_t row_bits, uint32_t cap) {
    constexpr int ITEMS = 8;
    constexpr uint32_t PART = 256u * ITEMS;
    __shared__ uint32_t s_hist[4][256];
    __shared__ uint32_t s_start[256], s_off[256], s_tot[4];
    __shared__ uint32_t s_id[PART];
    __shared__ uint32_t s_pk[PART];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t part = xcd_partition(blockIdx.x, gridDim.x);
    if (dev) num_visible = min(num_visible, dev[0]);
    if (part * 256u >= num_visible) return;
    uint32_t seg[4], pre[5];
    pre[0] = 0u;
#pragma unroll
    for (uint32_t w = 0; w < 4u; w++) {
        const uint32_t c0 = part * 256u + w * 64u;
        const uint32_t n = r.wave_runs[part * 4u + w];
        seg[w] = c0 == 0u || c0 >= num_visible ? 0u : cum[c0 - 1u];
        pre[w + 1] = pre[w] + n;
    }
    const uint32_t total = pre[4];
    if (total == 0u) return;
    s_off[t] = t < r.radix ? r.counts[(size_t)part * r.radix + t] : 0u;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (uint32_t e0 = 0; e0 < total; e0 += PART) {
        for (uint32_t i = t; i < 4u * 256u; i += 256u) (&s_hist[0][0])[i] = 0u;
        __syncthreads();
        uint32_t pk[ITEMS], id[ITEMS], pos[ITEMS];
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            // (a clamped element past the end: loaded, never ranked)
            const uint32_t e = min(e0 + wave * (64u * ITEMS) + (uint32_t)j * 64u + lane, total - 1u);
            uint32_t at = seg[0] + e;
#pragma unroll
            for (uint32_t w = 1; w < 4u; w++)
                if (e >= pre[w]) at = seg[w] + (e - pre[w]);
            at = min(at, cap - 1u);
            pk[j] = r.run_pk[at];
            id[j] = r.run_id[at];
        }
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const bool valid = e0 + wave * (64u * ITEMS) + (uint32_t)j * 64u + lane < total;
            const uint32_t d = pk[j] >> 16;
            uint64_t peers = __ballot(valid);
            for (uint32_t b = 0; b < row_bits; b++) {
                const bool bit = (d >> b) & 1u;
                const uint64_t bal = __ballot(bit);
                peers &= bit ? bal : ~bal;
            }
            uint32_t before = 0u;
            if (valid) before = s_hist[wave][d];
            pos[j] = valid ? before + (uint32_t)__popcll(peers & lt_mask) : 0xFFFFFFFFu;
            if (valid && (peers >> lane) == 1ull) s_hist[wave][d] = before + (uint32_t)__popcll(peers);
        }
        __syncthreads();
        uint32_t n = 0u;  // of row t
#pragma unroll
        for (uint32_t w = 0; w < 4u; w++) {
            const uint32_t c = s_hist[w][t];
            s_hist[w][t] = n;
            n += c;
        }
        uint32_t count;
        s_start[t] = block_exclusive_scan<256>(n, s_tot, &count);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            if (pos[j] != 0xFFFFFFFFu) {
                const uint32_t d = pk[j] >> 16;
                const uint32_t at = s_start[d] + s_hist[wave][d] + pos[j];
                s_pk[at] = pk[j];
                s_id[at] = id[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const uint32_t i = (uint32_t)j * 256u + t;
            if (i < count) {
                const uint32_t k = s_pk[i], d = k >> 16;
                const uint32_t at = s_off[d] + (i - s_start[d]);
                if (at < cap) {  // always: the offsets partition the runs
                    r.sorted_pk[at] = (uint16_t)k;
                    r.sorted_id[at] = s_id[i];
                }
            }
        }
        __syncthreads();
        s_off[t] += n;
    }
}

// ---- chunks of a row --------------------------------------------------------------------

// The rows' runs and chunk groups, built by every workgroup that works on
// chunks: row d holds the sorted runs [base[d], base[d + 1]), in chunks of
// kChunk, `group` of which make a group; its groups are [first[d], first[d + 1]).
struct RowTable {
    uint32_t base[257], first[257];
};
template <int THREADS>
__device__ __forceinline__ void build_rows(RowTable& tab, const TileRuns& r, uint32_t tile_bh, uint32_t* s_tot) {
    const uint32_t t = threadIdx.x;
    uint32_t b0 = 0u, b1 = 0u;
    if (t < 256u) {
        // a row's first run is its offset in partition 0; radix > tile_bh, and
        // the column after the last row holds the number of runs
        b0 = r.counts[min(t, tile_bh)];
        b1 = r.counts[min(t + 1u, tile_bh)];
        tab.base[t] = b0;
        if (t == 255u) tab.base[256] = b1;
    }
    const uint32_t groups = ((b1 - b0 + kChunk - 1u) / kChunk + r.chunk_group - 1u) / r.chunk_group;
    uint32_t total;
    const uint32_t first = block_exclusive_scan<THREADS>(t < 256u ? groups : 0u, s_tot, &total);
    if (t < 256u) tab.first[t] = first;
    if (t == 0u) tab.first[256] = total;
    __syncthreads();
}

// One workgroup per group of chunks (a loop over them): chunk_cols of its
// chunks, group_cols of the group, and its pairs added to the row's.  The rows'
// sums lie 256 bytes apart: adds to one line are done one after the other, about
// 10 ns each, and with the sums side by side they took 20 of the kernel's 30 us
// at 1080p (10 us now; 49 us before at 3840x2160).
__global__ __launch_bounds__(256) void count_runs_kernel(TileRuns r, uint32_t tile_bh) {
    __shared__ RowTable s_rows;
    __shared__ uint32_t s_tot[4];
    __shared__ uint32_t s_diff[kCols + 1];
    __shared__ uint32_t s_row;
    const uint32_t t = threadIdx.x;
    build_rows<256>(s_rows, r, tile_bh, s_tot);
    const uint32_t groups = s_rows.first[256];
    for (uint32_t g = blockIdx.x; g < groups; g += gridDim.x) {
        if (s_rows.first[t] <= g && g < s_rows.first[t + 1u]) s_row = t;
        s_diff[t] = 0u;
        if (t == 0u) s_diff[kCols] = 0u;
        __syncthreads();
        const uint32_t row = s_row, end = s_rows.base[row + 1u];
        const uint32_t run0 = s_rows.base[row] + (g - s_rows.first[row]) * r.chunk_group * kChunk;
        uint32_t running = 0u, all = 0u;
        for (uint32_t j = 0; j < r.chunk_group; j++) {
            const uint32_t b = run0 + j * kChunk;
            if (b >= end) break;
            uint32_t pk[kChunk / 256u];
#pragma unroll
            for (uint32_t q = 0; q < kChunk / 256u; q++) pk[q] = r.sorted_pk[min(b + q * 256u + t, end - 1u)];
#pragma unroll
            for (uint32_t q = 0; q < kChunk / 256u; q++) {
                if (b + q * 256u + t < end) {
                    const uint32_t x0 = pk[q] >> 8, x1 = x0 + (pk[q] & 255u) + 1u;
                    atomicAdd(&s_diff[x0], 1u);
                    atomicSub(&s_diff[min(x1, kCols)], 1u);
                }
            }
            __syncthreads();
            // pairs in column t: the runs open there
            const uint32_t d = s_diff[t];
            uint32_t sum;
            const uint32_t open = block_exclusive_scan<256>(d, s_tot, &sum) + d;
            s_diff[t] = 0u;
            if (t == 0u) s_diff[kCols] = 0u;
            r.chunk_cols[((size_t)g * r.chunk_group + j) * kCols + t] = (uint16_t)running;
            running += open;
            __syncthreads();
        }
        r.group_cols[(size_t)g * kCols + t] = running;
        (void)block_exclusive_scan<256>(running, s_tot, &all);
        if (t == 0u) atomicAdd(&r.row_pairs[row * kRowStride], all);
        __syncthreads();
    }
}

// One workgroup per tile row, one thread per column: the groups' counts become
// the pairs before them in the row's column, the row's tiles get their ranges.
__global__ __launch_bounds__(256) void scan_tiles_kernel(TileRuns r, uint32_t tile_bw, uint32_t tile_bh,
                                                          uint32_t* __restrict__ offsets) {
    __shared__ RowTable s_rows;
    __shared__ uint32_t s_tot[4];
    const uint32_t t = threadIdx.x, row = blockIdx.x;
    const uint32_t mine = t < row ? r.row_pairs[t * kRowStride] : 0u;
    build_rows<256>(s_rows, r, tile_bh, s_tot);
    uint32_t before;
    (void)block_exclusive_scan<256>(mine, s_tot, &before);
    uint32_t run = 0u;
    const uint32_t g1 = s_rows.first[row + 1u];
    for (uint32_t g = s_rows.first[row]; g < g1; g += 16u) {
        uint32_t x[16];
#pragma unroll
        for (uint32_t q = 0; q < 16u; q++) x[q] = r.group_cols[(size_t)min(g + q, g1 - 1u) * kCols + t];
#pragma unroll
        for (uint32_t q = 0; q < 16u; q++) {
            if (g + q < g1) {
                r.group_cols[(size_t)(g + q) * kCols + t] = run;
                run += x[q];
            }
        }
    }
    uint32_t total;
    const uint32_t start = before + block_exclusive_scan<256>(run, s_tot, &total);
    r.tile_base[row * kCols + t] = start;
    if (t < tile_bw)
        reinterpret_cast<uint2*>(offsets)[row * tile_bw + t] = run ? make_uint2(start, start + run) : make_uint2(0u, 0u);
}

// ---- pairs ------------------------------------------------------------------------------

__device__ __forceinline__ uint64_t wave_excl_xor_u64(uint64_t x) {
    uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    auto scan = [](uint32_t v) {
        v ^= dpp_u32<0x111, 0xF>(v);
        v ^= dpp_u32<0x112, 0xF>(v);
        v ^= dpp_u32<0x114, 0xF>(v);
        v ^= dpp_u32<0x118, 0xF>(v);
        v ^= dpp_u32<0x142, 0xA>(v);
        v ^= dpp_u32<0x143, 0xC>(v);
        return v;
    };
    lo = scan(lo) ^ lo;
    hi = scan(hi) ^ hi;
    return ((uint64_t)hi << 32) | lo;
}

// One workgroup per chunk (a loop over them).  Bit b of s_open[w][x] says that
// run 64 w + b covers column x: a run flips its bit where it starts and where
// it ends, and an xor scan along the columns turns flips into cover.  A pair's
// rank among its column's pairs of the word is then the set bits below its
// run's.  A wave lays the pairs of a word's 64 runs out one after the other and
// places 64 per step in LDS by column; the sorted pairs go out as one
// contiguous run per column.  Two workgroups fit a CU (79 KB of LDS each): 53 us
// at 1080p, 677 us at 3840x2160 (55 us and 736 us without the loads ahead),
// where the vector instructions alone take about 270 us and the rest is their
// latency over 16 waves a CU.  (A chunk of more pairs than the LDS holds goes by
// groups of columns, each thread walking the bits of one word and column.)
__global__ __launch_bounds__(kExpandThreads) void expand_runs_kernel(TileRuns r, uint32_t tile_bw, uint32_t tile_bh,
                                                                      uint32_t m_cap,
                                                                      uint32_t* __restrict__ tile_ids,
                                                                      uint32_t* __restrict__ cgids) {
    constexpr uint32_t T = kExpandThreads;
    __shared__ RowTable s_rows;
    __shared__ unsigned long long s_open[kChunkWords][kCols];
    // the column's pairs in the words before, plus, where all the chunk's pairs
    // are staged at once, the chunk's in the columns before
    __shared__ uint16_t s_before[kChunkWords][kCols];
    __shared__ uint32_t s_pair[kExpandPairs];  // column << 16 | run, sorted
    __shared__ uint32_t s_id[kChunk];
    __shared__ uint32_t s_shift[T / 64][64];
    __shared__ uint32_t s_start[kCols + 1];  // the chunk's pairs in the columns before
    __shared__ uint32_t s_delta[kCols];      // from there to the pair's place
    __shared__ uint32_t s_tot[T / 64], s_row[2], s_to;
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    build_rows<T>(s_rows, r, tile_bh, s_tot);
    const uint32_t chunks = s_rows.first[256] * r.chunk_group;
    // workgroups of one XCD (consecutive ids are dealt to the eight in turn)
    // take neighbouring chunks, which write neighbouring pairs
    const uint32_t per = (chunks + 7u) / 8u, step = gridDim.x >> 3, ch0 = (blockIdx.x & 7u) * per;
    uint32_t k = blockIdx.x >> 3;
    auto exists = [&](uint32_t i) { return i < per && ch0 + i < chunks; };
    if (!exists(k)) return;
    // the row of chunk i, to s_row[slot]
    auto locate = [&](uint32_t i, uint32_t slot) {
        const uint32_t g = (ch0 + i) / r.chunk_group;
        if (t < 256u && s_rows.first[t] <= g && g < s_rows.first[t + 1u]) s_row[slot] = t;
    };
    // A chunk's runs (a wave holds words wave and wave + T / 64, a run a lane)
    // and its columns' places are read while the chunk before it is taken apart,
    // and have arrived before that chunk's stores: a later wait for a load would
    // cover the stores too.
    struct Chunk {
        uint32_t row, runs, to;  // runs: to the row's end; a chunk takes kChunk of them
        uint32_t pk[kChunk / T], id[kChunk / T];
    };
    auto load = [&](uint32_t i, uint32_t slot) {
        Chunk c = {};
        const uint32_t ch = ch0 + i, g = ch / r.chunk_group;
        c.row = s_row[slot];
        const uint32_t end = s_rows.base[c.row + 1u];
        const uint32_t b = s_rows.base[c.row] + (ch - s_rows.first[c.row] * r.chunk_group) * kChunk;
        if (b >= end) return c;  // (uniform) a row's last group may lack chunks
        c.runs = end - b;
#pragma unroll
        for (uint32_t q = 0; q < kChunk / T; q++) {
            const uint32_t at = min(b + q * T + t, end - 1u);
            c.pk[q] = r.sorted_pk[at];
            c.id[q] = r.sorted_id[at];
        }
        if (t < kCols)
            c.to =
                r.tile_base[c.row * kCols + t] + r.group_cols[(size_t)g * kCols + t] + r.chunk_cols[(size_t)ch * kCols + t];
        return c;
    };
    locate(k, 0u);
    __syncthreads();
    Chunk c = load(k, 0u);
    for (uint32_t slot = 1u;; slot ^= 1u) {
        const uint32_t next = k + step;
        const bool more = exists(next);
        if (more) locate(next, slot);
#pragma unroll
        for (uint32_t i = 0; i < kChunkWords * kCols / 2u / T; i++)
            reinterpret_cast<ulonglong2*>(&s_open[0][0])[i * T + t] = make_ulonglong2(0ull, 0ull);
        __syncthreads();
        Chunk ahead = {};
        if (more) ahead = load(next, slot);
        if (c.runs == 0u) {
            if (!more) break;
            c = ahead;
            k = next;
            continue;
        }
#pragma unroll
        for (uint32_t q = 0; q < kChunk / T; q++) {
            const uint32_t i = q * T + t;
            s_id[i] = c.id[q];
            if (i < c.runs) {
                const uint32_t x0 = c.pk[q] >> 8, x1 = x0 + (c.pk[q] & 255u) + 1u;
                const unsigned long long bit = 1ull << (i & 63u);
                atomicXor(&s_open[i >> 6][x0], bit);
                if (x1 < kCols) atomicXor(&s_open[i >> 6][x1], bit);
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t q = 0; q < kChunkWords / (T / 64u); q++) {
            // a wave per word row, four columns a lane
            ulonglong2* p = reinterpret_cast<ulonglong2*>(&s_open[q * (T / 64u) + wave][4u * lane]);
            ulonglong2 a = p[0], d = p[1];
            a.y ^= a.x;
            d.x ^= a.y;
            d.y ^= d.x;
            const unsigned long long e = wave_excl_xor_u64(d.y);
            a.x ^= e, a.y ^= e, d.x ^= e, d.y ^= e;
            p[0] = a;
            p[1] = d;
        }
        __syncthreads();
        uint32_t n = 0u;
        uint32_t before[kChunkWords];
        if (t < kCols) {
#pragma unroll
            for (uint32_t w = 0; w < kChunkWords; w++) {
                before[w] = n;
                n += (uint32_t)__popcll(s_open[w][t]);
            }
        }
        uint32_t total;
        const uint32_t start = block_exclusive_scan<T>(n, s_tot, &total);
        if (t < kCols) {
            const uint32_t plus = total <= kExpandPairs ? start : 0u;
#pragma unroll
            for (uint32_t w = 0; w < kChunkWords; w++) s_before[w][t] = (uint16_t)(before[w] + plus);
            s_start[t] = start;
            s_delta[t] = c.to - start;
        }
        if (t == 0u) s_start[kCols] = total;
        __syncthreads();
        // as many whole columns as fit the LDS at a time (a column holds at
        // most kChunk pairs); nearly always all of them
        for (uint32_t from = 0; from < kCols;) {
            const uint32_t w0 = s_start[from];
            uint32_t upto = kCols;
            if (total - w0 > kExpandPairs) {  // (uniform)
                if (t == 0u) s_to = 0u;
                __syncthreads();
                if (t < kCols && t > from && s_start[t] - w0 <= kExpandPairs) atomicMax(&s_to, t);
                __syncthreads();
                upto = s_to;
            }
            const uint32_t w1 = s_start[upto];
            if (total <= kExpandPairs) {
#pragma unroll
                for (uint32_t q = 0; q < kChunk / T; q++) {
                    const uint32_t w = q * (T / 64u) + wave;
                    const uint32_t len = w * 64u + lane < c.runs ? (c.pk[q] & 255u) + 1u : 0u;
                    const uint32_t incl = wave_incl_add_u32(len), first = incl - len;
                    const uint32_t pairs = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
                    s_shift[wave][lane] = (c.pk[q] >> 8) - first;  // a pair's column less its place
                    wave_lds_fence();
                    for (uint32_t p0 = 0; p0 < pairs; p0 += 64u) {
                        // the run of pair p0 + lane: the word's runs are its
                        // first lanes, so it is the number of runs that start at
                        // or before the pair, less one
                        const uint32_t d = first - p0;
                        const bool starts = len != 0u && d < 64u;
                        const uint64_t earlier = __builtin_amdgcn_ballot_w64(len != 0u && first < p0);
                        const uint32_t bit = starts ? 1u << (d & 31u) : 0u;
                        const uint32_t lo = wave_or_u32(d < 32u ? bit : 0u), hi = wave_or_u32(d < 32u ? 0u : bit);
                        const uint64_t at_start = ((uint64_t)hi << 32) | lo;
                        const uint32_t run = (uint32_t)__popcll(earlier) + lanes_below(at_start) +
                                             (uint32_t)((at_start >> lane) & 1ull) - 1u;
                        const uint32_t i = p0 + lane;
                        if (i < pairs) {
                            const uint32_t x = i + s_shift[wave][run];
                            const uint64_t below = s_open[w][x] & ((1ull << run) - 1ull);
                            s_pair[s_before[w][x] + (uint32_t)__popcll(below)] = x << 16 | w * 64u | run;
                        }
                    }
                    wave_lds_fence();
                }
            } else {
                for (uint32_t i = wave; i < kChunkWords * (kCols / 64u); i += T / 64u) {
                    const uint32_t w = i / (kCols / 64u), x = (i % (kCols / 64u)) * 64u + lane;
                    if (x >= from && x < upto) {
                        uint64_t m = s_open[w][x];
                        uint32_t at = s_start[x] - w0 + s_before[w][x];
                        const uint32_t v = x << 16 | w * 64u;
                        while (m) {
                            s_pair[at++] = v + (uint32_t)__builtin_ctzll(m);
                            m &= m - 1ull;
                        }
                    }
                }
            }
            __syncthreads();
#pragma unroll
            for (uint32_t q = 0; q < kChunk / T; q++) asm volatile("" : "+v"(ahead.pk[q]), "+v"(ahead.id[q]));
            asm volatile("" : "+v"(ahead.to));
            for (uint32_t i = t; i < w1 - w0; i += T) {
                const uint32_t v = s_pair[i], x = v >> 16;
                const uint32_t at = s_delta[x] + w0 + i;
                if (at < m_cap) {  // always: the counts partition the pairs
                    cgids[at] = s_id[v & 0xFFFFu];
                    tile_ids[at] = c.row * tile_bw + x;
                }
            }
            __syncthreads();
            from = upto;
        }
        if (!more) break;
        c = ahead;
        k = next;
    }
}

size_t tile_runs_plan(uint32_t num_splats, uint32_t tile_bh, TileRuns* r) {
    r->parts = std::max(1u, div_up(num_splats, 256));
    r->block_parts = 16u;
    while ((uint64_t)r->block_parts * r->block_parts < r->parts) r->block_parts *= 2u;
    r->radix = 2u;
    while (r->radix <= tile_bh) r->radix *= 2u;
    return (size_t)div_up(r->parts, r->block_parts) * r->radix;
}

void tile_runs_chunks(uint32_t m, uint32_t tile_bh, uint32_t* chunk_group, size_t* chunks, size_t* groups) {
    // about 4,096 groups where runs hold four pairs
    *chunk_group = std::min(16u, std::max(1u, div_up(m / (4u * kChunk), 4096u)));
    *groups = (size_t)m / ((size_t)kChunk * *chunk_group) + tile_bh;
    *chunks = *groups * *chunk_group;
}

bh_status sort_tile_runs(bh_ctx* ctx, const TileRuns& r, uint32_t tile_bw, uint32_t tile_bh, const uint32_t* cum,
                         uint32_t num_visible, const uint32_t* dev, uint32_t m_cap, uint32_t* tile_ids,
                         uint32_t* cgids, uint32_t* offsets) {
    launch_radix_scan(ctx, "tile_runs_scan", r.counts, r.blk, r.parts, r.block_parts, r.radix);
    uint32_t row_bits = 0;
    while ((1u << row_bits) < tile_bh) row_bits++;
    {
        KernelTimer t(ctx, "tile_runs_scatter");
        launch(ctx, scatter_runs_kernel, dim3(r.parts), dim3(256), 0u, r, cum, num_visible, dev, row_bits, m_cap);
    }
    const uint64_t most = (uint64_t)m_cap / kChunk + tile_bh;  // chunks at most
    {
        KernelTimer t(ctx, "tile_runs_count");
        launch(ctx, count_runs_kernel, dim3((uint32_t)std::min<uint64_t>(most, 2048u)), dim3(256), 0u, r, tile_bh);
    }
    {
        KernelTimer t(ctx, "tile_runs_offsets");
        launch(ctx, scan_tiles_kernel, dim3(tile_bh), dim3(256), 0u, r, tile_bw, tile_bh, offsets);
    }
    KernelTimer t(ctx, "tile_runs_expand");
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((most + 7u) / 8u * 8u, 512u);
    launch(ctx, expand_runs_kernel, dim3(blocks), dim3(kExpandThreads), 0u, r, tile_bw, tile_bh, m_cap, tile_ids, cgids);
    return check_launch(ctx, "tile runs");
}

}  // namespace bh
