// Binning of packed tile rectangles by tile rows, for gfx950.
//
// A rectangle of w x h tiles is h runs of w consecutive tiles.  Instead of
// emitting its w h (tile, id) pairs and radix sorting them, the rectangles are
// split in two steps, each one a counting sort of intervals:
//  1. every Gaussian's row interval [y0, y0 + h) puts one 8-byte run
//     (id, x0 | w << 16) into the segment of each of its tile rows;
//  2. within a row segment every run's column interval [x0, x0 + w) puts the
//     id into the list of each of its tiles.
// A step counts with differences (+1 at the interval's begin, -1 at its end,
// one prefix sum per partition), so counting costs two LDS atomics per
// interval, however long it is, and the pairs themselves exist only as the
// final ids: per pair 4 bytes are written, per run 8 are written and read
// twice.  The pair sort this replaces moved 52 bytes per pair (8 written by
// the emission, 16 by each pass, 4 read by a counting pass and by the edges,
// 4 read again): at 1M Gaussians and 1080p (6.6M pairs, 1.9M runs) its kernels
// took 126 us and these take 62; at 3M large Gaussians 1540 us, and 445 in the
// stable form, after a depth sort of 150, which also replaces 3440 us of
// ordering the tiles' runs.  What bounds the placements is LDS (the
// per-pair accesses and their bank conflicts) and its latency: the arrays leave
// room for five workgroups per CU, six of the column placements of up to 128
// columns, four of the stable row placement of more.
//
// Stable form (STABLE): the intervals of a partition are placed in their
// order, by 64-lane column masks in LDS (an interval's rank in a column is the
// population count of the mask below its lane), so that Gaussians given in
// depth order leave every tile's list in depth order.  The masks come from two
// toggles per interval and a prefix xor over the columns (column_masks; an LDS
// atomic per pair took 302 us instead of 284 for 97M pairs, and walks of the
// masks by lanes that own columns 301 to 485).  Otherwise one returning
// LDS atomic per pair places it (about half of the LDS work), and the order
// inside a tile is the caller's to set.
//
// A partition is 1024 intervals (512 took 31 us instead of 25 at 1M Gaussians:
// half as long runs of stores).  Its values are staged in LDS in column
// order (stable: half a partition at a time), so that each column's values are
// stored contiguously; with more values than the stage holds (long intervals,
// whose columns then hold many values anyway) they are stored directly.
#include "common.hpp"

namespace jsa {
namespace {

constexpr int kRbThreads = 256;
constexpr int kRbWaves = kRbThreads / kWave;
constexpr int kRbPart = kRowBinPart;                // intervals per partition
constexpr int kRbPer = kRbPart / kRbThreads;        // and per lane
static_assert(kRowBinAxis == kRbThreads, "one thread per column");

// Columns (rows) that the LDS arrays hold: 128 up to 128 tiles, which leaves
// room for more workgroups per CU, else 256.
inline bool narrow(int tiles) { return tiles <= 128; }

struct Interval {
    int lo, len;        // columns [lo, lo + len) (len = 0: none)
};

__device__ __forceinline__ void add_differences(int* v, int ncols, Interval iv) {
    if (iv.len <= 0) return;
    atomicAdd(&v[iv.lo], 1);
    if (iv.lo + iv.len < ncols) atomicAdd(&v[iv.lo + iv.len], -1);
}

// LDS of one round of a placement: values V, staged up to CAP of them.
template <typename V, int COLS, int CAP, bool STABLE>
struct PlaceShared {
    // per wave and column: differences, counts, then the next position (relative
    // to the round's first value in column order)
    alignas(16) int cnt[kRbWaves][COLS];
    // STABLE: the lanes (low, high word) that cover a column; two arrays, so
    // that the columns of a wave spread over all banks (one of 16-byte cells
    // with the position: 301 us instead of 284, at 256 columns 204 for 144)
    uint32_t lo[STABLE ? kRbWaves : 1][STABLE ? COLS : 1];
    uint32_t hi[STABLE ? kRbWaves : 1][STABLE ? COLS : 1];
    int first[COLS + 1];            // column c's values are first[c] .. first[c + 1]
    int delta[COLS];                // and go to delta[c] + position
    V out[CAP];
    uint32_t tmp[kRbWaves];
};

// Per-column counts of a wave's own intervals: v[c] holds the differences on
// entry and the counts on return; COLS / 64 columns per lane.
template <int COLS>
__device__ __forceinline__ void wave_counts(int* v, int lane) {
    if constexpr (COLS == 256) {
        int4* q = reinterpret_cast<int4*>(v) + lane;
        int4 d = *q;
        d.y += d.x;
        d.z += d.y;
        d.w += d.z;
        const int before = wave_inclusive_sum(d.w) - d.w;
        *q = make_int4(d.x + before, d.y + before, d.z + before, d.w + before);
    } else {
        static_assert(COLS == 128, "2 or 4 columns per lane");
        int2* q = reinterpret_cast<int2*>(v) + lane;
        int2 d = *q;
        d.y += d.x;
        const int before = wave_inclusive_sum(d.y) - d.y;
        *q = make_int2(d.x + before, d.y + before);
    }
}

template <typename V, int COLS, int CAP, bool STABLE>
__device__ __forceinline__ void clear_place(PlaceShared<V, COLS, CAP, STABLE>& sh) {
    if ((int)threadIdx.x < COLS) {
#pragma unroll
        for (int w = 0; w < kRbWaves; ++w) sh.cnt[w][threadIdx.x] = 0;
    }
}

// Inclusive prefix xor over the 64 lanes (full EXEC), by the DPP row shifts and
// row broadcasts.
__device__ __forceinline__ uint32_t wave_xor_scan(uint32_t v) {
    int a = (int)v;
    a ^= __builtin_amdgcn_update_dpp(0, a, 0x111, 0xf, 0xf, true);
    a ^= __builtin_amdgcn_update_dpp(0, a, 0x112, 0xf, 0xf, true);
    a ^= __builtin_amdgcn_update_dpp(0, a, 0x114, 0xf, 0xf, true);
    a ^= __builtin_amdgcn_update_dpp(0, a, 0x118, 0xf, 0xf, true);
    a ^= __builtin_amdgcn_update_dpp(0, a, 0x142, 0xa, 0xf, true);
    a ^= __builtin_amdgcn_update_dpp(0, a, 0x143, 0xc, 0xf, true);
    return (uint32_t)a;
}

// The lanes whose interval covers each of the calling lane's N columns (64 lanes
// times N consecutive ones): the intervals toggle their lane's bit at their begin
// and past their end, and a prefix xor over the columns turns the toggles into
// masks.  Two LDS atomics per interval, however long.  lo, hi: LDS of the wave,
// a word per column each.
template <int N>
__device__ __forceinline__ void column_masks(Interval iv, uint32_t* lo, uint32_t* hi,
                                             uint64_t* mask) {
    constexpr int COLS = N * kWave;
    const int lane = lane_id(), c0 = lane * N;
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < N; ++j) {
        lo[c0 + j] = 0u;
        hi[c0 + j] = 0u;
    }
    wave_lds_sync();
    if (iv.len > 0) {
        uint32_t* own = lane < 32 ? lo : hi;
        const uint32_t bit = 1u << (lane & 31);
        atomicXor(&own[iv.lo], bit);
        if (iv.lo + iv.len < COLS) atomicXor(&own[iv.lo + iv.len], bit);
    }
    wave_lds_sync();
    uint32_t l[N], h[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        l[j] = lo[c0 + j] ^ (j > 0 ? l[j > 0 ? j - 1 : 0] : 0u);
        h[j] = hi[c0 + j] ^ (j > 0 ? h[j > 0 ? j - 1 : 0] : 0u);
    }
    const uint32_t bl = wave_xor_scan(l[N - 1]) ^ l[N - 1];
    const uint32_t bh = wave_xor_scan(h[N - 1]) ^ h[N - 1];
#pragma unroll
    for (int j = 0; j < N; ++j)
        mask[j] = (uint64_t)(l[j] ^ bl) | (uint64_t)(h[j] ^ bh) << 32;
}

// One round of a placement: val[k] of interval iv[k] (k-th 64-lane block of
// the wave's PER * 64 intervals) into every column of the interval.  Column c's
// values go to out_g[column_base(thread c) ..) in interval order (STABLE) or
// any order.  Nothing is written at or past cap.  Returns the number of the
// thread's column's values.  Called by the whole workgroup with cleared LDS;
// ends with a barrier.
template <int PER, typename V, int COLS, int CAP, bool STABLE>
__device__ __forceinline__ int place(PlaceShared<V, COLS, CAP, STABLE>& sh, const Interval* iv,
                                     const V* val, int ncols, int column_base, V* out_g,
                                     int cap) {
    constexpr int N = COLS / kWave;
    const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
    uint64_t mask[STABLE ? PER : 1][N];
    if constexpr (STABLE) {
        int cnt[N] = {};
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            column_masks<N>(iv[k], sh.lo[wave], sh.hi[wave], mask[k]);
#pragma unroll
            for (int j = 0; j < N; ++j) cnt[j] += __popcll(mask[k][j]);
        }
#pragma unroll
        for (int j = 0; j < N; ++j) sh.cnt[wave][lane * N + j] = cnt[j];
    } else {
#pragma unroll
        for (int k = 0; k < PER; ++k) add_differences(sh.cnt[wave], COLS, iv[k]);
        wave_lds_sync();
        wave_counts<COLS>(sh.cnt[wave], lane);
    }
    __syncthreads();
    int total = 0, before[kRbWaves];
#pragma unroll
    for (int w = 0; w < kRbWaves; ++w) {
        before[w] = total;
        total += tid < COLS ? sh.cnt[w][tid] : 0;
    }
    const int first = (int)block_exclusive_scan256((uint32_t)total, sh.tmp);
    if (tid < COLS) {
#pragma unroll
        for (int w = 0; w < kRbWaves; ++w) sh.cnt[w][tid] = first + before[w];
        sh.first[tid] = first;
        sh.delta[tid] = column_base - first;
    }
    if (tid == COLS - 1) sh.first[COLS] = first + total;
    __syncthreads();
    const bool staged = sh.first[COLS] <= CAP;      // uniform
    auto put = [&](int c, int pos, const V& v) {
        if (staged) {
            sh.out[pos] = v;
        } else {
            const uint32_t at = (uint32_t)sh.delta[c] + (uint32_t)pos;
            if (at < (uint32_t)cap) out_g[at] = v;
        }
    };
    int* pos = sh.cnt[wave];
    int next[N];
    if constexpr (STABLE) {
#pragma unroll
        for (int j = 0; j < N; ++j) next[j] = pos[lane * N + j];
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const Interval me = iv[k];
        if constexpr (STABLE) {
            uint32_t* lo = sh.lo[wave];
            uint32_t* hi = sh.hi[wave];
            wave_lds_sync();
#pragma unroll
            for (int j = 0; j < N; ++j) {
                lo[lane * N + j] = (uint32_t)mask[k][j];
                hi[lane * N + j] = (uint32_t)(mask[k][j] >> 32);
                pos[lane * N + j] = next[j];
                next[j] += __popcll(mask[k][j]);
            }
            wave_lds_sync();
            const uint32_t bit = 1u << (lane & 31);
            const uint32_t mlo = lane < 32 ? bit - 1u : ~0u, mhi = lane < 32 ? 0u : bit - 1u;
            for (int i = 0; i < me.len; ++i) {
                const int c = me.lo + i;
                put(c, pos[c] + __popc(lo[c] & mlo) + __popc(hi[c] & mhi), val[k]);
            }
        } else {
            for (int i = 0; i < me.len; ++i) {
                const int c = me.lo + i;
                put(c, atomicAdd(&pos[c], 1), val[k]);
            }
        }
    }
    __syncthreads();
    if (staged) {
        // 16 lanes per column: a column's values are one contiguous run
        for (int c = tid >> 4; c < ncols; c += kRbThreads / 16) {
            const int end = sh.first[c + 1];
            const uint32_t to = (uint32_t)sh.delta[c];
            for (int i = sh.first[c] + (tid & 15); i < end; i += 16)
                if (to + (uint32_t)i < (uint32_t)cap) out_g[to + (uint32_t)i] = sh.out[i];
        }
    }
    __syncthreads();
    return total;
}

// A partition's intervals in rounds of PER per lane: the stage of a stable
// placement (whose masks take LDS too) holds half a partition.  Returns where the
// thread's column's values end.
template <int PER, typename V, int COLS, int CAP, bool STABLE>
__device__ __forceinline__ int place_all(PlaceShared<V, COLS, CAP, STABLE>& sh,
                                          const Interval* iv, const V* val, int ncols,
                                          int column_base, V* out_g, int cap) {
    static_assert(kRbPer % PER == 0, "whole rounds");
#pragma unroll
    for (int r = 0; r < kRbPer; r += PER) {
        if (r > 0) {
            clear_place(sh);
            __syncthreads();
        }
        column_base = clamped_sum(
            column_base,
            (uint32_t)place<PER>(sh, iv + r, val + r, ncols, column_base, out_g, cap), cap);
    }
    return column_base;
}
// Interval k (of kRbPer) of a lane, in rounds of PER: its index within the
// partition.
template <int PER>
__device__ __forceinline__ int interval_index(int k) {
    const int wave = threadIdx.x >> 6, lane = lane_id();
    return (k / PER) * (PER * kRbThreads) + wave * (PER * kWave) + (k % PER) * kWave + lane;
}
constexpr int round_per(bool stable) { return stable ? 2 : kRbPer; }

// A Gaussian's rectangle clipped to the grid (a rectangle outside it, never
// the projection's, sets bit 4 of err).
__device__ __forceinline__ uint2 grid_rect(uint2 rc, int tiles_x, int tiles_y, bool& bad) {
    int x0, x1, y0, y1;
    unpack_rect(rc, x0, x1, y0, y1);
    bad = rect_count(rc) > 0 && (x1 > tiles_x || y1 > tiles_y);
    if (!bad) return rc;
    x0 = min(x0, tiles_x);
    x1 = min(x1, tiles_x);
    y0 = min(y0, tiles_y);
    y1 = min(y1, tiles_y);
    return pack_rect(x0, x1, y0, y1);
}

// Where the pairs exceed the capacity, the first cap of them in emission order
// (Gaussian by Gaussian, a rectangle row by row) are binned: the Gaussians before
// `id` whole, of `id` the first `rows` rows, of the last of them (tile row `row`)
// the first `width` tiles, the others not at all.  id = n, row = -1: all pairs.
struct Cut {
    int id, rows, row, width;
};
// cum: the inclusive tile counts in id order (one load where nothing is cut).
__device__ __forceinline__ Cut emission_cut(const int* __restrict__ cum,
                                            const uint2* __restrict__ rects, int n, int cap) {
    if ((uint32_t)cum[n - 1] <= (uint32_t)cap) return {n, 0, -1, 0};
    int id = 0, hi = n - 1;         // the first id whose count exceeds cap
    while (id < hi) {
        const int mid = (id + hi) >> 1;
        if ((uint32_t)cum[mid] > (uint32_t)cap) hi = mid;
        else id = mid + 1;
    }
    const uint2 rc = rects[id];
    const uint32_t w = rc.y & 0xFFFFu;
    const uint32_t left =
        min((uint32_t)cap - (id > 0 ? (uint32_t)cum[id - 1] : 0u), rect_count(rc));
    const int rows = w > 0 ? (int)((left + w - 1) / w) : 0;
    if (rows == 0) return {id, 0, -1, 0};
    return {id, rows, (int)(rc.x >> 16) + rows - 1, (int)(left - (uint32_t)(rows - 1) * w)};
}
// Gaussian id's rectangle up to the cut (its last row whole: cut_run).
__device__ __forceinline__ uint2 cut_rect(uint2 rc, uint32_t id, const Cut& cut) {
    if (id < (uint32_t)cut.id) return rc;
    const uint32_t rows = id == (uint32_t)cut.id ? (uint32_t)cut.rows : 0u;
    return make_uint2(rc.x, (rc.y & 0xFFFFu) | min(rc.y >> 16, rows) << 16);
}
// The width of the cut's last row into its run (id, x0 | w << 16).
__device__ __forceinline__ void cut_run(uint2& run, const Cut& cut) {
    run.y = (run.y & 0xFFFFu) | min(run.y >> 16, (uint32_t)cut.width) << 16;
}

// Step 1, counting: partition b holds the Gaussians perm[1024 b ..) (the ids
// themselves where perm is null).  counts[row * row_stride + b * part_stride] =
// its runs per row,
// part_tot[b] = its pairs; with perm, in_order[i] = the rectangle of perm[i],
// so that the random gather is paid once (and up to the cut).  Also clears the tile
// bins and the error word and keeps the cut for the steps after it.
__global__ __launch_bounds__(kRbThreads) void row_count_kernel(
    int n, const uint32_t* __restrict__ perm, const uint2* __restrict__ rects,
    const int* __restrict__ cum, int cap, int tiles_x, int tiles_y, int row_stride,
    int part_stride, uint32_t* __restrict__ counts, uint32_t* __restrict__ part_tot,
    uint2* __restrict__ in_order, int num_tiles, int2* __restrict__ bins,
    Cut* __restrict__ cut_out, uint32_t* __restrict__ err) {
    __shared__ int s_d[kRbThreads];
    __shared__ uint32_t s_tmp[kRbWaves];
    const int tid = threadIdx.x, part = blockIdx.x;
    for (int t = part * kRbThreads + tid; t < num_tiles; t += gridDim.x * kRbThreads)
        bins[t] = make_int2(0, 0);
    uint2 rc[kRbPer];
    uint32_t id[kRbPer];
#pragma unroll
    for (int k = 0; k < kRbPer; ++k) {
        const int i = part * kRbPart + k * kRbThreads + tid;
        id[k] = i < n ? (perm ? perm[i] : (uint32_t)i) : 0u;
        rc[k] = i < n ? rects[id[k]] : make_uint2(0u, 0u);
    }
    const Cut cut = emission_cut(cum, rects, n, cap);
    if (part == 0 && tid == 0) {
        *err = 0u;
        *cut_out = cut;
    }
    s_d[tid] = 0;
    __syncthreads();
    uint32_t pairs = 0;
#pragma unroll
    for (int k = 0; k < kRbPer; ++k) {
        const int i = part * kRbPart + k * kRbThreads + tid;
        bool bad;
        pairs += rect_count(rc[k]);
        const uint2 kept = cut_rect(rc[k], id[k], cut);
        if (perm && i < n) in_order[i] = kept;
        const uint2 r = grid_rect(kept, tiles_x, tiles_y, bad);
        if (rect_count(r) > 0)
            add_differences(s_d, kRbThreads, {(int)(r.x >> 16), (int)(r.y >> 16)});
    }
    __syncthreads();
    const uint32_t d = (uint32_t)s_d[tid];
    const uint32_t c = block_exclusive_scan256(d, s_tmp) + d;      // wraps back to the count
    if (tid < tiles_y) counts[(size_t)tid * row_stride + (size_t)part * part_stride] = c;
    const uint32_t t = block_exclusive_scan256(pairs, s_tmp) + pairs;
    if (tid == kRbThreads - 1) part_tot[part] = t;
}

// Step 1, placement: the runs of partition b into the row segments, which lie
// end to end in runs[0 .. sum of row_len).  rects in perm's order; counts: exclusive
// over the partitions of a row (column_scan), row_len their totals, or with fold the
// counts themselves, and workgroup 0 writes row_len.  Workgroup 0 also writes the
// exact pair total and bit 8 of err where it exceeds cap.
template <bool STABLE, int COLS>
__global__ __launch_bounds__(kRbThreads) void row_place_kernel(
    int n, const uint32_t* __restrict__ perm, const uint2* __restrict__ rects, int tiles_x,
    int tiles_y, int parts, bool fold, const uint32_t* __restrict__ counts,
    uint32_t* __restrict__ row_len, const uint32_t* __restrict__ part_tot,
    uint2* __restrict__ runs, int cap, const Cut* __restrict__ cut_in,
    unsigned long long* __restrict__ total_out, uint32_t* __restrict__ err) {
    constexpr int PER = round_per(STABLE);
    __shared__ PlaceShared<uint2, COLS, 3072, STABLE> sh;
    __shared__ uint64_t s_sum[kRbWaves];
    const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6, part = blockIdx.x;
    Interval iv[kRbPer];
    uint2 val[kRbPer];
    bool bad_any = false;
    const Cut cut = *cut_in;
#pragma unroll
    for (int k = 0; k < kRbPer; ++k) {
        const int i = part * kRbPart + interval_index<PER>(k);
        const uint32_t id = i < n ? (perm ? perm[i] : (uint32_t)i) : 0u;
        bool bad;
        const uint2 rc = grid_rect(cut_rect(i < n ? rects[i] : make_uint2(0u, 0u), id, cut),
                                   tiles_x, tiles_y, bad);
        bad_any = bad_any || bad;
        iv[k].lo = (int)(rc.x >> 16);
        iv[k].len = rect_count(rc) > 0 ? (int)(rc.y >> 16) : 0;
        val[k] = make_uint2(id, (rc.x & 0xFFFFu) | (rc.y << 16));
    }
    if (bad_any) atomicOr(err, 4u);
    clear_place(sh);
    // (the rows' runs may sum past 32 bits: positions past cap are all alike)
    uint2 own = make_uint2(0u, 0u);         // before this partition, of the row
    if (tid < tiles_y)
        own = fold ? fold_counts(counts, parts, part, tid)
                   : make_uint2(counts[(size_t)tid * parts + part], row_len[tid]);
    if (fold && part == 0 && tid < tiles_y) row_len[tid] = own.y;
    const uint64_t at = block_exclusive_scan256((uint64_t)own.y, s_sum) + own.x;
    const int base = (int)min(at, (uint64_t)cap);
    const int past = place_all<PER>(sh, iv, val, tiles_y, base, runs, cap);
    if ((unsigned)cut.row < (unsigned)tiles_y) {    // uniform: more pairs than the capacity
        // the run of the cut's last row, if it is among this partition's, which are
        // [base, past) of the row's thread
        if (tid == cut.row) {
            sh.first[0] = base;
            sh.first[1] = past;
        }
        __syncthreads();
        for (int i = sh.first[0] + tid; i < sh.first[1]; i += kRbThreads)
            if (runs[i].x == (uint32_t)cut.id) cut_run(runs[i], cut);
    }
    if (part != 0) return;
    uint64_t sum = 0;
    for (int i = tid; i < parts; i += kRbThreads) sum += part_tot[i];
    sum = wave_inclusive_sum(sum);
    if (lane == kWave - 1) s_sum[wave] = sum;
    __syncthreads();
    if (tid == 0) {
        sum = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
        *total_out = (unsigned long long)sum;
        if (sum > (uint64_t)cap) atomicOr(err, 8u);
    }
}

// Step 2's partitions: row r's runs [e0[r], e0[r + 1]) in partitions
// [p0[r], p0[r + 1]) of up to kRbPart, none at or past cap.
struct RowTable {
    int e0[kRowBinAxis + 1], p0[kRowBinAxis + 1];
};

// Called by the whole workgroup (kRbThreads threads); ends with a barrier.
__device__ __forceinline__ void row_table(RowTable& rt, const uint32_t* __restrict__ row_len,
                                          int tiles_y, int cap, uint64_t* s_tmp) {
    const int tid = threadIdx.x;
    const uint64_t len = tid < tiles_y ? row_len[tid] : 0u;
    const uint64_t e = block_exclusive_scan256(len, s_tmp);
    const uint64_t lim = (uint64_t)cap;
    const uint64_t b = min(e, lim), n = min(e + len, lim) - b;
    const uint64_t np = (n + kRbPart - 1) / kRbPart;
    const uint64_t p = block_exclusive_scan256(np, s_tmp);
    rt.e0[tid] = (int)b;
    rt.p0[tid] = (int)p;
    if (tid == kRbThreads - 1) {
        rt.e0[kRowBinAxis] = (int)(b + n);
        rt.p0[kRowBinAxis] = (int)(p + np);
    }
    __syncthreads();
}

// The row of partition p (largest r with p0[r] <= p; an empty row's p0 equals
// the next one's, so the search lands on the row that holds p).
__device__ __forceinline__ int row_of(const RowTable& rt, int p) {
    int lo = 0, hi = kRowBinAxis;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (rt.p0[mid] <= p) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Persistent walk over the partitions: XCD x (workgroups are dealt round
// robin) takes a contiguous band, so that the partial lines of one row's lists
// meet in one L2.
template <typename F>
__device__ __forceinline__ void for_partitions(int total, F body) {
    const int per = (total + 7) / 8, x = blockIdx.x & 7;
    for (int q = blockIdx.x >> 3; q < per; q += gridDim.x >> 3) {
        const int p = x * per + q;
        if (p < total) body(p);
    }
}

// counts[column] = the runs [begin, end) that cover the column, all 256 of them.
// Called by the whole workgroup.
__device__ __forceinline__ void count_columns(const uint2* __restrict__ runs, int begin, int end,
                                              int* s_d, uint32_t* s_tmp,
                                              uint32_t* __restrict__ counts) {
    const int tid = threadIdx.x;
    uint32_t w[kRbPer];
#pragma unroll
    for (int k = 0; k < kRbPer; ++k) {
        const int i = k * kRbThreads + tid;
        w[k] = i < end - begin ? runs[begin + i].y : 0u;
    }
    s_d[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kRbPer; ++k)
        add_differences(s_d, kRbThreads, {(int)(w[k] & 0xFFFFu), (int)(w[k] >> 16)});
    __syncthreads();
    const uint32_t d = (uint32_t)s_d[tid];
    const uint32_t c = block_exclusive_scan256(d, s_tmp) + d;
    counts[tid] = c;
}

// Step 2, counting: counts[p * 256 + column] = the runs of partition p that
// cover the column; desc[p] = (row, first run, end, whether it is the row's
// first partition), desc[-1].x the number of partitions.
__global__ __launch_bounds__(kRbThreads) void col_count_kernel(
    const uint2* __restrict__ runs, const uint32_t* __restrict__ row_len, int tiles_y, int cap,
    uint32_t* __restrict__ counts, int4* __restrict__ desc) {
    __shared__ RowTable rt;
    __shared__ int s_d[kRbThreads];
    __shared__ uint32_t s_tmp[kRbWaves];
    __shared__ uint64_t s_tmp64[kRbWaves];
    const int tid = threadIdx.x;
    row_table(rt, row_len, tiles_y, cap, s_tmp64);
    if (blockIdx.x == 0 && tid == 0) desc[-1] = make_int4(rt.p0[kRowBinAxis], 0, 0, 0);
    for_partitions(rt.p0[kRowBinAxis], [&](int p) {
        const int r = row_of(rt, p);
        const int begin = rt.e0[r] + (p - rt.p0[r]) * kRbPart;
        const int end = part_end(begin, rt.e0[r + 1], kRbPart);
        if (tid == 0) desc[p] = make_int4(r, begin, end, p == rt.p0[r] ? 1 : 0);
        count_columns(runs, begin, end, s_d, s_tmp, counts + (size_t)p * kRowBinAxis);
    });
}

constexpr int kScanThreads = 1024;
struct ScanShared {
    uint32_t sum[kScanThreads];
    uint64_t w[kRbWaves];
};
// The counts of partitions [p0, p0 + parts), 256 columns each of which the first
// COLS may be set, become each partition's first position in its column's list,
// relative to the columns' first; first_out[c] the column's first position, [256]
// the total (all at most cap).  1024 / COLS groups of threads share the
// partitions, whose loads are what it waits for (489 partitions of 50 rows: 26 us
// with four groups of 256 columns, 11 with sixteen of 64).
template <int COLS>
__device__ __forceinline__ void scan_columns(ScanShared& sh, int p0, int parts, int cap,
                                             uint32_t* __restrict__ counts,
                                             uint32_t* __restrict__ first_out) {
    constexpr int kGroups = kScanThreads / COLS;
    const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
    const int c = tid & (COLS - 1), g = tid / COLS;
    const uint64_t lim = (uint64_t)cap;
    const int q0 = p0 + (int)((long long)parts * g / kGroups);
    const int q1 = p0 + (int)((long long)parts * (g + 1) / kGroups);
    uint32_t sum = 0;
#pragma unroll 8
    for (int q = q0; q < q1; ++q) sum += counts[(size_t)q * kRowBinAxis + c];
    sh.sum[tid] = sum;
    __syncthreads();
    uint64_t total = 0, before = 0;
#pragma unroll
    for (int k = 0; k < kGroups; ++k) {
        const uint32_t v = sh.sum[k * COLS + c];
        before += k < g ? v : 0u;
        total += v;
    }
    // exclusive over the columns (every group computes the same)
    const uint64_t incl = wave_inclusive_sum(total);
    if (g == 0 && lane == kWave - 1) sh.w[wave] = incl;
    __syncthreads();
    uint64_t first = incl - total, all = 0;
#pragma unroll
    for (int w = 0; w < COLS / kWave; ++w) {
        first += w < (c >> 6) ? sh.w[w] : 0u;
        all += sh.w[w];
    }
    if (tid <= kRowBinAxis) first_out[tid] = (uint32_t)min(tid < COLS ? first : all, lim);
    uint64_t run = first + before;
#pragma unroll 8
    for (int q = q0; q < q1; ++q) {
        const size_t at = (size_t)q * kRowBinAxis + c;
        const uint32_t v = counts[at];
        counts[at] = (uint32_t)min(run, lim);
        run += v;
    }
}
// The instantiation for columns [0, n).
#define JSA_SCAN(n, LAUNCH)                                                                   \
    do {                                                                                      \
        if ((n) <= 64) LAUNCH(64);                                                            \
        else if ((n) <= 128) LAUNCH(128);                                                     \
        else LAUNCH(256);                                                                     \
    } while (0)

// Step 2, offsets, one workgroup per row: counts become each partition's first
// position in the column's list, relative to the row's first pair;
// tile_first[row * 257 + column] the tile's first position, [.. + 256] the
// row's pairs (all at most cap).
template <int COLS>
__global__ __launch_bounds__(kScanThreads) void col_scan_kernel(
    const uint32_t* __restrict__ row_len, int tiles_y, int cap,
    uint32_t* __restrict__ counts, uint32_t* __restrict__ tile_first) {
    __shared__ ScanShared sh;
    __shared__ uint64_t s_e[kRbWaves], s_p[kRbWaves];
    __shared__ int s_range[2];
    const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
    const int c = tid & (kRowBinAxis - 1), g = tid / kRowBinAxis, row = blockIdx.x;
    // this row's partitions (row_table's numbers, by the first 256 threads)
    const uint64_t lim = (uint64_t)cap;
    uint64_t len = 0, e = 0, np = 0, p = 0;
    if (g == 0) {
        len = c < tiles_y ? row_len[c] : 0u;
        e = wave_inclusive_sum(len);
        if (lane == kWave - 1) s_e[wave] = e;
    }
    __syncthreads();
    if (g == 0) {
        for (int w = 0; w < wave; ++w) e += s_e[w];
        const uint64_t b = min(e - len, lim);
        np = (min(e, lim) - b + kRbPart - 1) / kRbPart;
        p = wave_inclusive_sum(np);
        if (lane == kWave - 1) s_p[wave] = p;
    }
    __syncthreads();
    if (g == 0) {
        for (int w = 0; w < wave; ++w) p += s_p[w];
        if (c == row) {
            s_range[0] = (int)(p - np);
            s_range[1] = (int)p;
        }
    }
    __syncthreads();
    scan_columns<COLS>(sh, s_range[0], s_range[1] - s_range[0], cap, counts,
                       tile_first + (size_t)row * (kRowBinAxis + 1));
}

// Step 2, placement: the ids of every partition's runs into the tiles' lists
// (rows end to end), and the bins of the rows that have runs.
template <bool STABLE, int COLS>
__global__ __launch_bounds__(kRbThreads) void col_place_kernel(
    const uint2* __restrict__ runs, const int4* __restrict__ desc, int tiles_x, int tiles_y,
    int cap, const uint32_t* __restrict__ counts, const uint32_t* __restrict__ tile_first,
    uint32_t* __restrict__ ids, int2* __restrict__ bins) {
    constexpr int PER = round_per(STABLE);
    __shared__ PlaceShared<uint32_t, COLS, STABLE ? (COLS == 128 ? 4096 : 3072) : 5120, STABLE> sh;
    __shared__ int s_row0[kRowBinAxis];
    __shared__ uint64_t s_tmp[kRbWaves];
    const int tid = threadIdx.x;
    const uint64_t pairs =
        tid < tiles_y ? tile_first[(size_t)tid * (kRowBinAxis + 1) + kRowBinAxis] : 0u;
    s_row0[tid] = (int)min(block_exclusive_scan256(pairs, s_tmp), (uint64_t)cap);
    const int parts = uniform_i(desc[-1].x);
    for_partitions(parts, [&](int p) {
        const int4 d = desc[p];
        Interval iv[kRbPer];
        uint32_t id[kRbPer];
#pragma unroll
        for (int k = 0; k < kRbPer; ++k) {
            const int i = interval_index<PER>(k);
            const uint2 run = i < d.z - d.y ? runs[d.y + i] : make_uint2(0u, 0u);
            id[k] = run.x;
            iv[k] = {(int)(run.y & 0xFFFFu), (int)(run.y >> 16)};
        }
        clear_place(sh);
        __syncthreads();
        const int row0 = s_row0[d.x];
        const int base =
            tid < tiles_x ? clamped_sum(row0, counts[(size_t)p * kRowBinAxis + tid], cap) : 0;
        if (d.w && tid < tiles_x) {
            const uint32_t* tf = tile_first + (size_t)d.x * (kRowBinAxis + 1) + tid;
            const int b = clamped_sum(row0, tf[0], cap), e = clamped_sum(row0, tf[1], cap);
            if (e > b) bins[d.x * tiles_x + tid] = make_int2(b, e);
        }
        place_all<PER>(sh, iv, id, tiles_x, base, ids, cap);
    });
}

// ---- batches ----
// The same two steps over the items of many views: a partition of items lies in
// one view, a "row" is a tile row of a view, r = the view's row_off + y, and the
// offsets that one view's workgroups find by themselves come from tables.  (Rows
// of the tallest view for every view: 2000 views of 32 x 32 and one of 4096 rows of
// pixels took 6370 us instead of 1270, and 1.1 GB more.)  12
// views of 500k Gaussians at 800 x 800 (26M pairs of 6M items): 192 us in eight
// launches, where emitting the pairs and sorting them by tile took 442 in
// thirteen; step 2552 -> 2280 us.

// The view that owns partition p.
__device__ __forceinline__ int view_of_part(const ViewRec* __restrict__ views, int num_views,
                                            int p) {
    int lo = 0, hi = num_views;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (views[mid].part_off <= p) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Step 1, counting (row_count_kernel): counts[p * 256 + y], part_tot[p].
__global__ __launch_bounds__(kRbThreads) void batch_row_count_kernel(
    const ViewRec* __restrict__ views, int num_views, const uint2* __restrict__ rects,
    uint32_t* __restrict__ counts, uint32_t* __restrict__ part_tot, int num_bins,
    int2* __restrict__ bins, uint32_t* __restrict__ err) {
    __shared__ int s_d[kRbThreads];
    __shared__ uint32_t s_tmp[kRbWaves];
    const int tid = threadIdx.x, part = blockIdx.x;
    if (part == 0 && tid == 0) *err = 0u;
    for (int t = part * kRbThreads + tid; t < num_bins; t += gridDim.x * kRbThreads)
        bins[t] = make_int2(0, 0);
    const ViewRec vr = views[view_of_part(views, num_views, part)];
    const int local = (part - vr.part_off) * kRbPart;
    s_d[tid] = 0;
    __syncthreads();
    uint32_t pairs = 0;
#pragma unroll
    for (int k = 0; k < kRbPer; ++k) {
        const int i = local + k * kRbThreads + tid;
        const uint2 rc = i < vr.n ? rects[vr.item_off + i] : make_uint2(0u, 0u);
        bool bad;
        pairs += rect_count(rc);
        const uint2 r = grid_rect(rc, vr.tiles_x, vr.tiles_y, bad);
        if (rect_count(r) > 0)
            add_differences(s_d, kRbThreads, {(int)(r.x >> 16), (int)(r.y >> 16)});
    }
    __syncthreads();
    const uint32_t d = (uint32_t)s_d[tid];
    counts[(size_t)part * kRowBinAxis + tid] = block_exclusive_scan256(d, s_tmp) + d;
    const uint32_t t = block_exclusive_scan256(pairs, s_tmp) + pairs;
    if (tid == kRbThreads - 1) part_tot[part] = t;
}

// Step 1, offsets: a view's rows are the columns of its partitions' counts;
// row_first[view * 257 + y] the row's first run, relative to the view's; row_len and
// row_view the runs and the view of every row.
template <int COLS>
__global__ __launch_bounds__(kScanThreads) void batch_row_scan_kernel(
    const ViewRec* __restrict__ views, int cap, uint32_t* __restrict__ counts,
    uint32_t* row_first, uint32_t* __restrict__ row_len, int* __restrict__ row_view) {
    __shared__ ScanShared sh;
    const ViewRec vr = views[blockIdx.x];
    uint32_t* first = row_first + (size_t)blockIdx.x * (kRowBinAxis + 1);
    scan_columns<COLS>(sh, vr.part_off, (vr.n + kRbPart - 1) / kRbPart, cap, counts, first);
    __syncthreads();            // first is written by several waves
    const int y = threadIdx.x;
    if (y < vr.tiles_y) {
        row_len[vr.row_off + y] = first[y + 1] - first[y];
        row_view[vr.row_off + y] = blockIdx.x;
    }
}

// Exclusive scan of get(0..n) by one workgroup of 1024 threads, in rounds;
// put(i, exclusive sum, value).  Returns the total.
template <typename G, typename P>
__device__ __forceinline__ uint64_t scan_rounds(int n, uint64_t* s_tmp, G get, P put) {
    uint64_t carry = 0;
    for (int b = 0; b < n; b += 1024) {
        const int i = b + (int)threadIdx.x;
        const uint64_t v = i < n ? get(i) : 0u;
        const uint64_t e = block_exclusive_scan<16>(v, s_tmp);
        if (i < n) put(i, carry + e, v);
        if (threadIdx.x == 1023) s_tmp[16] = e + v;
        __syncthreads();
        carry += s_tmp[16];
        __syncthreads();
    }
    return carry;
}

// Workgroup 0: every row's first run (row_off) and partition (row_part, R + 1
// entries) of step 2, and those partitions' descriptors (col_count_kernel's).
// Workgroup 1: every partition's first pair in item order (part_pair), and the
// totals: *total, *count = min(total, cap), bit 8 of err.
__global__ __launch_bounds__(1024) void batch_table_kernel(
    int rows, const uint32_t* __restrict__ row_len, int cap, int* __restrict__ row_off,
    int* __restrict__ row_part, int4* __restrict__ desc, int parts,
    const uint32_t* __restrict__ part_tot, uint32_t* __restrict__ part_pair,
    int* __restrict__ count, unsigned long long* __restrict__ total,
    uint32_t* __restrict__ err) {
    __shared__ uint64_t s_tmp[17];
    const uint64_t lim = (uint64_t)cap;
    if (blockIdx.x == 1) {
        const uint64_t sum = scan_rounds(
            parts, s_tmp, [&](int i) { return (uint64_t)part_tot[i]; },
            [&](int i, uint64_t e, uint64_t) { part_pair[i] = (uint32_t)min(e, lim); });
        if (threadIdx.x == 0) {
            *total = (unsigned long long)sum;
            *count = (int)min(sum, lim);
            if (sum > lim) atomicOr(err, 8u);
        }
        return;
    }
    auto len = [&](int r) { return (uint64_t)row_len[r]; };
    scan_rounds(rows, s_tmp, len, [&](int r, uint64_t e, uint64_t v) {
        row_off[r] = (int)min(e, lim);
        row_part[r] = part_count((int)min(e, lim), (int)min(e + v, lim), kRbPart);  // for now
    });
    const uint64_t all = scan_rounds(
        rows, s_tmp, [&](int r) { return (uint64_t)row_part[r]; },
        [&](int r, uint64_t e, uint64_t v) {
            row_part[r] = (int)e;
            const int begin = row_off[r];
            const int end = (int)min((uint64_t)begin + len(r), lim);
            for (int q = 0; q < (int)v; ++q) {
                const int at = begin + q * kRbPart;
                desc[(int)e + q] = make_int4(r, at, part_end(at, end, kRbPart), q == 0);
            }
        });
    if (threadIdx.x == 0) {
        row_part[rows] = (int)all;
        desc[-1] = make_int4((int)all, 0, 0, 0);
    }
}

// Step 1, placement (row_place_kernel), and every item's first pair.
template <int COLS>
__global__ __launch_bounds__(kRbThreads) void batch_row_place_kernel(
    const ViewRec* __restrict__ views, int num_views, const uint2* __restrict__ rects,
    const uint32_t* __restrict__ counts, const int* __restrict__ row_off, const uint32_t* __restrict__ part_pair,
    uint2* __restrict__ runs, uint32_t* __restrict__ item_first, int cap,
    uint32_t* __restrict__ err) {
    constexpr int PER = round_per(false);
    __shared__ PlaceShared<uint2, COLS, 3072, false> sh;
    __shared__ uint32_t s_pairs[kRbWaves];
    const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6, part = blockIdx.x;
    const int v = view_of_part(views, num_views, part);
    const ViewRec vr = views[v];
    const int local = (part - vr.part_off) * kRbPart;
    static_assert(PER == kRbPer, "a wave's items are consecutive");
    Interval iv[kRbPer];
    uint2 val[kRbPer];
    uint32_t before[kRbPer], pairs = 0;
    bool bad_any = false;
#pragma unroll
    for (int k = 0; k < kRbPer; ++k) {
        const int i = local + interval_index<PER>(k);
        const uint2 own = i < vr.n ? rects[vr.item_off + i] : make_uint2(0u, 0u);
        const uint32_t n = rect_count(own), incl = wave_inclusive_sum(n);
        before[k] = pairs + incl - n;
        pairs += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        bool bad;
        const uint2 rc = grid_rect(own, vr.tiles_x, vr.tiles_y, bad);
        bad_any = bad_any || bad;
        iv[k].lo = (int)(rc.x >> 16);
        iv[k].len = rect_count(rc) > 0 ? (int)(rc.y >> 16) : 0;
        val[k] = make_uint2((uint32_t)vr.item_off + (uint32_t)i, (rc.x & 0xFFFFu) | (rc.y << 16));
    }
    if (bad_any) atomicOr(err, 4u);
    if (lane == 0) s_pairs[wave] = pairs;
    clear_place(sh);
    __syncthreads();
    if (item_first) {
        uint32_t at = part_pair[part];
        for (int w = 0; w < wave; ++w) at += s_pairs[w];
#pragma unroll
        for (int k = 0; k < kRbPer; ++k) {
            const int i = local + interval_index<PER>(k);
            if (i < vr.n) item_first[vr.item_off + i] = min(at + before[k], (uint32_t)cap);
        }
    }
    const int base =
        tid < vr.tiles_y
            ? clamped_sum(row_off[vr.row_off], counts[(size_t)part * kRowBinAxis + tid], cap)
            : 0;
    place_all<PER>(sh, iv, val, vr.tiles_y, base, runs, cap);
}

// Step 2, counting, over the descriptors.
__global__ __launch_bounds__(kRbThreads) void batch_col_count_kernel(
    const uint2* __restrict__ runs, const int4* __restrict__ desc,
    uint32_t* __restrict__ counts) {
    __shared__ int s_d[kRbThreads];
    __shared__ uint32_t s_tmp[kRbWaves];
    const int tid = threadIdx.x;
    for_partitions(uniform_i(desc[-1].x), [&](int p) {
        const int4 d = desc[p];
        count_columns(runs, d.y, d.z, s_d, s_tmp, counts + (size_t)p * kRowBinAxis);
    });
}

// Step 2, offsets, one workgroup per row.
template <int COLS>
__global__ __launch_bounds__(kScanThreads) void batch_col_scan_kernel(
    const int* __restrict__ row_part, int cap, uint32_t* __restrict__ counts,
    uint32_t* __restrict__ tile_first) {
    __shared__ ScanShared sh;
    const int row = blockIdx.x, p0 = row_part[row];
    scan_columns<COLS>(sh, p0, row_part[row + 1] - p0, cap, counts,
                       tile_first + (size_t)row * (kRowBinAxis + 1));
}

// Every row's first pair.
__global__ __launch_bounds__(1024) void batch_pair_scan_kernel(
    int rows, const uint32_t* __restrict__ tile_first, int cap, int* __restrict__ row_pair) {
    __shared__ uint64_t s_tmp[17];
    scan_rounds(
        rows, s_tmp,
        [&](int r) {
            return (uint64_t)tile_first[(size_t)r * (kRowBinAxis + 1) + kRowBinAxis];
        },
        [&](int r, uint64_t e, uint64_t) { row_pair[r] = (int)min(e, (uint64_t)cap); });
}

// Step 2, placement (col_place_kernel).
template <int COLS>
__global__ __launch_bounds__(kRbThreads) void batch_col_place_kernel(
    const ViewRec* __restrict__ views, const int* __restrict__ row_view,
    const uint2* __restrict__ runs, const int4* __restrict__ desc, int cap, const uint32_t* __restrict__ counts,
    const uint32_t* __restrict__ tile_first, const int* __restrict__ row_pair,
    uint32_t* __restrict__ ids, int2* __restrict__ bins) {
    constexpr int PER = round_per(false);
    __shared__ PlaceShared<uint32_t, COLS, 5120, false> sh;
    const int tid = threadIdx.x;
    for_partitions(uniform_i(desc[-1].x), [&](int p) {
        const int4 d = desc[p];
        const int v = row_view[d.x], ty = d.x - views[v].row_off;
        const int tiles_x = views[v].tiles_x;
        Interval iv[kRbPer];
        uint32_t id[kRbPer];
#pragma unroll
        for (int k = 0; k < kRbPer; ++k) {
            const int i = interval_index<PER>(k);
            const uint2 run = i < d.z - d.y ? runs[d.y + i] : make_uint2(0u, 0u);
            id[k] = run.x;
            iv[k] = {(int)(run.y & 0xFFFFu), (int)(run.y >> 16)};
        }
        clear_place(sh);
        __syncthreads();
        const int row0 = row_pair[d.x];
        const int base =
            tid < tiles_x ? clamped_sum(row0, counts[(size_t)p * kRowBinAxis + tid], cap) : 0;
        if (d.w && tid < tiles_x) {
            const uint32_t* tf = tile_first + (size_t)d.x * (kRowBinAxis + 1) + tid;
            const int b = clamped_sum(row0, tf[0], cap), e = clamped_sum(row0, tf[1], cap);
            if (e > b) bins[views[v].bin_off + ty * tiles_x + tid] = make_int2(b, e);
        }
        place_all<PER>(sh, iv, id, tiles_x, base, ids, cap);
    });
}

// Tile id of every list entry (only where the caller asks for it).
__global__ void tile_ids_kernel(const int2* __restrict__ bins, uint32_t* __restrict__ tiles) {
    const int2 b = bins[blockIdx.x];
    for (int i = b.x + (int)threadIdx.x; i < b.y; i += blockDim.x) tiles[i] = blockIdx.x;
}

constexpr size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

}  // namespace

RowBinPlan row_bin_plan(int n, int tiles_x, int tiles_y, int cap) {
    RowBinPlan p{};
    p.n = n;
    p.tiles_x = tiles_x;
    p.tiles_y = tiles_y;
    p.cap = cap > 0 ? cap : 1;
    p.parts = (n + kRbPart - 1) / kRbPart;
    p.fold = p.parts <= kFoldParts;
    p.max_col_parts = p.cap / kRbPart + tiles_y;
    size_t o = 0;
    const size_t parts = (size_t)(p.parts > 0 ? p.parts : 1);
    p.cut = o; o = align256(o + sizeof(Cut));
    p.row_len = o; o = align256(o + 4ull * kRowBinAxis);
    p.row_counts = o; o = align256(o + 4ull * kRowBinAxis * parts);
    p.part_tot = o; o = align256(o + 4ull * parts);
    p.tile_first = o; o = align256(o + 4ull * (kRowBinAxis + 1) * (size_t)kRowBinAxis);
    p.desc = o; o = align256(o + 16ull * ((size_t)p.max_col_parts + 1));
    p.col_counts = o; o = align256(o + 4ull * kRowBinAxis * (size_t)p.max_col_parts);
    p.scratch_bytes = o;
    return p;
}

hipError_t row_bin(const RowBinPlan& p, const uint32_t* perm, const uint2* rects,
                   const int* cum, uint2* in_order, uint2* runs, uint32_t* ids, uint32_t* tiles_sorted,
                   int2* bins, unsigned long long* total, uint32_t* err, void* scratch,
                   hipStream_t s) {
    if (p.tiles_x > kRowBinAxis || p.tiles_y > kRowBinAxis || p.n <= 0)
        return hipErrorInvalidValue;
    uint8_t* b = static_cast<uint8_t*>(scratch);
    auto U = [&](size_t off) { return reinterpret_cast<uint32_t*>(b + off); };
    int4* desc = reinterpret_cast<int4*>(b + p.desc) + 1;
    Cut* cut = reinterpret_cast<Cut*>(b + p.cut);
    const int tiles = p.tiles_x * p.tiles_y;
    hipError_t e;
    row_count_kernel<<<p.parts, kRbThreads, 0, s>>>(
        p.n, perm, rects, cum, p.cap, p.tiles_x, p.tiles_y, p.fold ? 1 : p.parts,
        p.fold ? kRowBinAxis : 1, U(p.row_counts), U(p.part_tot), in_order, tiles, bins, cut, err);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (!p.fold && (e = column_scan(U(p.row_counts), p.parts, U(p.row_len), p.tiles_y, s)) !=
                       hipSuccess)
        return e;
#define JSA_ROW(ST, COLS)                                                                     \
    row_place_kernel<ST, COLS><<<p.parts, kRbThreads, 0, s>>>(                                \
        p.n, perm, perm ? in_order : rects, p.tiles_x, p.tiles_y, p.parts, p.fold,            \
        U(p.row_counts), U(p.row_len), U(p.part_tot), runs, p.cap, cut, total, err)
    if (narrow(p.tiles_y)) {
        if (perm) JSA_ROW(true, 128); else JSA_ROW(false, 128);
    } else {
        if (perm) JSA_ROW(true, 256); else JSA_ROW(false, 256);
    }
#undef JSA_ROW
    if ((e = hipGetLastError()) != hipSuccess) return e;
    stage_mark(kMarkEmitted, s);
    // persistent: as many workgroups as fit the chip, or one per partition
    const int most = 8 * ((p.max_col_parts + 7) / 8);
    const int grid = most < 2048 ? most : 2048;
    col_count_kernel<<<grid, kRbThreads, 0, s>>>(runs, U(p.row_len), p.tiles_y, p.cap,
                                                 U(p.col_counts), desc);
    if ((e = hipGetLastError()) != hipSuccess) return e;
#define JSA_LAUNCH(COLS)                                                                      \
    col_scan_kernel<COLS><<<p.tiles_y, kScanThreads, 0, s>>>(                                 \
        U(p.row_len), p.tiles_y, p.cap, U(p.col_counts), U(p.tile_first))
    JSA_SCAN(p.tiles_x, JSA_LAUNCH);
#undef JSA_LAUNCH
    if ((e = hipGetLastError()) != hipSuccess) return e;
#define JSA_COL(ST, COLS)                                                                     \
    col_place_kernel<ST, COLS><<<grid, kRbThreads, 0, s>>>(                                   \
        runs, desc, p.tiles_x, p.tiles_y, p.cap, U(p.col_counts), U(p.tile_first), ids, bins)
    if (narrow(p.tiles_x)) {
        if (perm) JSA_COL(true, 128); else JSA_COL(false, 128);
    } else {
        if (perm) JSA_COL(true, 256); else JSA_COL(false, 256);
    }
#undef JSA_COL
    if ((e = hipGetLastError()) != hipSuccess) return e;
    stage_mark(kMarkTileSorted, s);
    if (tiles_sorted) {
        tile_ids_kernel<<<tiles, 256, 0, s>>>(bins, tiles_sorted);
        e = hipGetLastError();
    }
    return e;
}

BatchRowPlan batch_row_plan(int num_views, int parts, int rows, int max_x, int max_y, int cap) {
    BatchRowPlan p{};
    p.num_views = num_views;
    p.parts = parts;
    p.max_x = max_x;
    p.max_y = max_y;
    p.rows = rows;
    p.cap = cap > 0 ? cap : 1;
    p.max_col_parts = p.cap / kRbPart + p.rows;
    const size_t np = (size_t)(parts > 0 ? parts : 1), nr = (size_t)(rows > 0 ? rows : 1);
    size_t o = 0;
    p.counts = o; o = align256(o + 4ull * kRowBinAxis * np);
    p.part_tot = o; o = align256(o + 4ull * np);
    p.part_pair = o; o = align256(o + 4ull * np);
    p.row_first = o; o = align256(o + 4ull * (kRowBinAxis + 1) * (size_t)num_views);
    p.row_view = o; o = align256(o + 4ull * nr);
    p.row_len = o; o = align256(o + 4ull * nr);
    p.row_off = o; o = align256(o + 4ull * nr);
    p.row_part = o; o = align256(o + 4ull * (nr + 1));
    p.row_pair = o; o = align256(o + 4ull * nr);
    p.tile_first = o; o = align256(o + 4ull * (kRowBinAxis + 1) * nr);
    p.desc = o; o = align256(o + 16ull * ((size_t)p.max_col_parts + 1));
    p.col_counts = o; o = align256(o + 4ull * kRowBinAxis * (size_t)p.max_col_parts);
    p.scratch_bytes = o;
    return p;
}

hipError_t batch_row_bin(const BatchRowPlan& p, const ViewRec* views, const uint2* rects,
                         uint2* runs, uint32_t* ids, int num_bins, int2* bins,
                         uint32_t* item_first, int* count, unsigned long long* total,
                         uint32_t* err, void* scratch, hipStream_t s) {
    uint8_t* b = static_cast<uint8_t*>(scratch);
    auto U = [&](size_t off) { return reinterpret_cast<uint32_t*>(b + off); };
    auto I = [&](size_t off) { return reinterpret_cast<int*>(b + off); };
    int4* desc = reinterpret_cast<int4*>(b + p.desc) + 1;
    hipError_t e;
    batch_row_count_kernel<<<p.parts, kRbThreads, 0, s>>>(
        views, p.num_views, rects, U(p.counts), U(p.part_tot), num_bins, bins, err);
    if ((e = hipGetLastError()) != hipSuccess) return e;
#define JSA_LAUNCH(COLS)                                                                      \
    batch_row_scan_kernel<COLS><<<p.num_views, kScanThreads, 0, s>>>(                         \
        views, p.cap, U(p.counts), U(p.row_first), U(p.row_len), I(p.row_view))
    JSA_SCAN(p.max_y, JSA_LAUNCH);
#undef JSA_LAUNCH
    if ((e = hipGetLastError()) != hipSuccess) return e;
    batch_table_kernel<<<2, 1024, 0, s>>>(p.rows, U(p.row_len), p.cap, I(p.row_off),
                                          I(p.row_part), desc, p.parts, U(p.part_tot),
                                          U(p.part_pair), count, total, err);
    if ((e = hipGetLastError()) != hipSuccess) return e;
#define JSA_ROW(COLS)                                                                         \
    batch_row_place_kernel<COLS><<<p.parts, kRbThreads, 0, s>>>(                              \
        views, p.num_views, rects, U(p.counts), I(p.row_off), U(p.part_pair), runs,           \
        item_first, p.cap, err)
    if (narrow(p.max_y)) JSA_ROW(128);
    else JSA_ROW(256);
#undef JSA_ROW
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const int most = 8 * ((p.max_col_parts + 7) / 8);
    const int grid = most < 2048 ? most : 2048;
    batch_col_count_kernel<<<grid, kRbThreads, 0, s>>>(runs, desc, U(p.col_counts));
    if ((e = hipGetLastError()) != hipSuccess) return e;
#define JSA_LAUNCH(COLS)                                                                      \
    batch_col_scan_kernel<COLS><<<p.rows, kScanThreads, 0, s>>>(                              \
        I(p.row_part), p.cap, U(p.col_counts), U(p.tile_first))
    JSA_SCAN(p.max_x, JSA_LAUNCH);
#undef JSA_LAUNCH
    if ((e = hipGetLastError()) != hipSuccess) return e;
    batch_pair_scan_kernel<<<1, 1024, 0, s>>>(p.rows, U(p.tile_first), p.cap, I(p.row_pair));
    if ((e = hipGetLastError()) != hipSuccess) return e;
#define JSA_COL(COLS)                                                                         \
    batch_col_place_kernel<COLS><<<grid, kRbThreads, 0, s>>>(                                 \
        views, I(p.row_view), runs, desc, p.cap, U(p.col_counts), U(p.tile_first),            \
        I(p.row_pair), ids, bins)
    if (narrow(p.max_x)) JSA_COL(128);
    else JSA_COL(256);
#undef JSA_COL
    return hipGetLastError();
}

}  // namespace jsa
