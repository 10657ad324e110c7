// Cut points from 32-bit keys grouped by feature (HistCut::get_cut_points_single, src/thundergbm/hist_cut.cu:232-286): the
// values of a feature become a segment of their own first - one radix step on the column index, or a transposition where
// every row stores every column - and four radix steps sort all segments side by side. Against sorting (feature, value)
// pairs of 64 bits that is half of the bytes per step and a step less; the distinct values are counted and
// numbered tile by tile instead of through an index per value. Streaming passes, bound by memory and by the ranking
// inside a tile: 280 M values of 28 features 13.4 -> 7.9 ms.
#include <algorithm>
#include <vector>

#include "device_api.h"

namespace tgbm {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kTile = 4096;  // values per tile; a tile belongs to one feature
constexpr int kRounds = kTile / kBlock;

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }
__device__ __forceinline__ int wave_id() { return threadIdx.x >> 6; }
__device__ __forceinline__ int lanes_below(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
}

// Order-preserving map float -> uint32 (-0.0 is folded into +0.0 so that == duplicates share a key).
__device__ __forceinline__ unsigned float_key(float v) {
    if (v == 0.f) v = 0.f;
    const unsigned u = __float_as_uint(v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_float(unsigned k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// The tiles of all segments, numbered segment by segment.
struct Segments {
    const unsigned *start;    // [F + 1] first value
    const unsigned *end;      // [F] behind the last one
    const int *tile_begin;    // [F + 1] first tile
    int F, n_tiles;
};
struct Tile {
    int feature, index, of;  // the index-th of `of` tiles of its feature
    unsigned base;
    int count;               // (0: behind the feature's last value, see k_transpose_cells)
};
__device__ __forceinline__ Tile find_tile(const Segments &sg, int tile) {
    int lo = 0, hi = sg.F;  // the last feature whose first tile is not behind (features without values have no tile)
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (sg.tile_begin[mid] <= tile) lo = mid; else hi = mid;
    }
    Tile t;
    t.feature = lo;
    t.index = tile - sg.tile_begin[lo];
    t.of = sg.tile_begin[lo + 1] - sg.tile_begin[lo];
    t.base = sg.start[lo] + (unsigned)t.index * kTile;
    t.count = (int)min((unsigned)kTile, max(sg.end[lo], t.base) - t.base);
    return t;
}

// ---- values into segments
// Every row stores every column: a transposition, 64 rows x 64 columns through LDS.
__global__ __launch_bounds__(kBlock) void k_transpose_keys(int n, int C, const float *__restrict__ x, unsigned *__restrict__ keys) {
    __shared__ unsigned s[64][65];
    const int r0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
    const int lane = lane_id(), w = wave_id();
#pragma unroll 4
    for (int r = w; r < 64; r += kWaves)
        if (r0 + r < n && c0 + lane < C) s[r][lane] = float_key(x[(size_t)(r0 + r) * C + c0 + lane]);
    __syncthreads();
#pragma unroll 4
    for (int c = w; c < 64; c += kWaves)
        if (r0 + lane < n && c0 + c < C) keys[(size_t)(c0 + c) * n + r0 + lane] = s[lane][c];
}

// The same for cells of which some hold no value (is_stored): their keys are the largest there are, which sorts them
// behind the values. stored[f] += values of the feature.
constexpr int kCellRows = 256;  // rows per workgroup
constexpr unsigned kNoValue = ~0u;
__global__ __launch_bounds__(kBlock) void k_transpose_cells(DenseCells cells, int F, unsigned *__restrict__ keys, unsigned *__restrict__ stored) {
    __shared__ unsigned s[64][65];
    __shared__ unsigned s_cnt[kWaves][64];
    const int c0 = blockIdx.y * 64, lane = lane_id(), w = wave_id();
    unsigned count = 0;
    for (int r0 = blockIdx.x * kCellRows; r0 < min(cells.n, ((int)blockIdx.x + 1) * kCellRows); r0 += 64) {
#pragma unroll 4
        for (int r = w; r < 64; r += kWaves)
            if (r0 + r < cells.n && c0 + lane < F) {
                const float v = cells.x[(size_t)(r0 + r) * cells.columns + c0 + lane];
                const bool in = is_stored(v, cells.minus_zero_is_stored);
                count += in ? 1u : 0u;
                s[r][lane] = in ? float_key(v) : kNoValue;
            }
        __syncthreads();
#pragma unroll 4
        for (int c = w; c < 64; c += kWaves)
            if (r0 + lane < cells.n && c0 + c < F) keys[(size_t)(c0 + c) * cells.n + r0 + lane] = s[lane][c];
        __syncthreads();
    }
    s_cnt[w][lane] = count;
    __syncthreads();
    if (w == 0 && c0 + lane < F) {
#pragma unroll
        for (int i = 1; i < kWaves; ++i) count += s_cnt[i][lane];
        atomicAdd(&stored[c0 + lane], count);
    }
}

// counts[feature * tiles + tile]: entries of the tile (a run of kTile CSR entries) in the feature's column.
__global__ __launch_bounds__(kBlock) void k_column_count(long nnz, int F, const int *__restrict__ col, int n_tiles,
                                                        unsigned *__restrict__ counts) {
    __shared__ unsigned s_cnt[256];
    s_cnt[threadIdx.x] = 0;
    __syncthreads();
    const long base = (long)blockIdx.x * kTile;
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
        const long i = base + k * kBlock + threadIdx.x;
        if (i < nnz) atomicAdd(&s_cnt[col[i]], 1u);
    }
    __syncthreads();
    if ((int)threadIdx.x < F) counts[(size_t)threadIdx.x * n_tiles + blockIdx.x] = s_cnt[threadIdx.x];
}

// The tile's keys go out column by column (ordered in LDS, so that runs of them leave together; inside a column the
// order does not matter).
__global__ __launch_bounds__(kBlock) void k_column_scatter(long nnz, int F, const int *__restrict__ col, const float *__restrict__ val,
                                                          int n_tiles, const unsigned *__restrict__ counts,
                                                          const unsigned *__restrict__ offsets, unsigned *__restrict__ keys) {
    __shared__ unsigned s_key[kTile];
    __shared__ uint8_t s_col[kTile];
    __shared__ unsigned s_next[256], s_delta[256], s_wsum[kWaves];
    const long base = (long)blockIdx.x * kTile;
    const int lane = lane_id(), w = wave_id();
    {
        const int f = threadIdx.x;
        const size_t at = (size_t)f * n_tiles + blockIdx.x;
        const unsigned c = f < F ? counts[at] : 0u, to = f < F ? offsets[at] : 0u;
        unsigned inc = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const unsigned t = __shfl_up(inc, d);
            if (lane >= d) inc += t;
        }
        if (lane == 63) s_wsum[w] = inc;
        __syncthreads();
        unsigned before = inc - c;
        for (int i = 0; i < w; ++i) before += s_wsum[i];
        s_next[f] = before;
        s_delta[f] = to - before;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
        const long i = base + k * kBlock + threadIdx.x;
        if (i < nnz) {
            const int f = col[i];
            const unsigned p = atomicAdd(&s_next[f], 1u);
            s_key[p] = float_key(val[i]);
            s_col[p] = (uint8_t)f;
        }
    }
    __syncthreads();
    const int count = (int)min((long)kTile, nnz - base);
    for (int p = threadIdx.x; p < count; p += kBlock) keys[s_delta[s_col[p]] + (unsigned)p] = s_key[p];
}

// out[f] = in[first entry of feature f], out[F] = *total; first entry: f * stride, or tile_begin[f] (the total behind the end)
__global__ void k_pick_starts(int F, const unsigned *__restrict__ in, int stride, const int *__restrict__ tile_begin, int n_tiles,
                              const unsigned *__restrict__ total, unsigned *__restrict__ out) {
    for (int f = blockIdx.x * blockDim.x + threadIdx.x; f <= F; f += gridDim.x * blockDim.x) {
        if (f == F) out[f] = *total;
        else if (tile_begin == nullptr) out[f] = in[(size_t)f * stride];
        else out[f] = tile_begin[f] < n_tiles ? in[tile_begin[f]] : *total;
    }
}

// ---- radix steps of 8 bits inside the segments
// counts of tile t of a feature: [256 * first tile + digit * tiles + t], so that one scan over all gives the positions
__global__ __launch_bounds__(kBlock) void k_segment_count(Segments sg, const unsigned *__restrict__ keys, int shift,
                                                         unsigned *__restrict__ counts) {
    __shared__ unsigned s_cnt[kWaves][256];
    const int w = wave_id();
#pragma unroll
    for (int i = 0; i < kWaves; ++i) s_cnt[i][threadIdx.x] = 0;
    const Tile t = find_tile(sg, blockIdx.x);
    unsigned k[kRounds];
#pragma unroll
    for (int b = 0; b < kRounds; ++b) k[b] = keys[t.base + min(b * kBlock + (int)threadIdx.x, t.count - 1)];
    __syncthreads();
#pragma unroll
    for (int b = 0; b < kRounds; ++b)
        if (b * kBlock + (int)threadIdx.x < t.count) atomicAdd(&s_cnt[w][(k[b] >> shift) & 255u], 1u);
    __syncthreads();
    unsigned sum = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) sum += s_cnt[i][threadIdx.x];
    counts[(size_t)256 * (blockIdx.x - t.index) + (size_t)threadIdx.x * t.of + t.index] = sum;
}

// (the ranking of k_radix_scatter: every wavefront ranks its quarter of the tile round by round, in order)
__global__ __launch_bounds__(kBlock) void k_segment_scatter(Segments sg, const unsigned *__restrict__ in, unsigned *__restrict__ out,
                                                           int shift, const unsigned *__restrict__ offsets) {
    __shared__ unsigned s_key[kTile];
    __shared__ unsigned s_run[kWaves][256];  // per wavefront and digit: count, then the next local position
    __shared__ unsigned s_delta[256];        // per digit: global position of its first key - local position of it
    __shared__ unsigned s_wsum[kWaves];
    const int w = wave_id(), lane = lane_id();
    const Tile t = find_tile(sg, blockIdx.x);
    for (int d = lane; d < 256; d += 64) s_run[w][d] = 0;
    unsigned keys[kRounds];
#pragma unroll
    for (int b = 0; b < kRounds; ++b) keys[b] = in[t.base + min(w * (kTile / kWaves) + b * 64 + lane, t.count - 1)];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int b = 0; b < kRounds; ++b)
        if (w * (kTile / kWaves) + b * 64 + lane < t.count) atomicAdd(&s_run[w][(keys[b] >> shift) & 255u], 1u);
    __syncthreads();
    {
        const int d = threadIdx.x;
        unsigned c[kWaves], tot = 0;
#pragma unroll
        for (int i = 0; i < kWaves; ++i) {
            c[i] = s_run[i][d];
            tot += c[i];
        }
        unsigned inc = tot;
#pragma unroll
        for (int k = 1; k < 64; k <<= 1) {
            const unsigned u = __shfl_up(inc, k);
            if (lane >= k) inc += u;
        }
        if (lane == 63) s_wsum[w] = inc;
        __syncthreads();
        unsigned run = inc - tot;
        for (int i = 0; i < w; ++i) run += s_wsum[i];
        s_delta[d] = offsets[(size_t)256 * (blockIdx.x - t.index) + (size_t)d * t.of + t.index] - run;
#pragma unroll
        for (int i = 0; i < kWaves; ++i) {
            s_run[i][d] = run;
            run += c[i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < kRounds; ++b) {
        const bool valid = w * (kTile / kWaves) + b * 64 + lane < t.count;
        const unsigned d = (keys[b] >> shift) & 255u;
        unsigned long long mask = __ballot(valid);  // lanes holding the same digit (match-any built from eight ballots)
#pragma unroll
        for (int bit_i = 0; bit_i < 8; ++bit_i) {
            const bool bit = (d >> bit_i) & 1u;
            const unsigned long long m = __ballot(bit);
            mask &= bit ? m : ~m;
        }
        const unsigned first = valid ? s_run[w][d] : 0u;
        const int rank = lanes_below(mask);
        __builtin_amdgcn_wave_barrier();
        if (valid) {
            s_key[first + rank] = keys[b];
            if (rank == 0) s_run[w][d] = first + (unsigned)__popcll(mask);
        }
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    for (int i = threadIdx.x; i < t.count; i += kBlock) {
        const unsigned key = s_key[i];
        out[s_delta[(key >> shift) & 255u] + (unsigned)i] = key;
    }
}

// ---- short segments
// A feature of up to kShortSegment values is sorted by one workgroup, which keeps the keys in registers and orders them through LDS
// (four steps like k_segment_scatter's), and leaves the distinct ones in order in the segment. One launch for the 30 of the steps
// tile by tile, each of which takes 2 to 10 us and a gap whatever the number of keys. The LDS that 16 384 keys take leaves two
// workgroups a CU. Bound by the chain of the steps: 8 features of 10 000 values 38 us, 119 of up to 1605 15 us, where the launches
// took 95 and their gaps as much again (a call with 40 trees 4.79 -> 4.70 and 4.14 -> 4.02 ms).
constexpr int kSortBlock = 1024, kSortWaves = kSortBlock / 64;
constexpr int kShortSegment = 16 * kSortBlock;
template <int ROUNDS>
__global__ __launch_bounds__(kSortBlock) void k_sort_feature(const unsigned *__restrict__ start, const unsigned *__restrict__ stored,
                                                             const unsigned *__restrict__ in, unsigned *__restrict__ out,
                                                             unsigned *__restrict__ distinct) {
    extern __shared__ unsigned s_key[];  // [ROUNDS * kSortBlock]
    __shared__ unsigned s_run[kSortWaves][256];  // per wavefront and digit: count, then the next position
    __shared__ unsigned s_wsum[kSortWaves];
    const int w = wave_id(), lane = lane_id();
    const unsigned base = start[blockIdx.x];
    const int len = (int)(start[blockIdx.x + 1] - base);
    const int values = stored != nullptr ? (int)stored[blockIdx.x] : len;  // (the rest are empty cells, whose keys are the largest)
    const int rounds = (len + kSortBlock - 1) / kSortBlock;  // (at most ROUNDS) of 64 keys for every wavefront
    const int i0 = w * (rounds * 64) + lane;
    unsigned key[ROUNDS];
#pragma unroll
    for (int b = 0; b < ROUNDS; ++b) key[b] = b < rounds && i0 + b * 64 < len ? in[base + (unsigned)(i0 + b * 64)] : ~0u;  // (behind all others: they come last)
    for (int shift = 0; shift < 32; shift += 8) {
        for (int d = lane; d < 256; d += 64) s_run[w][d] = 0;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int b = 0; b < ROUNDS; ++b)
            if (b < rounds) atomicAdd(&s_run[w][key[b] >> shift & 255u], 1u);
        __syncthreads();
        unsigned c[kSortWaves], tot = 0, inc = 0;
        if (threadIdx.x < 256) {
#pragma unroll
            for (int i = 0; i < kSortWaves; ++i) {
                c[i] = s_run[i][threadIdx.x];
                tot += c[i];
            }
            inc = tot;
#pragma unroll
            for (int k = 1; k < 64; k <<= 1) {
                const unsigned u = __shfl_up(inc, k);
                if (lane >= k) inc += u;
            }
            if (lane == 63) s_wsum[w] = inc;
        }
        __syncthreads();
        if (threadIdx.x < 256) {
            unsigned run = inc - tot;
            for (int i = 0; i < w; ++i) run += s_wsum[i];
#pragma unroll
            for (int i = 0; i < kSortWaves; ++i) {
                s_run[i][threadIdx.x] = run;
                run += c[i];
            }
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < ROUNDS; ++b) {
            if (b >= rounds) continue;
            const unsigned d = key[b] >> shift & 255u;
            unsigned long long mask = ~0ull;  // lanes holding the same digit
#pragma unroll
            for (int bit_i = 0; bit_i < 8; ++bit_i) {
                const bool bit = (d >> bit_i) & 1u;
                const unsigned long long m = __ballot(bit);
                mask &= bit ? m : ~m;
            }
            const unsigned first = s_run[w][d];
            const int rank = lanes_below(mask);
            __builtin_amdgcn_wave_barrier();
            s_key[first + rank] = key[b];
            if (rank == 0) s_run[w][d] = first + (unsigned)__popcll(mask);
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < ROUNDS; ++b)
            if (b < rounds) key[b] = s_key[i0 + b * 64];
        // (the next step's keys go to s_key behind three barriers)
    }
    unsigned long long first[ROUNDS];  // bit l: the key of lane l is the first of its value
    unsigned total = 0;
#pragma unroll
    for (int b = 0; b < ROUNDS; ++b) {
        const int i = i0 + b * 64;
        first[b] = __ballot(b < rounds && i < values && (i == 0 || s_key[max(i - 1, 0)] != key[b]));
        total += (unsigned)__popcll(first[b]);
    }
    if (lane == 0) s_wsum[w] = total;
    __syncthreads();
    unsigned rank = 0;
    for (int i = 0; i < w; ++i) rank += s_wsum[i];
    if (w == kSortWaves - 1 && lane == 0) distinct[blockIdx.x] = rank + total;
#pragma unroll
    for (int b = 0; b < ROUNDS; ++b) {
        if (first[b] >> lane & 1ull) out[base + rank + (unsigned)lanes_below(first[b])] = key[b];
        rank += (unsigned)__popcll(first[b]);
    }
}

// The strided selection (k_distinct_emit) from a feature's distinct keys.
__global__ __launch_bounds__(kBlock) void k_pick_cuts(const unsigned *__restrict__ start, const unsigned *__restrict__ distinct,
                                                     const unsigned *__restrict__ keys, const int *__restrict__ cut_row_ptr, int max_bin,
                                                     float *__restrict__ cut_val, int *__restrict__ cut_fid) {
    const int f = blockIdx.x, cb = cut_row_ptr[f], count = cut_row_ptr[f + 1] - cb;
    const unsigned step = max(distinct[f] / (unsigned)max_bin, 1u);
    for (int i = threadIdx.x; i < count; i += kBlock) {
        cut_val[cb + i] = key_float(keys[start[f] + (unsigned)i * step]);
        cut_fid[cb + i] = f;
    }
}

// ---- distinct values of the sorted segments
// A wavefront owns a quarter of the tile, 64 neighbouring keys a round (16 neighbours per thread instead: 539 us for the 280 M
// keys of 28 features). Bit l of first[b]: the key of lane l in round b is the first of its value.
__device__ __forceinline__ unsigned first_of_value(const Tile &t, const unsigned *__restrict__ keys, unsigned (&k)[kRounds],
                                                   unsigned long long (&first)[kRounds]) {
    const int i0 = wave_id() * (kTile / kWaves), lane = lane_id();
#pragma unroll
    for (int b = 0; b < kRounds; ++b) k[b] = keys[t.base + min(i0 + b * 64 + lane, t.count - 1)];
    // the key in front of the quarter (lane 0's matters); a quarter behind the tile's end has no keys and reads nothing there
    unsigned last = ~k[0];
    if (i0 < t.count && (i0 > 0 || t.index > 0)) last = keys[t.base + (unsigned)i0 - 1u];
    unsigned total = 0;
#pragma unroll
    for (int b = 0; b < kRounds; ++b) {
        const unsigned up = __shfl_up(k[b], 1);
        first[b] = __ballot(i0 + b * 64 + lane < t.count && k[b] != (lane == 0 ? last : up));
        total += __popcll(first[b]);
        last = __shfl(k[b], 63);
    }
    return total;
}

__global__ __launch_bounds__(kBlock) void k_distinct_count(Segments sg, const unsigned *__restrict__ keys, unsigned *__restrict__ counts) {
    __shared__ unsigned s[kWaves];
    const Tile t = find_tile(sg, blockIdx.x);
    if (t.count == 0) {
        if (threadIdx.x == 0) counts[blockIdx.x] = 0u;
        return;
    }
    unsigned k[kRounds];
    unsigned long long first[kRounds];
    const unsigned c = first_of_value(t, keys, k, first);
    if (lane_id() == 0) s[wave_id()] = c;
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = s[0] + s[1] + s[2] + s[3];
}

// Strided selection (hist_cut.cu:259-265): with m distinct values and step = m / max_bin, all of them if step == 0, else the
// values at ranks 0, step, 2 step, ... (max_bin of them). before: distinct values before the tile; ustart: before the feature
__global__ __launch_bounds__(kBlock) void k_distinct_emit(Segments sg, const unsigned *__restrict__ keys, const unsigned *__restrict__ before,
                                                         const unsigned *__restrict__ ustart, const int *__restrict__ cut_row_ptr,
                                                         int max_bin, float *__restrict__ cut_val, int *__restrict__ cut_fid) {
    __shared__ unsigned s[kWaves];
    const Tile t = find_tile(sg, blockIdx.x);
    if (t.count == 0) return;
    unsigned k[kRounds];
    unsigned long long first[kRounds];
    const unsigned c = first_of_value(t, keys, k, first);
    if (lane_id() == 0) s[wave_id()] = c;
    __syncthreads();
    unsigned rank = before[blockIdx.x] - ustart[t.feature];
    for (int i = 0; i < wave_id(); ++i) rank += s[i];
    const unsigned step = max((ustart[t.feature + 1] - ustart[t.feature]) / (unsigned)max_bin, 1u);
    const bool all = (ustart[t.feature + 1] - ustart[t.feature]) < (unsigned)max_bin;
    const int cb = cut_row_ptr[t.feature];
#pragma unroll
    for (int b = 0; b < kRounds; ++b) {
        if (first[b] >> lane_id() & 1ull) {
            const unsigned r = rank + (unsigned)lanes_below(first[b]), number = r / step;
            if (number * step == r && (all || number < (unsigned)max_bin)) {
                cut_val[cb + (int)number] = key_float(k[b]);
                cut_fid[cb + (int)number] = t.feature;
            }
        }
        rank += (unsigned)__popcll(first[b]);
    }
}

template <int ROUNDS>
void sort_features_launch(hipStream_t s, int F, const unsigned *start, const unsigned *stored, const unsigned *in, unsigned *out, unsigned *distinct) {
    const size_t lds = sizeof(unsigned) * ROUNDS * kSortBlock;
    static LdsOptIn opt_in;
    if (lds > 32 * 1024) opt_in({reinterpret_cast<const void *>(&k_sort_feature<ROUNDS>)});
    k_sort_feature<ROUNDS><<<(unsigned)F, kSortBlock, lds, s>>>(start, stored, in, out, distinct);
}

void sort_features(hipStream_t s, int F, int longest, const unsigned *start, const unsigned *stored, const unsigned *in, unsigned *out,
                   unsigned *distinct) {
    if (longest <= 2 * kSortBlock) sort_features_launch<2>(s, F, start, stored, in, out, distinct);
    else if (longest <= 4 * kSortBlock) sort_features_launch<4>(s, F, start, stored, in, out, distinct);
    else if (longest <= 8 * kSortBlock) sort_features_launch<8>(s, F, start, stored, in, out, distinct);
    else sort_features_launch<16>(s, F, start, stored, in, out, distinct);
}

}  // namespace

DeviceCuts build_cut_points_by_feature(hipStream_t s, int F, long nnz, const float *d_val, const int *d_col, bool full_rows,
                                       int max_num_bin, const DenseCells *cells) {
    DeviceCuts out;
    const unsigned feature_grid = (unsigned)((F + kBlock) / kBlock);
    ScanScratch scratch;
    unsigned *keys[2] = {nullptr, nullptr}, *d_start = nullptr, *d_total = nullptr;
    const size_t n_keys = cells != nullptr ? (size_t)cells->n * F : (size_t)nnz;
    for (unsigned *&k : keys) device_alloc_to(k, sizeof(unsigned) * n_keys);
    device_alloc_to(d_start, sizeof(unsigned) * ((size_t)F + 1));
    device_alloc_to(d_total, sizeof(unsigned));
    std::vector<unsigned> start((size_t)F + 1);
    unsigned *d_stored = nullptr;  // behind the features' last values
    std::vector<unsigned> stored;
    if (cells != nullptr) {
        device_alloc_to(d_stored, sizeof(unsigned) * (size_t)F);
        HIP_CHECK(hipMemsetAsync(d_stored, 0, sizeof(unsigned) * (size_t)F, s));
        for (int f = 0; f <= F; ++f) start[(size_t)f] = (unsigned)((long)f * cells->n);
        k_transpose_cells<<<dim3((unsigned)((cells->n + kCellRows - 1) / kCellRows), (unsigned)((F + 63) / 64)), kBlock, 0, s>>>(*cells, F, keys[0],
                                                                                                                       d_stored);
        HIP_CHECK(hipMemcpyAsync(d_start, start.data(), sizeof(unsigned) * start.size(), hipMemcpyHostToDevice, s));
        stored.resize((size_t)F);
        HIP_CHECK(hipMemcpyAsync(stored.data(), d_stored, sizeof(unsigned) * stored.size(), hipMemcpyDeviceToHost, s));
        HIP_CHECK(hipStreamSynchronize(s));
    } else if (full_rows) {
        const long n = nnz / F;
        for (int f = 0; f <= F; ++f) start[(size_t)f] = (unsigned)(f * n);
        k_transpose_keys<<<dim3((unsigned)((n + 63) / 64), (unsigned)((F + 63) / 64)), kBlock, 0, s>>>((int)n, F, d_val, keys[0]);
        HIP_CHECK(hipMemcpyAsync(d_start, start.data(), sizeof(unsigned) * start.size(), hipMemcpyHostToDevice, s));
    } else {
        const int tiles = (int)((nnz + kTile - 1) / kTile);
        unsigned *counts = nullptr, *offsets = nullptr;
        device_alloc_to(counts, sizeof(unsigned) * (size_t)F * tiles);
        device_alloc_to(offsets, sizeof(unsigned) * (size_t)F * tiles);
        k_column_count<<<(unsigned)tiles, kBlock, 0, s>>>(nnz, F, d_col, tiles, counts);
        device_exclusive_scan(s, counts, offsets, (long)F * tiles, d_total, scratch);
        k_column_scatter<<<(unsigned)tiles, kBlock, 0, s>>>(nnz, F, d_col, d_val, tiles, counts, offsets, keys[0]);
        k_pick_starts<<<feature_grid, kBlock, 0, s>>>(F, offsets, tiles, nullptr, 0, d_total, d_start);
        HIP_CHECK(hipMemcpyAsync(start.data(), d_start, sizeof(unsigned) * start.size(), hipMemcpyDeviceToHost, s));
        HIP_CHECK(hipStreamSynchronize(s));
        device_free(counts);
        device_free(offsets);
    }
    out.feature_nnz.resize((size_t)F);
    long longest = 0;
    for (int f = 0; f < F; ++f) {
        const long keys_of = (long)(start[(size_t)f + 1] - start[(size_t)f]);
        out.feature_nnz[(size_t)f] = cells != nullptr ? (long)stored[(size_t)f] : keys_of;
        longest = std::max(longest, keys_of);
    }
    std::vector<int> crp((size_t)F + 1, 0);
    // the cut points' places, once the number of distinct values of every feature is known
    auto place = [&](const std::vector<unsigned> &distinct) {
        for (int f = 0; f < F; ++f) {
            const unsigned m = distinct[(size_t)f];
            crp[(size_t)f + 1] = crp[(size_t)f] + (m / (unsigned)max_num_bin == 0 ? (int)m : max_num_bin);
        }
        out.n_bins = crp[(size_t)F];
        device_alloc_to(out.cut_row_ptr, sizeof(int) * crp.size());
        device_alloc_to(out.cut_val, sizeof(float) * (size_t)std::max(out.n_bins, 1));
        device_alloc_to(out.cut_fid, sizeof(int) * (size_t)std::max(out.n_bins, 1));
        HIP_CHECK(hipMemcpyAsync(out.cut_row_ptr, crp.data(), sizeof(int) * crp.size(), hipMemcpyHostToDevice, s));
    };
    std::vector<unsigned> distinct((size_t)F);
    if (longest <= kShortSegment) {
        unsigned *d_distinct = nullptr;
        device_alloc_to(d_distinct, sizeof(unsigned) * (size_t)F);
        sort_features(s, F, (int)longest, d_start, d_stored, keys[0], keys[1], d_distinct);
        HIP_CHECK(hipMemcpyAsync(distinct.data(), d_distinct, sizeof(unsigned) * distinct.size(), hipMemcpyDeviceToHost, s));
        HIP_CHECK(hipStreamSynchronize(s));
        place(distinct);
        k_pick_cuts<<<(unsigned)F, kBlock, 0, s>>>(d_start, d_distinct, keys[1], out.cut_row_ptr, max_num_bin, out.cut_val, out.cut_fid);
        HIP_CHECK(hipStreamSynchronize(s));
        device_free(d_distinct);
    } else {
        std::vector<int> tile_begin((size_t)F + 1, 0);
        for (int f = 0; f < F; ++f)
            tile_begin[(size_t)f + 1] = tile_begin[(size_t)f] + (int)((start[(size_t)f + 1] - start[(size_t)f] + kTile - 1) / kTile);
        const int n_tiles = tile_begin[(size_t)F];
        int *d_tile_begin = nullptr;
        unsigned *counts = nullptr, *offsets = nullptr;
        device_alloc_to(d_tile_begin, sizeof(int) * tile_begin.size());
        device_alloc_to(counts, sizeof(unsigned) * 256 * (size_t)n_tiles);
        device_alloc_to(offsets, sizeof(unsigned) * 256 * (size_t)n_tiles);
        HIP_CHECK(hipMemcpyAsync(d_tile_begin, tile_begin.data(), sizeof(int) * tile_begin.size(), hipMemcpyHostToDevice, s));
        Segments sg{d_start, d_start + 1, d_tile_begin, F, n_tiles};
        int cur = 0;
        for (int shift = 0; shift < 32; shift += 8, cur ^= 1) {
            k_segment_count<<<(unsigned)n_tiles, kBlock, 0, s>>>(sg, keys[cur], shift, counts);
            device_exclusive_scan(s, counts, offsets, 256l * n_tiles, d_total, scratch);
            k_segment_scatter<<<(unsigned)n_tiles, kBlock, 0, s>>>(sg, keys[cur], keys[cur ^ 1], shift, offsets);
        }
        if (cells != nullptr) {  // (the empty cells lie behind the values now)
            for (int f = 0; f < F; ++f) stored[(size_t)f] += start[(size_t)f];
            HIP_CHECK(hipMemcpyAsync(d_stored, stored.data(), sizeof(unsigned) * stored.size(), hipMemcpyHostToDevice, s));
            sg.end = d_stored;
        }
        k_distinct_count<<<(unsigned)n_tiles, kBlock, 0, s>>>(sg, keys[cur], counts);
        device_exclusive_scan(s, counts, offsets, n_tiles, d_total, scratch);
        unsigned *d_ustart = keys[cur ^ 1];  // (free by now, and at least one value long)
        if ((size_t)F + 1 > n_keys) device_alloc_to(d_ustart, sizeof(unsigned) * ((size_t)F + 1));
        k_pick_starts<<<feature_grid, kBlock, 0, s>>>(F, offsets, 0, d_tile_begin, n_tiles, d_total, d_ustart);
        std::vector<unsigned> ustart((size_t)F + 1);
        HIP_CHECK(hipMemcpyAsync(ustart.data(), d_ustart, sizeof(unsigned) * ustart.size(), hipMemcpyDeviceToHost, s));
        HIP_CHECK(hipStreamSynchronize(s));
        for (int f = 0; f < F; ++f) distinct[(size_t)f] = ustart[(size_t)f + 1] - ustart[(size_t)f];
        place(distinct);
        k_distinct_emit<<<(unsigned)n_tiles, kBlock, 0, s>>>(sg, keys[cur], offsets, d_ustart, out.cut_row_ptr, max_num_bin, out.cut_val,
                                                           out.cut_fid);
        HIP_CHECK(hipStreamSynchronize(s));
        if (d_ustart != keys[cur ^ 1]) device_free(d_ustart);
        device_free(d_tile_begin);
        device_free(counts);
        device_free(offsets);
    }
    HIP_CHECK_LAUNCHES("cut points");
    scratch.release();
    for (unsigned *k : keys) device_free(k);
    device_free(d_start);
    if (d_stored != nullptr) device_free(d_stored);
    device_free(d_total);
    return out;
}

}  // namespace tgbm
