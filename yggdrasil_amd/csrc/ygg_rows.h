// The rows (stream, token) of a layer grouped by the expert they take, for the forms that run a layer over all rows of a
// call at once (ygg_float_scan.hip, ygg_scan.hip): a counting sort and its tiles.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace ygg::rows {

constexpr int kTile = 32;            // rows of a tile of one expert (two 16-row matrix tiles)
constexpr int kHistRows = 2048;      // least rows of one counting workgroup
constexpr int kHistGroups = 128;     // most counting workgroups
constexpr int kSortLeaves = 16384;   // most experts of a layer the sort's LDS histogram holds

inline size_t up256(size_t v) { return (v + 255) / 256 * 256; }

// The rows of one layer: N of them, leaf[i] the expert of row i or -1 for a row past its stream's end. Sorted, order
// holds the rows by expert and tiles the runs of at most kTile of one expert (expert, first place in order, rows).
struct Sort {
    int N, E, sorted, max_tiles;
    int groups, per;  // counting workgroups, rows of each
    int *leaf;
    int *rank;        // place of a row among its leaf's of its workgroup
    int *order;
    int4 *tiles;
    int *ntiles;
    int *hist;        // [groups][E] rows per leaf of each workgroup, then of the ones before it
    int *count;       // [E] rows per leaf
    int2 *off;        // [E] a leaf's first place in order and its first tile
    int *done;        // finished workgroups of rows_plan, zero before the sort
};

inline int hist_groups(int64_t N) {
    const int64_t g = (N + kHistRows - 1) / kHistRows;
    return (int)(g < kHistGroups ? g : kHistGroups);
}
// workspace bytes of a sort of at most N rows, where they are sorted: fixed (with the arrays' rounding up) and per row
inline int64_t sort_fixed_bytes(int64_t N, int E, bool sorted) {
    return 256 * 9 + (sorted ? (int64_t)E * (12 + 16 + 4 * hist_groups(N)) : 0);
}
constexpr int64_t kSortRowBytes = 12 + 1;

// The most rows, at most N, whose workspace fits: need(rows) bytes, more for more rows (a sort's arrays among them from
// where its rows are sorted on), in `bytes`; 0 if none.
template <class Need> inline int64_t rows_that_fit(int64_t N, int64_t bytes, Need need) {
    int64_t lo = 0, hi = N;
    while (lo < hi) {
        const int64_t mid = hi - (hi - lo) / 2;
        if (need(mid) <= bytes) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

template <class Take> inline void lay_out(Sort &s, int N, int E, bool sorted, Take take) {
    s.N = N;
    s.E = E;
    s.sorted = sorted;
    s.max_tiles = sorted ? N / kTile + E : 0;
    s.leaf = (int *)take((size_t)N * 4);
    if (!sorted) return;
    s.groups = hist_groups(N);
    s.per = ((N + s.groups - 1) / s.groups + 1023) / 1024 * 1024;
    s.groups = (N + s.per - 1) / s.per;
    s.done = (int *)take(4);
    s.ntiles = (int *)take(4);
    s.count = (int *)take((size_t)E * 4);
    s.off = (int2 *)take((size_t)E * 8);
    s.hist = (int *)take((size_t)E * s.groups * 4);
    s.tiles = (int4 *)take((size_t)s.max_tiles * 16);
    s.rank = (int *)take((size_t)N * 4);
    s.order = (int *)take((size_t)N * 4);
}

// a tile's leaf, first place and rows, or no rows; unsorted rows are tiles of one (i the same in the whole wavefront)
__device__ __forceinline__ int4 tile_at(const Sort &s, int i) {
    int4 t;
    if (s.sorted) {
        t = s.tiles[i];
    } else {
        const int r = s.leaf[i];
        t = make_int4(r, i, r >= 0 ? 1 : 0, 0);
    }
    return make_int4(__builtin_amdgcn_readfirstlane(t.x), __builtin_amdgcn_readfirstlane(t.y),
                     __builtin_amdgcn_readfirstlane(t.z), 0);
}
__device__ __forceinline__ int tiles_of(const Sort &s) { return s.sorted ? *s.ntiles : s.N; }
__device__ __forceinline__ int row_at(const Sort &s, int place) { return s.sorted ? s.order[place] : place; }

// (by one workgroup before the sort)
__device__ __forceinline__ void sort_clear(const Sort &s) {
    if (s.sorted && threadIdx.x == 0) *s.done = 0;
}

// The counting sort of sort a (blockIdx.y = 0) or b. First each workgroup counts its rows' leaves in LDS, whose additions
// also give a row its place among its leaf's there (counting by device-wide additions instead took 370 us for 840k rows
// and 16384 leaves; the three kernels take 45). EB: the histogram's size.
template <int EB> __global__ __launch_bounds__(1024) void rows_count(const Sort a, const Sort b) {
    __shared__ int hist[EB];
    const Sort &s = blockIdx.y ? b : a;
    const int tid = threadIdx.x, E = s.E, first = blockIdx.x * s.per, end = first + s.per < s.N ? first + s.per : s.N;
    for (int e = tid; e < E; e += 1024) hist[e] = 0;
    __syncthreads();
    for (int row = first + tid; row < end; row += 1024) {
        const int r = s.leaf[row];
        if (r >= 0) s.rank[row] = atomicAdd(&hist[r], 1);
    }
    __syncthreads();
    for (int e = tid; e < E; e += 1024) s.hist[(size_t)blockIdx.x * E + e] = hist[e];
}

// Then per leaf (a thread) the rows of the workgroups before each; the last workgroup to finish sums the leaves' rows into
// their first places and tiles.
template <int EB> __global__ __launch_bounds__(1024) void rows_plan(const Sort a, const Sort b) {
    __shared__ int cnt[EB];
    __shared__ int wsum[16][2], last;
    const Sort &s = blockIdx.y ? b : a;
    const int tid = threadIdx.x, E = s.E, mine = blockIdx.x * 1024 + tid;
    if (mine < E) {
        int sum = 0;
        for (int g = 0; g < s.groups; g += 8) {
            int v[8];
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = g + k < s.groups ? s.hist[(size_t)(g + k) * E + mine] : 0;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                if (g + k < s.groups) s.hist[(size_t)(g + k) * E + mine] = sum;
                sum += v[k];
            }
        }
        __hip_atomic_store(&s.count[mine], sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __threadfence();
    __syncthreads();
    if (tid == 0) {
        const int before = __hip_atomic_fetch_add(s.done, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        last = before == (int)gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    for (int e = tid; e < E; e += 1024)
        cnt[e] = __hip_atomic_load(&s.count[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    // exclusive sums of the counts and of the tiles, each thread a run of leaves
    const int per = (E + 1023) / 1024, e0 = tid * per;
    int rows = 0, tl = 0;
    for (int e = e0; e < e0 + per && e < E; e++) {
        rows += cnt[e];
        tl += (cnt[e] + kTile - 1) / kTile;
    }
    const int lane = tid & 63, wave = tid >> 6;
    int ir = rows, it = tl;
    for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(ir, o), y = __shfl_up(it, o);
        if (lane >= o) ir += x, it += y;
    }
    if (lane == 63) wsum[wave][0] = ir, wsum[wave][1] = it;
    __syncthreads();
    int pr = ir - rows, pt = it - tl, total = 0;
    for (int w = 0; w < 16; w++) {
        if (w < wave) pr += wsum[w][0], pt += wsum[w][1];
        total += wsum[w][1];
    }
    for (int e = e0; e < e0 + per && e < E; e++) {
        s.off[e] = make_int2(pr, pt);
        pr += cnt[e];
        pt += (cnt[e] + kTile - 1) / kTile;
    }
    if (tid == 0) *s.ntiles = total;
}

// At last every row goes to its place, and the first row of each tile writes the tile (a leaf that most rows take has
// thousands).
static __global__ __launch_bounds__(256) void rows_scatter(const Sort a, const Sort b) {
    const Sort &s = blockIdx.y ? b : a;
    const int row = blockIdx.x * 256 + threadIdx.x;
    if (row >= s.N) return;
    const int r = s.leaf[row];
    if (r < 0) return;
    const int2 off = s.off[r];
    const int at = s.hist[(size_t)(row / s.per) * s.E + r] + s.rank[row];
    s.order[off.x + at] = row;
    if (at % kTile == 0) {
        const int left = s.count[r] - at;
        s.tiles[off.y + at / kTile] = make_int4(r, off.x + at, left < kTile ? left : kTile, 0);
    }
}

// sorts `a` and, with both, `b` (of as many rows)
static inline void launch_sort(const Sort &a, const Sort &b, bool both, hipStream_t st) {
    const int E = both && b.E > a.E ? b.E : a.E, ny = both ? 2 : 1;
    auto go = [&](auto count, auto plan) {
        hipLaunchKernelGGL(count, dim3(a.groups, ny), dim3(1024), 0, st, a, b);
        hipLaunchKernelGGL(plan, dim3((E + 1023) / 1024, ny), dim3(1024), 0, st, a, b);
    };
    if (E <= 1024) go(rows_count<1024>, rows_plan<1024>);
    else if (E <= 4096) go(rows_count<4096>, rows_plan<4096>);
    else go(rows_count<kSortLeaves>, rows_plan<kSortLeaves>);
    hipLaunchKernelGGL(rows_scatter, dim3((a.N + 255) / 256, both ? 2 : 1), dim3(256), 0, st, a, b);
}

}  // namespace ygg::rows
