// The float step over many known tokens, layer by layer (ygg_float_run_scratch). The step of ygg_float.hip walks a
// stream token by token through every layer, so a token waits for all layers of the one before it. When the tokens are
// known only one term of the step is a recurrence, h(t) = u(t) + A_r(t) h(t - 1) inside each block of 16 coordinates;
// the route, the layer input, the expert's own input u = T_r[x] + U'_r (V' rms(h_below)) and the readout of a token need
// nothing of the token before it in the same layer. So each layer runs over all rows (stream, token) of a chunk:
//   fl_route    leaf and layer input of every row; 16 rows per workgroup
//   rows_count, counting sort of the rows by leaf, and its tiles of at most 32 rows of one expert (ygg_rows.h)
//   rows_plan, rows_scatter
//   fl_input    u: per tile the product of its rows' layer inputs and the expert's U', on the f32 / f64 matrix cores,
//               plus the table rows
//   fl_scan     the recurrence: 16 lanes per stream and block, A_r loaded ahead by token
// and after the last layer fl_readout (z = P_r h of every layer by the same tiles) and fl_logits (Q z, one product over
// the layers' ranks). The rows of few tokens are not sorted (a tile is one row then).
//
// Measured against the token-by-token kernel (whole calls, f32 unless said): 9 streams x 100 tokens of the medium
// trained shape 3 635 -> 169 us; scoring 256 x 128 of the large one 6 597 -> 884; f64 calibration of 500 x 200 of the
// medium one 45.6 -> 1.63 ms. The general step kernel is bound by the dependent loads and barriers of a layer (7 us
// each), this form by its launches (17 to 26 of 4 us) at a thousand rows and by the experts' bytes at tens of thousands.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "ygg_float.h"
#include "ygg_rows.h"

using namespace ygg::flt;
using namespace ygg::rows;

namespace {

// A scan's wavefront loads this many rows past a stream's last without a look (tokens ahead and a run of them).
constexpr int kPad = 64;

template <typename T> struct Vec;    // the 16-byte vector of T
template <> struct Vec<float> {
    using type = float4;
    static __device__ __forceinline__ float at(const float4 &v, int i) { return ((const float *)&v)[i]; }
};
template <> struct Vec<double> {
    using type = double2;
    static __device__ __forceinline__ double at(const double2 &v, int i) { return ((const double *)&v)[i]; }
};
template <typename T> constexpr int kVE = 16 / (int)sizeof(T);

// D(16 x 16) += A(16 x 4) B(4 x 16): lane l gives A[l % 16][l / 16] and B[l / 16][l % 16] and holds D[acc_row][l % 16]
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
template <typename T> struct Acc;
template <> struct Acc<float> { using type = f32x4; };
template <> struct Acc<double> { using type = f64x4; };
__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f64x4 mma(double a, double b, f64x4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
// the row of D that component i of lane group q = l / 16 holds
template <typename T> __device__ __forceinline__ int acc_row(int i, int q) { return sizeof(T) == 4 ? 4 * q + i : 4 * i + q; }

// v moved across lanes by a DPP control (both halves of a double)
template <int CTRL> __device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL> __device__ __forceinline__ double dpp(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// the sum over aligned groups of 16 lanes, in every lane
template <typename T> __device__ __forceinline__ T sum16(T v) {
    v += dpp<0xB1>(v);     // quad_perm 1 0 3 2
    v += dpp<0x4E>(v);     // quad_perm 2 3 0 1
    v += dpp<0x141>(v);    // row_half_mirror
    v += dpp<0x140>(v);    // row_mirror
    return v;
}
template <typename T> __device__ __forceinline__ T load_or_zero(const T *p, bool ok) { return ok ? *p : T(0); }
template <typename T> __device__ __forceinline__ typename Vec<T>::type load_vec(const T *p, bool ok) {
    typename Vec<T>::type v{};
    if (ok) v = *(const typename Vec<T>::type *)p;
    return v;
}

// One chunk of a call: Bc streams from s0, Tc of their Tn tokens from t0; row i = s Tc + t. Workspace arrays per layer
// lie N rows apart.
template <typename T> struct Chunk {
    const int32_t *tokens;
    int Tn, s0, Bc, t0, Tc, N;
    int ZLW, ZW;
    T *state, *logits;
    int32_t *leaves;
    double *stats;
    T *h;             // [L][N][n] (and kPad rows): u, then the states
    T *zl;            // [L][N][ZLW]: layer inputs, zero past R2
    T *z;             // [N][ZW]: readouts, layer l's at l R
    Sort by[YGG_MAX_LAYERS];      // the rows of each layer by expert
    int *r;           // [N + kPad] experts of the current layer's rows, 0 past a stream's end
    int *stop;        // [Bc] a stream's first token outside [0, V), or Tn

    __device__ __forceinline__ int len(int s) const {     // rows of stream s this chunk computes
        const int k = stop[s] - t0;
        return k < 0 ? 0 : (k < Tc ? k : Tc);
    }
    __device__ __forceinline__ size_t token_at(int row) const {
        const int s = row / Tc;
        return (size_t)(s0 + s) * Tn + t0 + (row - s * Tc);
    }
};

// Per stream (a workgroup) its end in this chunk, and layer 0's leaves (the tokens); the sort's counters cleared. The
// streams' ends carry over to the next chunk.
template <typename T> __global__ __launch_bounds__(256) void fl_begin(const FloatDevModel<T> m, const Chunk<T> c) {
    __shared__ int first;
    const int tid = threadIdx.x, s = blockIdx.x;
    for (int l = 0; l < m.L && s == 0; l++) sort_clear(c.by[l]);
    if (s == 0 && tid < kPad) c.r[c.N + tid] = 0;
    const int was = c.t0 ? c.stop[s] : c.Tn;
    if (tid == 0) first = was;
    __syncthreads();
    const size_t at = (size_t)(c.s0 + s) * c.Tn + c.t0, row0 = (size_t)s * c.Tc;
    for (int t = tid; t < c.Tc; t += 256) {
        const int x = c.tokens[at + t];
        if (x < 0 || x >= m.V) atomicMin(&first, c.t0 + t);
    }
    __syncthreads();
    const int stop = first;
    if (tid == 0) {
        c.stop[s] = stop;
        if (stop < was) atomicOr(m.err, 1u);
    }
    for (int t = tid; t < c.Tc; t += 256) {
        const int x = c.tokens[at + t];
        const bool live = c.t0 + t < stop;
        c.by[0].leaf[row0 + t] = live ? x : -1;
        c.r[row0 + t] = live ? x : 0;
        if (live && c.leaves) c.leaves[(at + t) * m.L] = x;
    }
}

// The route of layer l and its layer input: 16 rows per workgroup, 16 lanes per row. The descent reads one node row per
// level (rows of a layer stay in L2) with its input row in registers; the product V' rms(h) of the 16 rows is
// split over the wavefronts by coordinates. EPL: router inputs per lane at most; VW: their vector width (kVE where the
// token part is whole vectors, else 1). LV: levels a step; two (a node and both its children loaded together, half again
// the bytes) for few rows, which wait for the loads, one for many. The workgroups' LDS is theirs by n and R2 (route_of),
// the partial sums where the rows were: a workgroup waits for its loads most of the time, so what counts is how many fit
// a CU (100k f64 rows of the medium trained shape: 66 KB of LDS and two of them 124 us, 17 KB and eight 83).
template <typename T, int EPL, int VW, int LV>
__global__ __launch_bounds__(256) void fl_route(const FloatDevModel<T> m, const Chunk<T> c, int l) {
    constexpr int VE = kVE<T>, KC = 4 * VE, CGS = kMaxR2 / (16 * VE);
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const FloatLayerDev<T> &y = m.layers[l];
    const int n = m.n, F = m.F, LD = n + VE, width = F + (m.router_state ? n : 0);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rl = tid & 15, rr = tid >> 4;
    const int row = blockIdx.x * 16 + rr;
    const int s = row / c.Tc;
    const bool live = row < c.N && row - s * c.Tc < c.len(s);
    T *const f16 = (T *)lds, *const part = (T *)lds;      // rms(h_below) of the rows, LD apart; then [4][16][R2 + 1]
    {
        const T *h = c.h + ((size_t)(l - 1) * c.N + (live ? row : 0)) * n;
        typename Vec<T>::type v[kMaxN / (16 * VE)];
        T ss = T(0);
#pragma unroll
        for (int k = 0; k < kMaxN / (16 * VE); k++) {
            const int e = VE * (rl + 16 * k);
            v[k] = load_vec(h + e, live && e < n);
#pragma unroll
            for (int q = 0; q < VE; q++) ss = fma(Vec<T>::at(v[k], q), Vec<T>::at(v[k], q), ss);
        }
        const T rinv = T(1) / sqrt(sum16(ss) / T(n) + T(kRmsEps));
#pragma unroll
        for (int k = 0; k < kMaxN / (16 * VE); k++) {
            const int e = VE * (rl + 16 * k);
            if (e < n)
#pragma unroll
                for (int q = 0; q < VE; q++) f16[rr * LD + e + q] = Vec<T>::at(v[k], q) * rinv;
        }
    }
    __syncthreads();
    const size_t at = live ? c.token_at(row) : 0;
    if (live) {
        const T *emb = y.emb + (size_t)c.tokens[at] * F;
        T f[EPL];
#pragma unroll
        for (int k = 0; k < EPL / VW; k++) {
#pragma unroll
            for (int q = 0; q < VW; q++) {
                const int e = VW * (rl + 16 * k) + q;
                f[VW * k + q] = e < F ? emb[e] : (e < width ? f16[rr * LD + e - F] : T(0));
            }
        }
        // the lane's products with a node's row, loaded by load
        using Row = std::conditional_t<(VW > 1), typename Vec<T>::type, T>;
        constexpr int RW = VW > 1 ? EPL / VE : EPL;
        auto load = [&](Row (&wv)[RW], int at) {
            const T *w = y.W + (size_t)at * width;
#pragma unroll
            for (int k = 0; k < RW; k++) {
                const int e = VW * (rl + 16 * k);
                if constexpr (VW > 1) wv[k] = load_vec(w + e, e < width);
                else wv[k] = load_or_zero(w + e, e < width);
            }
        };
        auto score = [&](const Row (&wv)[RW]) {
            T p = T(0);
#pragma unroll
            for (int k = 0; k < RW; k++) {
                if constexpr (VW > 1) {
#pragma unroll
                    for (int q = 0; q < VE; q++) p = fma(f[VE * k + q], Vec<T>::at(wv[k], q), p);
                } else {
                    p = fma(f[k], wv[k], p);
                }
            }
            return sum16(p);
        };
        int node = 0, d = 0;
        if constexpr (LV == 2) {
            for (; d + 2 <= m.D; d += 2) {
                const int at[3] = {node, 2 * node + 1, 2 * node + 2};
                Row wv[3][RW];
                T bias[3];
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    load(wv[k], at[k]);
                    bias[k] = y.bias[at[k]];
                }
                T p[3];
#pragma unroll
                for (int k = 0; k < 3; k++) p[k] = score(wv[k]) + bias[k];
                const bool right = p[0] > T(0);
                node = 2 * (right ? at[2] : at[1]) + 1 + ((right ? p[2] : p[1]) > T(0) ? 1 : 0);
            }
        }
        for (; d < m.D; d++) {
            Row wv[RW];
            load(wv, node);
            const T bias = y.bias[node];
            node = 2 * node + 1 + (score(wv) + bias > T(0) ? 1 : 0);
        }
        if (rl == 0) {
            const int r = node - ((1 << m.D) - 1);
            c.by[l].leaf[row] = c.r[row] = r;
            if (c.leaves) c.leaves[at * m.L + l] = r;
        }
    } else if (row < c.N && rl == 0) {
        c.by[l].leaf[row] = -1;
        c.r[row] = 0;
    }
    if (!y.Vd) return;
    const int R2 = m.R2, kk = lane >> 4, cl = lane & 15;
    const bool whole = R2 % VE == 0;
    typename Acc<T>::type acc[CGS][VE];
#pragma unroll
    for (int g = 0; g < CGS; g++) {
#pragma unroll
        for (int q = 0; q < VE; q++) acc[g][q] = typename Acc<T>::type{};
        const int col = 16 * VE * g + VE * cl;
        if (16 * VE * g >= R2) break;
        for (int j = wave; j < n / KC; j += 4) {
            const int i0 = KC * j + VE * kk;
#pragma unroll
            for (int u = 0; u < VE; u++) {
                const T a = f16[cl * LD + i0 + u];
                const T *b = y.Vd + (size_t)(i0 + u) * R2 + col;
                typename Vec<T>::type bv{};
                if (whole) {
                    bv = load_vec(b, col < R2);
                } else {
#pragma unroll
                    for (int q = 0; q < VE; q++)
                        if (col + q < R2) ((T *)&bv)[q] = b[q];
                }
#pragma unroll
                for (int q = 0; q < VE; q++) acc[g][q] = mma(a, Vec<T>::at(bv, q), acc[g][q]);
            }
        }
    }
    __syncthreads();      // (every wavefront has read the rows)
#pragma unroll
    for (int g = 0; g < CGS; g++) {
        const int col = 16 * VE * g + VE * cl;
#pragma unroll
        for (int q = 0; q < VE; q++)
            if (col + q < R2)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    part[(wave * 16 + acc_row<T>(i, kk)) * (R2 + 1) + col + q] = acc[g][q][i];
    }
    __syncthreads();
    for (int i = tid; i < 16 * c.ZLW; i += 256) {
        const int k = i % c.ZLW, mrow = i / c.ZLW, to = blockIdx.x * 16 + mrow;
        if (to >= c.N) break;
        T z = T(0);
        if (k < R2) {
            auto of = [&](int w) { return part[(w * 16 + mrow) * (R2 + 1) + k]; };
            z = ((of(0) + of(1)) + of(2)) + of(3);
        }
        c.zl[((size_t)l * c.N + to) * c.ZLW + k] = z;
    }
}

// the maximum of a non-negative v over the wavefront into *p (non-negative doubles order as their bit patterns; most
// wavefronts find a larger one there and add nothing)
__device__ __forceinline__ void max_into(double *p, double v, int lane) {
    for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    if (lane == 0 && v > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax((unsigned long long *)p, (unsigned long long)__double_as_longlong(v));
}

// u = T_r[x] + U'_r zl of layer l: a wavefront per tile and 16 VE columns (each lane VE adjacent ones, so that U', the
// table rows and u move in 16-byte pieces)
template <typename T> __global__ __launch_bounds__(256) void fl_input(const FloatDevModel<T> m, const Chunk<T> c, int l) {
    constexpr int VE = kVE<T>, KC = 4 * VE;
    const FloatLayerDev<T> &y = m.layers[l];
    const int n = m.n, R2 = m.R2, CG = (n + 16 * VE - 1) / (16 * VE);
    const int lane = threadIdx.x & 63, kk = lane >> 4, cl = lane & 15;
    const int total = tiles_of(c.by[l]) * CG;
    double zmax = 0.0;      // (calibration) the largest layer input
    for (int w = blockIdx.x * 4 + (threadIdx.x >> 6); w < total; w += gridDim.x * 4) {
        const int4 tile = tile_at(c.by[l], w / CG);
        const int r = tile.x, cnt = tile.z;
        if (cnt == 0) continue;
        const int col = (w % CG) * 16 * VE + VE * cl;
        const bool cok = col < n, two = cnt > 16;
        int rows[2];
        for (int q = 0; q < 2; q++) rows[q] = row_at(c.by[l], tile.y + (16 * q + cl < cnt ? 16 * q + cl : 0));
        typename Acc<T>::type acc[2][VE];
#pragma unroll
        for (int q = 0; q < VE; q++) acc[0][q] = acc[1][q] = typename Acc<T>::type{};
        const T *up = y.Up ? y.Up + (size_t)r * R2 * n + col : nullptr;
        const T *z0 = c.zl + ((size_t)l * c.N + rows[0]) * c.ZLW, *z1 = c.zl + ((size_t)l * c.N + rows[1]) * c.ZLW;
        if (up) {
            for (int j = 0; j < c.ZLW / KC; j++) {
                const int k0 = KC * j + VE * kk;
                typename Vec<T>::type b[VE], a0 = load_vec(z0 + k0, true), a1 = load_vec(z1 + k0, two);
#pragma unroll
                for (int u = 0; u < VE; u++) b[u] = load_vec(up + (size_t)(k0 + u) * n, cok && k0 + u < R2);
                if (c.stats)
#pragma unroll
                    for (int u = 0; u < VE; u++)
                        zmax = fmax(zmax, fmax((double)fabs(Vec<T>::at(a0, u)), (double)fabs(Vec<T>::at(a1, u))));
#pragma unroll
                for (int u = 0; u < VE; u++)
#pragma unroll
                    for (int q = 0; q < VE; q++) acc[0][q] = mma(Vec<T>::at(a0, u), Vec<T>::at(b[u], q), acc[0][q]);
                if (two)
#pragma unroll
                    for (int u = 0; u < VE; u++)
#pragma unroll
                        for (int q = 0; q < VE; q++) acc[1][q] = mma(Vec<T>::at(a1, u), Vec<T>::at(b[u], q), acc[1][q]);
            }
        }
        for (int q = 0; q < 2; q++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int p = 16 * q + acc_row<T>(i, kk);
                if (p < cnt && cok) {
                    const int row = row_at(c.by[l], tile.y + p);
                    typename Vec<T>::type t = *(const typename Vec<T>::type *)(
                        y.table + ((size_t)r * m.V + c.tokens[c.token_at(row)]) * n + col);
#pragma unroll
                    for (int e = 0; e < VE; e++) ((T *)&t)[e] += q ? acc[1][e][i] : acc[0][e][i];
                    *(typename Vec<T>::type *)(c.h + ((size_t)l * c.N + row) * n + col) = t;
                }
            }
        }
    }
    if (c.stats) max_into(c.stats + (size_t)l * (3 + n / 16 + m.R) + 1, zmax, lane);
}

// a . h over the 16 coordinates of a block, h spread one per lane: column j's factor by a row broadcast; four partial sums
template <typename T, int J = 0> __device__ __forceinline__ void block_dot(const T (&a)[16], T h, T (&s)[4]) {
    if constexpr (J < 16) {
        s[J % 4] = fma(a[J], dpp<0x150 + J>(h), s[J % 4]);
        block_dot<T, J + 1>(a, h, s);
    }
}

// The recurrence of layer l, h(t) = u(t) + A_r(t) h(t - 1): 16 lanes per stream and block of 16 coordinates, four
// streams of one block per wavefront (past the last stream its duplicates, whose equal stores change nothing), the next PD
// tokens' A rows and inputs loaded ahead and their experts PD further. Loads run past a stream's end without a look (the
// rows behind it, or kPad more): what they bring is never used. A wavefront on a SIMD of its own issues an instruction
// every 4 cycles, so a step is kept short: the factors h_j come as row broadcasts inside the multiply-adds. Workgroup b
// takes block b % (n / 16): workgroups go to the XCDs in turn, so where n / 16 divides or is a multiple of 8 an XCD meets
// (n / 16) / 8 blocks, or one, whose share of the layer's A stays in its L2. Layer 0 (L0) takes its input from the table.
template <typename T, int PD, bool L0>
__global__ __launch_bounds__(64) void fl_scan(const FloatDevModel<T> m, const Chunk<T> c, int l) {
    constexpr int VE = kVE<T>, CH = 16 / VE;
    const FloatLayerDev<T> &y = m.layers[l];
    const int n = m.n, nb = n / 16, g = blockIdx.x % nb, lane = threadIdx.x & 63, i = lane & 15;
    const int sw = blockIdx.x / nb * 4 + (lane >> 4), s = sw < c.Bc ? sw : c.Bc - 1;
    const int len = c.len(s);
    int most = len, least = len;          // the most and the fewest tokens of the wavefront's streams
    for (int o = 16; o < 64; o <<= 1) {
        const int a = __shfl_xor(most, o), b = __shfl_xor(least, o);
        most = a > most ? a : most;
        least = b < least ? b : least;
    }
    most = __builtin_amdgcn_readfirstlane(most);
    least = __builtin_amdgcn_readfirstlane(least);
    if (most == 0) return;
    T *st = c.state + ((size_t)(c.s0 + s) * m.L + l) * n + g * 16 + i;
    T *h = c.h + ((size_t)l * c.N + (size_t)s * c.Tc) * n + g * 16 + i;
    const int *rs = c.r + (size_t)s * c.Tc;
    const T *table = y.table + g * 16 + i;
    T hv = *st;
    if (!y.A) {     // no recurrence
        for (int t = 0; t < len; t++) {
            hv = L0 ? table[(size_t)rs[t] * n] : h[(size_t)t * n];
            if (L0) h[(size_t)t * n] = hv;
        }
        *st = hv;
        return;
    }
    const T *A = y.A + (size_t)g * 256 + VE * i;
    const uint32_t stride = (uint32_t)nb * 256;      // entries of an expert's A
    typename Vec<T>::type a[PD][CH];
    T u[PD];
    int r[PD];
    auto fetch = [&](int k, int d) {       // the token d rows on, whose expert is in r[k], into slot k
        // (the expert is used here and no earlier: hoisted, its use waits for every load up to its own, PD tokens early)
        asm volatile("" : "+v"(r[k]));
        const T *ab = A + (uint64_t)(uint32_t)r[k] * stride;
#pragma unroll
        for (int q = 0; q < CH; q++) a[k][q] = *(const typename Vec<T>::type *)(ab + q * 16 * VE);
        u[k] = L0 ? table[(uint64_t)(uint32_t)r[k] * (uint32_t)n] : h[(size_t)(d * n)];
    };
#pragma unroll
    for (int k = 0; k < PD; k++) r[k] = rs[k];
    // (in the loop's order: the waits at its top are those of the worse of the two ways in)
#pragma unroll
    for (int k = 0; k < PD; k++) {
        fetch(k, k);
        r[k] = rs[PD + k];
    }
    auto run = [&](auto tail, int left) {
#pragma unroll
        for (int k = 0; k < PD; k++) {
            T av[16], sums[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll
            for (int j = 0; j < 16; j++) av[j] = Vec<T>::at(a[k][j / VE], j % VE);
            block_dot<T>(av, hv, sums);
            const T hn = u[k] + ((sums[0] + sums[1]) + (sums[2] + sums[3]));
            const bool on = !decltype(tail)::value || k < left;
            hv = on ? hn : hv;
            if (on) h[(size_t)(k * n)] = hv;
            fetch(k, k + PD);
            r[k] = rs[k + 2 * PD];
        }
        h += (size_t)(PD * n);
        rs += PD;
    };
    int t0 = 0;
    for (; t0 + PD <= least; t0 += PD) run(std::false_type(), PD);
    for (; t0 < most; t0 += PD) run(std::true_type(), len - t0);
    *st = hv;
}

// z = P_r h of every layer (blockIdx.y): a wavefront per tile; CT column tiles of 16 ranks, each summed in VE chains (a
// shorter chain of additions rounds less). STATS: also the calibration maxima (cpu/export.py:127-153) of the states and
// of the readouts; places past a tile's rows repeat its first row, which changes no maximum.
template <typename T, int CT, bool STATS>
__global__ __launch_bounds__(256) void fl_readout(const FloatDevModel<T> m, const Chunk<T> c) {
    constexpr int VE = kVE<T>, KC = 4 * VE, G = kMaxN / 16;
    const int l = blockIdx.y;
    const FloatLayerDev<T> &y = m.layers[l];
    const int n = m.n, R = m.R, lane = threadIdx.x & 63, kk = lane >> 4, cl = lane & 15;
    const int total = tiles_of(c.by[l]);
    double hmax[STATS ? G : 1], rmax[STATS ? CT : 1];
    for (double &v : hmax) v = 0.0;
    for (double &v : rmax) v = 0.0;
    for (int w = blockIdx.x * 4 + (threadIdx.x >> 6); w < total; w += gridDim.x * 4) {
        const int4 tile = tile_at(c.by[l], w);
        const int r = tile.x, cnt = tile.z;
        if (cnt == 0) continue;
        const bool two = cnt > 16;
        int rows[2];
        for (int q = 0; q < 2; q++) rows[q] = row_at(c.by[l], tile.y + (16 * q + cl < cnt ? 16 * q + cl : 0));
        const T *h0 = c.h + ((size_t)l * c.N + rows[0]) * n, *h1 = c.h + ((size_t)l * c.N + rows[1]) * n;
        typename Acc<T>::type acc[2][CT][VE];
#pragma unroll
        for (int q = 0; q < CT; q++)
#pragma unroll
            for (int u = 0; u < VE; u++) acc[0][q][u] = acc[1][q][u] = typename Acc<T>::type{};
        auto step = [&](int j) {
            const int i0 = KC * j + VE * kk;
            const typename Vec<T>::type a0 = load_vec(h0 + i0, true), a1 = load_vec(h1 + i0, two);
            typename Vec<T>::type b[CT];
#pragma unroll
            for (int q = 0; q < CT; q++)
                b[q] = load_vec(y.P + ((size_t)r * R + 16 * q + cl) * n + i0, 16 * q + cl < R);
            double top = 0.0;
            if constexpr (STATS)
#pragma unroll
                for (int u = 0; u < VE; u++)
                    top = fmax(top, fmax((double)fabs(Vec<T>::at(a0, u)), (double)fabs(Vec<T>::at(a1, u))));
#pragma unroll
            for (int q = 0; q < CT; q++)
#pragma unroll
                for (int u = 0; u < VE; u++) acc[0][q][u] = mma(Vec<T>::at(a0, u), Vec<T>::at(b[q], u), acc[0][q][u]);
            if (two)
#pragma unroll
                for (int q = 0; q < CT; q++)
#pragma unroll
                    for (int u = 0; u < VE; u++) acc[1][q][u] = mma(Vec<T>::at(a1, u), Vec<T>::at(b[q], u), acc[1][q][u]);
            return top;
        };
        if constexpr (STATS) {
#pragma unroll
            for (int g = 0; g < G; g++)
                if (16 * g < n)
#pragma unroll
                    for (int j = 0; j < 16 / KC; j++) hmax[g] = fmax(hmax[g], step(16 / KC * g + j));
        } else {
            for (int j = 0; j < n / KC; j++) step(j);
        }
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int k = 16 * p + acc_row<T>(i, kk);
                if (k >= cnt) continue;
                T *z = c.z + (size_t)row_at(c.by[l], tile.y + k) * c.ZW + l * R;
#pragma unroll
                for (int q = 0; q < CT; q++) {
                    T v;
                    if constexpr (VE == 4) v = (acc[p][q][0][i] + acc[p][q][1][i]) + (acc[p][q][2][i] + acc[p][q][3][i]);
                    else v = acc[p][q][0][i] + acc[p][q][1][i];
                    if (16 * q + cl < R) z[16 * q + cl] = v;
                    if constexpr (STATS) rmax[q] = fmax(rmax[q], (double)fabs(v));
                }
            }
    }
    if constexpr (STATS) {
        double *st = c.stats + (size_t)l * (3 + n / 16 + R), top = 0.0;
#pragma unroll
        for (int g = 0; g < G; g++)
            if (16 * g < n) {
                max_into(st + 3 + g, hmax[g], lane);
                top = fmax(top, hmax[g]);
            }
        max_into(st, top, lane);
        top = 0.0;
#pragma unroll
        for (int q = 0; q < CT; q++) {
            // the maximum of column cl over the four lane groups
            double v = fmax(rmax[q], __shfl_xor(rmax[q], 16));
            v = fmax(v, __shfl_xor(v, 32));
            double *p = st + 3 + n / 16 + 16 * q + cl;
            if (kk == 0 && 16 * q + cl < R && v > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                atomicMax((unsigned long long *)p, (unsigned long long)__double_as_longlong(v));
            if (16 * q + cl < R) top = fmax(top, v);
        }
        max_into(st + 2, top, lane);
    }
}

// logits = bias + sum over the layers of Q z: 32 consecutive rows per workgroup, a wavefront per 16 VE classes (VEC: the
// classes are whole 16-byte vectors of the logits and of Q)
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void fl_logits(const FloatDevModel<T> m, const Chunk<T> c) {
    constexpr int VE = kVE<T>, KC = 4 * VE;
    const int C = m.classes, LR = m.L * m.R, lane = threadIdx.x & 63, kk = lane >> 4, cl = lane & 15;
    const T *Q = m.layers[0].Q;
    const int r0 = blockIdx.x * 32;
    for (int c0 = (threadIdx.x >> 6) * 16 * VE; c0 < C; c0 += 4 * 16 * VE) {
        // class of component q: adjacent ones with VEC, else 16 apart
        const int col = VEC ? c0 + VE * cl : c0 + cl, step = VEC ? 1 : 16;
        // (two chains of additions per sum, joined with the bias last)
        typename Acc<T>::type acc[2][2][VE];
        T bias[VE];
#pragma unroll
        for (int q = 0; q < VE; q++) {
            bias[q] = load_or_zero(m.output_bias + col + q * step, col + q * step < C);
            for (int p = 0; p < 2; p++) acc[p][0][q] = acc[p][1][q] = typename Acc<T>::type{};
        }
        const T *z0 = c.z + (size_t)(r0 + cl < c.N ? r0 + cl : 0) * c.ZW;
        const T *z1 = c.z + (size_t)(r0 + 16 + cl < c.N ? r0 + 16 + cl : 0) * c.ZW;
        for (int j = 0; j < c.ZW / KC; j++) {
            const int k0 = KC * j + VE * kk;
            typename Vec<T>::type a0 = load_vec(z0 + k0, true), a1 = load_vec(z1 + k0, true), b[VE];
#pragma unroll
            for (int u = 0; u < VE; u++) {
                const bool kok = k0 + u < LR;
                if (!kok) ((T *)&a0)[u] = ((T *)&a1)[u] = T(0);
                b[u] = typename Vec<T>::type{};
                if constexpr (VEC) {
                    b[u] = load_vec(Q + (size_t)(k0 + u) * C + col, kok && col < C);
                } else {
#pragma unroll
                    for (int q = 0; q < VE; q++)
                        ((T *)&b[u])[q] = load_or_zero(Q + (size_t)(k0 + u) * C + col + q * 16, kok && col + q * 16 < C);
                }
            }
#pragma unroll
            for (int u = 0; u < VE; u++)
#pragma unroll
                for (int q = 0; q < VE; q++) {
                    acc[0][u & 1][q] = mma(Vec<T>::at(a0, u), Vec<T>::at(b[u], q), acc[0][u & 1][q]);
                    acc[1][u & 1][q] = mma(Vec<T>::at(a1, u), Vec<T>::at(b[u], q), acc[1][u & 1][q]);
                }
        }
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = r0 + 16 * p + acc_row<T>(i, kk);
                if (row >= c.N) continue;
                const int s = row / c.Tc;
                if (row - s * c.Tc >= c.len(s)) continue;
                T *out = c.logits + c.token_at(row) * C + col;
                if constexpr (VEC) {
                    typename Vec<T>::type v;
#pragma unroll
                    for (int q = 0; q < VE; q++) ((T *)&v)[q] = bias[q] + (acc[p][0][q][i] + acc[p][1][q][i]);
                    if (col < C) *(typename Vec<T>::type *)out = v;
                } else {
#pragma unroll
                    for (int q = 0; q < VE; q++)
                        if (col + q * 16 < C) out[q * 16] = bias[q] + (acc[p][0][q][i] + acc[p][1][q][i]);
                }
            }
    }
}

// -log softmax(logits)[y] of each row in f64: a wavefront per 4 rows, 64 lanes over a row's classes, the 4 rows' loads
// issued together; bound by the f64 exponentials. 32 768 f32 rows of 256 classes: 24 us, where a copy in f64, its log
// softmax, a gather and a negation took 57.
template <typename T>
__global__ __launch_bounds__(256) void fl_nll(const T *__restrict__ logits, const int32_t *__restrict__ y, int64_t rows,
                                              int C, double *__restrict__ nll) {
    constexpr int K = kMaxClasses / 64;
    const int lane = threadIdx.x & 63;
    const int64_t r0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 4;
    T v[4][K], at[4];
    bool known[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int64_t row = r0 + q < rows ? r0 + q : rows - 1;
        const T *lg = logits + row * C;
        const int c = y[row];
        known[q] = c >= 0 && c < C;
        at[q] = lg[known[q] ? c : 0];
#pragma unroll
        for (int k = 0; k < K; k++) v[q][k] = lane + 64 * k < C ? lg[lane + 64 * k] : (T)-INFINITY;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        T top = v[q][0];
#pragma unroll
        for (int k = 1; k < K; k++) top = v[q][k] > top ? v[q][k] : top;
        for (int o = 32; o > 0; o >>= 1) {
            const T other = __shfl_xor(top, o);
            top = other > top ? other : top;
        }
        double sum = 0.0;
#pragma unroll
        for (int k = 0; k < K; k++) sum += lane + 64 * k < C ? exp((double)v[q][k] - (double)top) : 0.0;
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        if (lane == 0 && r0 + q < rows) nll[r0 + q] = known[q] ? log(sum) - ((double)at[q] - (double)top) : (double)NAN;
    }
}

// ------------------------------------------------------------------------------------------------------ host side
// Bytes of an expert's record (A, U' and P) a row reads
template <typename T> int64_t record_bytes(const FloatDevModel<T> &m) { return (int64_t)sizeof(T) * m.n * (16 + m.R2 + m.R); }

// Sorting pays once it keeps about 130 MB of experts' records from being read again: its launches cost 60 to 80 us. Rows
// where both are as fast, 1024 experts, depth 10 (n = 64 / 128 / 256): f32 about 14000 / 5000 / 2000, f64 6500 / 2500 /
// 1200, which is 130 to 160, 160 and 230 to 270 MB; 8192 rows in f32, sorted / not: 247 / 218, 283 / 321, 438 / 778 us.
constexpr int64_t kSortBytes = 130'000'000;
bool sort_pays(int64_t N, int E, int64_t record) { return E <= kSortLeaves && N > E && (N - E) * record >= kSortBytes; }

struct Plan {
    int64_t fixed, per_row;      // workspace bytes besides the rows' and the sorts', and per row (arrays rounded up apart)
    int L, E, ZLW, ZW;
    int64_t record;              // bytes of an expert's record
    // workspace bytes of a chunk of N rows, more for more rows
    int64_t bytes(int64_t N) const { return fixed + per_row * N + L * sort_fixed_bytes(N, E, sort_pays(N, E, record)); }
};

template <typename T> Plan plan_of(const FloatDevModel<T> &m, int64_t B) {
    Plan p{};
    p.L = m.L;
    const int64_t leaves = m.L > 1 ? (int64_t)1 << m.D : 1;
    p.E = (int)(leaves > m.V ? leaves : m.V);
    p.record = record_bytes(m);
    p.ZLW = (m.R2 + 15) / 16 * 16;
    p.ZW = (m.L * m.R + 15) / 16 * 16;
    p.per_row = (int64_t)sizeof(T) * ((int64_t)m.L * (m.n + p.ZLW) + p.ZW) + 4 + m.L * kSortRowBytes;
    p.fixed = 256 * 8 + B * 4 + kPad * (4 + (int64_t)m.n * sizeof(T));
    return p;
}

// Calls of fewer than 4 tokens stay on the step kernel, and so do transition blocks other than 16. A model without a
// step build of its own comes here from 4 tokens, where this form is far ahead of the general kernel: 4 tokens of 1 / 16 /
// 256 / 1024 streams took (us, general kernel / this form), at depth 10 and 5 layers, n = 64, R = 12, R2 = 16 in f32 399/75
// 411/82 399/95 1585/126; n = 256, R = R2 = 32 in f32 436/109 448/134 451/189 1799/345, in f64 492/133 499/165 503/324
// 1995/490; n = 256, R = R2 = 64, 8 layers of depth 6, f64 817/265 830/343 850/505 3360/727; n = 16, 2 layers of depth 3,
// f32 104/24 108/28 106/27 416/32; a token layer alone, n = 64, f64 55/16 56/18 56/18 221/24. (Fewer tokens were not
// compared.)
// With a step build (float_steps) the cheaper is estimated: a step's tokens, by rounds of the streams that fit the chip,
// against this form's launches, the records its rows read (1.2 TB/s) and the sort. Measured at 4 and 8 tokens: small,
// 1 stream 54/75 104/77, 256 58/96 112/105, 1024 71/150 139/169; medium 57/90 109/91, 76/125 146/146, 152/190 295/248;
// large 87/115 182/117, 121/230 230/326, 455/388 892/435. (The step's build for the calls that its plain one does not take
// is up to a third slower for one stream; the maxima cost both forms.)
constexpr int kScanTokens = 4;
constexpr int64_t kScratchCap = (int64_t)1 << 30;

template <typename T> bool takes(const FloatDevModel<T> &m, int64_t B, int64_t Tn) {
    if (m.b != 16 || B <= 0 || Tn < kScanTokens) return false;
    if (!float_steps(m)) return true;
    const int64_t N = B * Tn, leaves = m.L > 1 ? (int64_t)1 << m.D : 1, E = leaves > m.V ? leaves : m.V;
    const bool sorted = sort_pays(N, (int)E, record_bytes(m));
    const double step = (double)Tn * ((B * m.n + 65535) / 65536) * (12.5 + m.n * m.n / 4096.0);
    const double scan = 60 + m.n / 4.0 + (double)(sorted ? E : N) * record_bytes(m) * 8.3e-7 +
                        (sorted ? 60 + (double)N * m.n * sizeof(T) * 1.8e-5 : 0.0);
    return scan < step;
}

template <typename T> int64_t scratch_of(const FloatDevModel<T> &m, int64_t B, int64_t Tn) {
    if (!takes(m, B, Tn)) return 0;
    const Plan p = plan_of(m, B);
    return (int64_t)up256(std::min(p.bytes(B * Tn), std::max(kScratchCap, p.bytes(64))));
}

// Rows below which the route takes two levels a step.
constexpr int kFewRows = 8192;

template <typename T, int EPL> void route_of(const FloatDevModel<T> &m, const Chunk<T> &c, int l, hipStream_t st) {
    const size_t rows = 16 * (size_t)(m.n + kVE<T>), parts = 64 * (size_t)(m.R2 + 1), lds = std::max(rows, parts) * sizeof(T);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((c.N + 15) / 16), dim3(256), lds, st, m, c, l); };
    if (m.F % kVE<T>) go(fl_route<T, EPL, 1, 1>);
    else if (c.N < kFewRows) go(fl_route<T, EPL, kVE<T>, 2>);
    else go(fl_route<T, EPL, kVE<T>, 1>);
}

template <typename T>
int scan_run(const FloatDevModel<T> &m, const int32_t *tokens, int B, int Tn, T *state, T *logits, int32_t *leaves,
             double *stats, void *scratch, int64_t bytes, hipStream_t st) {
    const Plan p = plan_of(m, B);
    // a chunk's rows; whole calls where they fit, else runs of at least 128 tokens of as many streams as fit
    const int64_t rows = rows_that_fit((int64_t)B * Tn, bytes, [&](int64_t N) { return p.bytes(N); });
    if (rows < 1) return fail(YGG_ERR_ARG, "float scratch of %lld bytes is too small", (long long)bytes);
    int64_t Tc = Tn, Bc = B;
    if ((int64_t)B * Tn > rows) {
        Tc = rows / B > 128 ? rows / B : 128;
        if (Tc > Tn) Tc = Tn;
        if (Tc > rows) Tc = rows;
        Bc = rows / Tc < B ? rows / Tc : B;
    }
    const int width = m.F + (m.router_state ? m.n : 0);
    for (int s0 = 0; s0 < B; s0 += (int)Bc)
        for (int t0 = 0; t0 < Tn; t0 += (int)Tc) {
            Chunk<T> c{};
            c.tokens = tokens;
            c.Tn = Tn;
            c.s0 = s0;
            c.Bc = (int)(B - s0 < Bc ? B - s0 : Bc);
            c.t0 = t0;
            c.Tc = (int)(Tn - t0 < Tc ? Tn - t0 : Tc);
            c.N = c.Bc * c.Tc;
            c.ZLW = p.ZLW;
            c.ZW = p.ZW;
            const bool sorted = sort_pays(c.N, p.E, p.record);
            c.state = state;
            c.logits = logits;
            c.leaves = leaves;
            c.stats = stats;
            uint8_t *w = (uint8_t *)scratch;
            auto take = [&](size_t k) {
                uint8_t *q = w;
                w += up256(k);
                return q;
            };
            const size_t N = (size_t)c.N;
            c.stop = (int *)take((size_t)B * 4);
            for (int l = 0; l < m.L; l++) lay_out(c.by[l], c.N, l ? 1 << m.D : m.V, sorted, take);
            c.z = (T *)take(N * p.ZW * sizeof(T));
            c.zl = (T *)take(N * m.L * p.ZLW * sizeof(T));
            c.r = (int *)take((N + kPad) * 4);
            c.h = (T *)take((N * m.L + kPad) * m.n * sizeof(T));
            if (w - (uint8_t *)scratch > bytes) return fail(YGG_ERR_ARG, "float scratch of %lld bytes is too small", (long long)bytes);
            auto scan = [&](int l) {
                constexpr int PD = sizeof(T) == 4 ? 8 : 5;
                const dim3 grid((c.Bc + 3) / 4 * (m.n / 16));
                if (l) hipLaunchKernelGGL((fl_scan<T, PD, false>), grid, dim3(64), 0, st, m, c, l);
                else hipLaunchKernelGGL((fl_scan<T, PD, true>), grid, dim3(64), 0, st, m, c, l);
            };
            hipLaunchKernelGGL(fl_begin<T>, dim3(c.Bc), dim3(256), 0, st, m, c);
            scan(0);
            for (int l = 1; l < m.L; l++) {
                if (width <= 128) route_of<T, 8>(m, c, l, st);
                else if (width <= 192) route_of<T, 12>(m, c, l, st);
                else if (width <= 320) route_of<T, 20>(m, c, l, st);
                else route_of<T, 32>(m, c, l, st);
                if (sorted) launch_sort(c.by[l], c.by[0], l == 1, st);
                const int64_t waves = (int64_t)(sorted ? c.by[l].max_tiles : c.N) * ((m.n + 16 * kVE<T> - 1) / (16 * kVE<T>));
                const int64_t wgs = (waves + 3) / 4;
                // (with the maxima each wavefront ends with additions of its own)
                const int64_t cap = stats ? 1024 : 8192;
                hipLaunchKernelGGL(fl_input<T>, dim3((unsigned)(wgs < cap ? wgs : cap)), dim3(256), 0, st, m, c, l);
                scan(l);
            }
            if (m.L == 1 && sorted) launch_sort(c.by[0], c.by[0], false, st);
            if (logits || stats) {
                const int64_t wgs = ((int64_t)(sorted ? c.N / kTile + p.E : c.N) + 3) / 4, most = stats ? 256 : 8192;
                const dim3 grid((unsigned)(wgs < most ? wgs : most), m.L);
                auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, m, c); };
                if (m.R <= 16) stats ? go(fl_readout<T, 1, true>) : go(fl_readout<T, 1, false>);
                else if (m.R <= 32) stats ? go(fl_readout<T, 2, true>) : go(fl_readout<T, 2, false>);
                else stats ? go(fl_readout<T, 4, true>) : go(fl_readout<T, 4, false>);
            }
            if (logits) {
                // 16-byte stores where every row of logits starts on 16 bytes
                const bool vec = m.classes % kVE<T> == 0 && (uintptr_t)logits % 16 == 0;
                const dim3 grid((c.N + 31) / 32);
                if (vec) hipLaunchKernelGGL((fl_logits<T, true>), grid, dim3(256), 0, st, m, c);
                else hipLaunchKernelGGL((fl_logits<T, false>), grid, dim3(256), 0, st, m, c);
            }
        }
    HIP_TRY(hipGetLastError());
    return YGG_OK;
}

}  // namespace

extern "C" {

int64_t ygg_float_scratch(const ygg_fmodel *m, int B, int T) {
    if (!m || B < 0 || T < 0) return 0;
    return m->precision == 32 ? scratch_of(m->m32, B, T) : scratch_of(m->m64, B, T);
}

int ygg_float_run_scratch(const ygg_fmodel *m, const int32_t *d_tokens, int B, int T, void *d_state, void *d_logits,
                          int32_t *d_leaves, double *d_stats, void *d_scratch, int64_t scratch_bytes, void *stream) {
    if (!m) return fail(YGG_ERR_ARG, "model is NULL");
    if (B < 0 || T < 0) return fail(YGG_ERR_ARG, "negative B (%d) or T (%d)", B, T);
    if (ygg_float_scratch(m, B, T) == 0)
        return ygg_float_run(m, d_tokens, B, T, d_state, d_logits, d_leaves, d_stats, stream);
    if (!d_state || !d_tokens) return fail(YGG_ERR_ARG, "tokens or state is NULL");
    if (!d_scratch || (uintptr_t)d_scratch % 256) return fail(YGG_ERR_ARG, "scratch is NULL or not on 256 bytes");
    DeviceGuard g;
    HIP_TRY(g.set(m->device));
    if (m->precision == 32)
        return scan_run(m->m32, d_tokens, B, T, (float *)d_state, (float *)d_logits, d_leaves, d_stats, d_scratch,
                        scratch_bytes, (hipStream_t)stream);
    return scan_run(m->m64, d_tokens, B, T, (double *)d_state, (double *)d_logits, d_leaves, d_stats, d_scratch,
                    scratch_bytes, (hipStream_t)stream);
}

int ygg_float_nll(const ygg_fmodel *m, const void *d_logits, const int32_t *d_next, int64_t rows, double *d_nll,
                  void *stream) {
    if (!m) return fail(YGG_ERR_ARG, "model is NULL");
    if (rows < 0 || rows > (int64_t)1 << 34) return fail(YGG_ERR_ARG, "%lld rows", (long long)rows);
    if (rows == 0) return YGG_OK;
    if (!d_logits || !d_next || !d_nll) return fail(YGG_ERR_ARG, "logits, next tokens or result is NULL");
    DeviceGuard g;
    HIP_TRY(g.set(m->device));
    const dim3 grid((unsigned)((rows + 15) / 16));
    if (m->precision == 32)
        hipLaunchKernelGGL(fl_nll<float>, grid, dim3(256), 0, (hipStream_t)stream, (const float *)d_logits, d_next, rows,
                           m->m32.classes, d_nll);
    else
        hipLaunchKernelGGL(fl_nll<double>, grid, dim3(256), 0, (hipStream_t)stream, (const double *)d_logits, d_next, rows,
                           m->m64.classes, d_nll);
    HIP_TRY(hipGetLastError());
    return YGG_OK;
}

}  // extern "C"
