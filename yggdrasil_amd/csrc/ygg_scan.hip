// The int8 step over many known tokens, layer by layer. The step kernels (ygg_kernel_fast.h) walk a stream token by
// token through every layer, and every token of every stream reads its experts' whole records. With the tokens known
// only the transition is a recurrence, q(t) = sat8((A16 q(t - 1) + half >> shift) + u(t)) inside each block of 16
// coordinates; the route, the layer input zl, the input u = T_r[x] + rint(f32(U'_r zl) m_ul), the readout and the logits of
// a token need nothing of the token before it in the same layer. So each layer runs over all rows (stream, token) of a
// chunk of the call:
//   s8_route    rho, leaf and layer input of every row
//   rows_count, counting sort of the rows by leaf and its tiles of at most 32 rows of one expert (ygg_rows.h)
//   rows_plan, rows_scatter
//   s8_tiles    per tile the inputs u of the layer and, for the layer below by its own tiles, the readouts zq, as int8
//               matrix products of the expert's U' (U_r) and P with the tile's rows
//   s8_scan     the recurrence: 16 lanes per stream and block, A16 loaded ahead by token
// and at the end s8_rows (the last layer's states row by row), s8_tiles for its readouts and s8_logits. Same integers and
// the same f32 operations in the same order as the step kernels (cpu/ygg.cpp:222-459), so the results are equal to the
// bit. u is held in 16 bits: it is clamped there, and |A16 q + half >> shift| <= 2^14 + 1 at shift >= 12, so the
// clamped sum saturates where the whole one does (scan_takes rules out inputs whose 32-bit sum could wrap).
//
// Calls of few rows are not sorted: s8_row takes a row's route, input and the readout below it in one wavefront, and
// s8_last the last layer's readouts.
//
// Measured (whole calls, token by token / layer by layer): 1 stream x 1001 tokens of the large trained shape 2 374 / 412
// us, 60 x 250 of the medium one factored 4 362 / 259, 4096 x 256 of the medium one 6 098 / 5 119 and of the large one
// 19.4 / 12.8 ms; configuration 4's model at 4096 x 1024 16.3 / 18.3, which the rule leaves token by token (scan_pays).
// At few rows it is bound by the recurrence's steps (70 ns each, the instructions of one wavefront) and the launches, at
// many by the A16 rows: 8.6 TB/s of them at configuration 4's model, 15 where an XCD's share stays in its L2.
//
// States and inputs pass between the kernels by block, [n / 16][row][16]: a scan's wavefront works on one block, so that an
// XCD (workgroups go to the XCDs in turn) meets one block's share of every expert's A16, an eighth of them at n = 128, and
// writes whole lines.
#include <algorithm>
#include <cmath>

#include "ygg_kernel_fast.h"
#include "ygg_launch.h"
#include "ygg_rows.h"
#include "ygg_scan.h"

namespace ygg {
namespace {

using namespace rows;

typedef int v4i32 __attribute__((ext_vector_type(4)));

// A scan's wavefront loads this many rows past a stream's last without a look (tokens ahead and a run of 16).
constexpr int kPad = 64;

struct ScanChunk {
    const int32_t *tokens;
    int Tn, s0, Bc, t0, Tc, N;
    int ZLW, ZQW;
    int8_t *state;
    YggIO io;
    int *x;           // [N + kPad] tokens, -1 past a stream's end
    uint32_t *rec;    // [N + kPad] byte offsets of the rows' gather records of the current layer (0 past a stream's end)
    int16_t *u;       // [n / 16][N][16] inputs of the current layer
    int8_t *q;        // [n / 16][N][16] states of the current layer
    int8_t *qr;       // [N][n] states of the layer below, row by row
    int8_t *zl;       // [N][ZLW] layer inputs
    int8_t *zq;       // [N][ZQW] readouts, layer l's at l R
    double2 *terms;   // [N] score: the sum of exponentials (0: no term) and the linear term of a row's NLL
    double4 *sums;    // [Bc] score: a stream's NllSum so far
    Sort by[2];       // rows by expert of layers of even and odd index
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

// Per stream (a workgroup) its end in this chunk, and layer 0's leaves (the tokens); the first sorts' counters cleared.
// The streams' ends carry over to the next chunk.
__global__ __launch_bounds__(256) void s8_begin(const YggDevModel m, const ScanChunk c) {
    __shared__ int first;
    const int tid = threadIdx.x, s = blockIdx.x;
    if (s == 0) {
        for (int p = 0; p < 2; p++) sort_clear(c.by[p]);
        if (tid < kPad) {
            c.x[c.N + tid] = -1;
            c.rec[c.N + tid] = 0u;
        }
    }
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
        c.x[row0 + t] = c.by[0].leaf[row0 + t] = live ? x : -1;
        c.rec[row0 + t] = live ? (uint32_t)x * (uint32_t)m.layers[0].gath_bytes : 0u;
        if (live && c.io.leaves) c.io.leaves[(at + t) * m.L] = x;
    }
}

// The 16-byte pieces (8 at n = 96) of an n-byte row that quad lane k holds: pieces k, k + 4, ...
template <int N> struct Pieces {
    static constexpr int W = N == 96 ? 8 : 16, K = N / W / 4, DW = W / 4;
};
template <int N> __device__ __forceinline__ void load_pieces(uint32_t (&w)[N / 16], const int8_t *row, int k) {
    using P = Pieces<N>;
#pragma unroll
    for (int j = 0; j < P::K; j++) {
        uint32_t v[P::DW];
        load_words<P::DW, P::W>(v, row + (k + 4 * j) * P::W);
#pragma unroll
        for (int i = 0; i < P::DW; i++) w[P::DW * j + i] = v[i];
    }
}

// The route of layer l (cpu/ygg.cpp:248-280) and its layer input (cpu/ygg.cpp:285-296): a wavefront per 16 rows, a quad
// per row, one node row per level; the 16 rows' product with V' on the matrix cores. Also leaves the states below row by
// row.
template <int N, bool GROUP>
__global__ __launch_bounds__(256) void s8_route(const YggDevModel m, const ScanChunk c, int l) {
    using P = Pieces<N>;
    constexpr int QW = N / 16, LD = N + 16;
    __shared__ __attribute__((aligned(16))) int8_t tile[4][16 * LD];
    const YggDevLayer &y = m.layers[l];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), k = lane & 3;
    const int r0 = (blockIdx.x * 4 + wave) * 16, row = r0 + (lane >> 2);
    if (blockIdx.x == 0) sort_clear(c.by[l & 1]);
    if (r0 >= c.N) return;
    const int x = row < c.N ? c.x[row] : -1;
    const bool live = x >= 0;
    uint32_t q[QW];
#pragma unroll
    for (int i = 0; i < QW; i++) q[i] = 0u;
    int8_t *mine = tile[wave] + (lane >> 2) * LD;
    if (live) {
#pragma unroll
        for (int j = 0; j < P::K; j++) {
            const int p = (k + 4 * j) * P::W;            // first coordinate of the piece
            uint32_t v[P::DW];
            load_words<P::DW, P::W>(v, c.q + ((size_t)(p / 16) * c.N + row) * 16 + p % 16);
#pragma unroll
            for (int i = 0; i < P::DW; i++) q[P::DW * j + i] = v[i];
        }
    }
    int S[P::K];
#pragma unroll
    for (int j = 0; j < P::K; j++) {
        const int p = (k + 4 * j) * P::W;
        S[j] = 0;
#pragma unroll
        for (int i = 0; i < P::DW; i++) {
            S[j] = dot4(q[P::DW * j + i], q[P::DW * j + i], S[j]);
            *(uint32_t *)(mine + p + 4 * i) = q[P::DW * j + i];
        }
        if (live) {
            int8_t *to = c.qr + (size_t)row * N + p;
            if constexpr (P::DW == 4) *(uint4 *)to = make_uint4(q[4 * j], q[4 * j + 1], q[4 * j + 2], q[4 * j + 3]);
            else *(uint2 *)to = make_uint2(q[2 * j], q[2 * j + 1]);
        }
    }
    float rho;
    if constexpr (GROUP) {
        // groups in order: group g's sum is S[g / 4] of quad lane g % 4
        float sum = 0.0f;
        auto add = [&](int g, int v) { sum = sum + y.r2b[g] * (float)v; };
#pragma unroll
        for (int j = 0; j < P::K; j++) {
            add(4 * j, __builtin_amdgcn_update_dpp(0, S[j], 0x00, 0xF, 0xF, false));
            add(4 * j + 1, __builtin_amdgcn_update_dpp(0, S[j], 0x55, 0xF, 0xF, false));
            add(4 * j + 2, __builtin_amdgcn_update_dpp(0, S[j], 0xAA, 0xF, 0xF, false));
            add(4 * j + 3, __builtin_amdgcn_update_dpp(0, S[j], 0xFF, 0xF, 0xF, false));
        }
        rho = 1.0f / sqrtf(sum * Fast<N>::kInvN + y.rms_eps);
    } else {
        int a = 0;
#pragma unroll
        for (int j = 0; j < P::K; j++) a += S[j];
        rho = 1.0f / sqrtf((float)sum4(a) * Fast<N>::kInvN + y.rms_eps);
    }
    if (live) {
        const float *thr = y.thr + (size_t)x * y.thr_stride;
        int ix = 1, base = 0, d0 = 0;
        for (int rd = 0; rd < m.n_rounds; rd++) {
            const int h = (m.round_pack >> (4 * rd)) & 15;
            const int blk = base + ((ix - (1 << d0)) << h);
            int j = 0;
            for (int d = 0; d < h; d++) {
                uint32_t w[QW];
                load_pieces<N>(w, y.w + (size_t)(blk + j) * N, k);
                const float th = thr[blk + j];
                int dot = 0;
#pragma unroll
                for (int i = 0; i < QW; i++) dot = dot4(w[i], q[i], dot);
                j = 2 * j + 1 + ((float)sum4(dot) * rho > th ? 1 : 0);
            }
            ix = (ix << h) + (j - ((1 << h) - 1));
            base += (1 << d0) << h;
            d0 += h;
        }
        if (k == 0) {
            c.by[l & 1].leaf[row] = ix - m.E;
            c.rec[row] = (uint32_t)(ix - m.E) * (uint32_t)y.gath_bytes;
            if (c.io.leaves) c.io.leaves[c.token_at(row) * m.L + l] = ix - m.E;
        }
    } else if (row < c.N && k == 0) {
        c.by[l & 1].leaf[row] = -1;
        c.rec[row] = 0u;
    }
    // the layer input: lane's row of V' is 16 p + lane % 16, its row of the tile lane % 16
    wave_sync();
    const int cl = lane & 15, kk = lane >> 4, to = r0 + cl;
    const float rm = __shfl(rho, 4 * cl);
    constexpr int KS = (N + 63) / 64;
    v4i32 qv[KS];
#pragma unroll
    for (int t = 0; t < KS; t++) {
        qv[t] = v4i32{0, 0, 0, 0};
        if (64 * t + 16 * kk < N) qv[t] = *(const v4i32 *)(tile[wave] + cl * LD + 64 * t + 16 * kk);
    }
    for (int p = 0; p < c.ZLW / 16; p++) {
        v4i32 d = {0, 0, 0, 0};
#pragma unroll
        for (int t = 0; t < KS; t++) {
            v4i32 v = {0, 0, 0, 0};
            if (64 * t + 16 * kk < N) v = *(const v4i32 *)(y.vl + (size_t)(16 * p + cl) * N + 64 * t + 16 * kk);
            d = __builtin_amdgcn_mfma_i32_16x16x64_i8(v, qv[t], d, 0, 0, 0);
        }
        uint32_t z = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float zf = (float)d[e] * y.mv[16 * p + 4 * kk + e];
            zf = zf * rm;
            z |= (uint32_t)(uint8_t)clamp127(cvt_rne(zf)) << (8 * e);
        }
        if (to < c.N) *(uint32_t *)(c.zl + (size_t)to * c.ZLW + 16 * p + 4 * kk) = z;
    }
}

// u of one tile of layer l: per 16 coordinates (rows of the matrix product) and 16 rows (its columns) U'_r zl, or first
// U_r v[x] with FACT; lane's coordinates are 16 b + 4 kk .. + 3 of rows lane % 16 and 16 + lane % 16 of the tile
// (cpu/ygg.cpp:311-377)
template <int N, bool FACT>
__device__ __forceinline__ void tile_input(const YggDevModel &m, const ScanChunk &c, int l, int4 tile, int lane) {
    const YggDevLayer &y = m.layers[l];
    const Sort &by = c.by[l & 1];
    const int r = tile.x, cnt = tile.z, cl = lane & 15, kk = lane >> 4, halves = cnt > 16 ? 2 : 1;
    const uint8_t *g = y.gath + (uint32_t)r * (uint32_t)y.gath_bytes;
    const int K4 = m.R2 / 4, F4 = m.K / 4;
    float fs = 0.0f;
    if constexpr (FACT) fs = *(const float *)(g + y.off_FS);
    int row[2], x[2];
    bool on[2];
    v4i32 z[2], vx[2];
    const int16_t *tr[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        on[h] = 16 * h + cl < cnt;
        row[h] = row_at(by, tile.y + (on[h] ? 16 * h + cl : 0));
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        x[h] = c.x[row[h]];
        z[h] = vx[h] = v4i32{0, 0, 0, 0};
        if (16 * kk < c.ZLW) z[h] = *(const v4i32 *)(c.zl + (size_t)row[h] * c.ZLW + 16 * kk);
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        if constexpr (FACT) {
            const uint32_t *v = (const uint32_t *)(y.vt + (size_t)x[h] * m.K);
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (4 * kk + e < F4) vx[h][e] = (int)v[4 * kk + e];
            tr[h] = (const int16_t *)(g + y.off_FB);
        } else {
            tr[h] = y.table + ((uint32_t)r * (uint32_t)y.table_sr + (uint32_t)x[h] * (uint32_t)y.table_sx);
        }
    }
#pragma unroll 4
    for (int b = 0; b < N / 16; b++) {
        const int i0 = 16 * b + 4 * kk;
        uint2 tw[2];
        tw[0] = *(const uint2 *)(tr[0] + i0);
        if (halves == 2) tw[1] = *(const uint2 *)(tr[1] + i0);
        v4i32 uw = {0, 0, 0, 0}, fw = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (4 * kk + e < K4) uw[e] = *(const int *)(g + y.off_U + ((4 * kk + e) * N + 16 * b + cl) * 4);
        if constexpr (FACT) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (4 * kk + e < F4) fw[e] = *(const int *)(g + y.off_F + ((4 * kk + e) * N + 16 * b + cl) * 4);
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h && halves == 1) break;
            const v4i32 d = __builtin_amdgcn_mfma_i32_16x16x64_i8(uw, z[h], v4i32{0, 0, 0, 0}, 0, 0, 0);
            v4i32 df = {0, 0, 0, 0};
            if constexpr (FACT) df = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw, vx[h], df, 0, 0, 0);
            uint32_t out[2];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t tv = e < 2 ? tw[h].x : tw[h].y;
                int in = (int)(int16_t)((e & 1) ? tv >> 16 : tv & 0xffff);
                if constexpr (FACT) {
                    const float fm = fs * y.mT[i0 + e];
                    in = wadd(cvt_rne((float)df[e] * fm), in);
                }
                const float scale = y.mulv ? y.mulv[i0 + e] : y.layer_input_scale;
                in = wadd(in, cvt_rne((float)d[e] * scale));
                in = in > 32767 ? 32767 : (in < -32768 ? -32768 : in);
                out[e / 2] = e & 1 ? (out[e / 2] & 0xffffu) | ((uint32_t)in << 16) : (uint32_t)in;
            }
            if (on[h]) *(uint2 *)(c.u + ((size_t)b * c.N + row[h]) * 16 + 4 * kk) = make_uint2(out[0], out[1]);
        }
    }
}

// zq of one tile of layer l (cpu/ygg.cpp:395-420), lane's ranks 16 t + 4 kk .. + 3 of row lane % 16 of the tile
template <int N>
__device__ __forceinline__ void tile_readout(const YggDevModel &m, const ScanChunk &c, int l, int4 tile, int lane) {
    constexpr int KS = (N + 63) / 64;
    const YggDevLayer &y = m.layers[l];
    const Sort &by = c.by[l & 1];
    const int r = tile.x, cnt = tile.z, cl = lane & 15, kk = lane >> 4, R = m.R;
    const int8_t *p = (const int8_t *)(y.gath + (uint32_t)r * (uint32_t)y.gath_bytes + y.off_P);
    const int RL = 64 / R, SP = N / RL, GP = SP % 16 == 0 ? 16 : (SP % 8 == 0 ? 8 : 4);    // the record's granules of P
    for (int h = 0; h < cnt; h += 16) {
        const bool on = h + cl < cnt;
        const int row = row_at(by, tile.y + (on ? h + cl : h));
        v4i32 qv[KS];
#pragma unroll
        for (int t = 0; t < KS; t++) {
            qv[t] = v4i32{0, 0, 0, 0};
            if (64 * t + 16 * kk < N) qv[t] = *(const v4i32 *)(c.qr + (size_t)row * N + 64 * t + 16 * kk);
        }
        for (int j0 = 0; j0 < R; j0 += 16) {
            v4i32 d = {0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < KS; t++) {
                const int i = 64 * t + 16 * kk, j = j0 + cl;
                v4i32 pv = {0, 0, 0, 0};
                if (i < N && j < R) {
                    if (GP == 16) {
                        pv = *(const v4i32 *)(p + ((i % SP / 16) * 64 + j * RL + i / SP) * 16);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const int ci = i + 4 * e;
                            pv[e] = *(const int *)(p + (ci % SP / GP * 64 + j * RL + ci / SP) * GP + ci % SP % GP);
                        }
                    }
                }
                d = __builtin_amdgcn_mfma_i32_16x16x64_i8(pv, qv[t], d, 0, 0, 0);
            }
            const int j = j0 + 4 * kk;
            if (on && j < R) {
                uint32_t z = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float scale = y.mz ? y.mz[(size_t)r * R + j + e] : y.readout_scale;
                    z |= (uint32_t)(uint8_t)clamp127(cvt_rne((float)d[e] * scale)) << (8 * e);
                }
                *(uint32_t *)(c.zq + (size_t)row * c.ZQW + l * R + j) = z;
            }
        }
    }
}

// wavefronts [0, inputs): u of layer l by its tiles; the others: zq of layer lz by that one's. A wavefront per tile.
template <int N, bool FACT>
__global__ __launch_bounds__(256) void s8_tiles(const YggDevModel m, const ScanChunk c, int l, int inputs, int lz,
                                                int readouts) {
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (w < inputs) {
        const int n = tiles_of(c.by[l & 1]);
        for (int i = w; i < n; i += inputs) {
            const int4 t = tile_at(c.by[l & 1], i);
            if (t.z) tile_input<N, FACT>(m, c, l, t, lane);
        }
    } else if (w - inputs < readouts) {
        const int n = tiles_of(c.by[lz & 1]);
        for (int i = w - inputs; i < n; i += readouts) {
            const int4 t = tile_at(c.by[lz & 1], i);
            if (t.z) tile_readout<N>(m, c, lz, t, lane);
        }
    }
}

// expert r's P (the lane's granules) and readout scale of the lane's row
template <class SH> __device__ __forceinline__ float load_readout(Gather<SH> &G, const YggDevLayer &y, int r, int lane) {
    const uint8_t *pp = y.gath + (uint32_t)r * (uint32_t)y.gath_bytes + y.off_P;
#pragma unroll
    for (int gi = 0; gi < SH::SP / SH::GP; gi++) {
        uint32_t tmp[SH::GP / 4];
        load_words<SH::GP / 4, SH::GP>(tmp, pp + (gi * 64 + lane) * SH::GP);
#pragma unroll
        for (int i = 0; i < SH::GP / 4; i++) G.pw[gi * (SH::GP / 4) + i] = tmp[i];
    }
    return y.mz ? y.mz[(uint32_t)r * SH::R + lane / SH::RL] : y.readout_scale;
}

// Row by row, for rows that are not sorted: a wavefront per row of layer l, in fast_kernel's lane mappings: the readout
// of the layer below (its expert's P loaded while the route runs), the route in rounds of up to 4 levels (3 or 4 dependent
// loads where s8_route's levels are 10 to 14), the layer input and u. A row's own weights are read once and nothing is
// shared, so it is bound by latency: 13 us with its launch for 1001 rows at n = 256, where s8_route and s8_tiles took 27.
template <class SH, bool GROUP, bool FACT>
__global__ __launch_bounds__(256) void s8_row(const YggDevModel m, const ScanChunk c, int l, int readout_below) {
    using F = SH;
    constexpr int N = SH::N, R = SH::R;
    __shared__ __attribute__((aligned(16))) int8_t qw[4][N], zw[4][SH::ZL], rw[4][SH::ZQ];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = blockIdx.x * 4 + wave;
    if (row >= c.N) return;
    const int x = __builtin_amdgcn_readfirstlane(c.x[row]);
    const YggDevLayer &y = m.layers[l], &yb = m.layers[l - 1];
    if (x < 0) {
        if (lane == 0) {
            c.by[l & 1].leaf[row] = -1;
            c.rec[row] = 0u;
        }
        return;
    }
    int8_t *q = qw[wave];
    if (lane < N / 16) *(uint4 *)(q + 16 * lane) = *(const uint4 *)(c.q + ((size_t)lane * c.N + row) * 16);
    const int rb = __builtin_amdgcn_readfirstlane(c.by[(l - 1) & 1].leaf[row]);
    Gather<SH> G;
    float scale = 0.0f;
    if (readout_below) scale = load_readout<SH>(G, yb, rb, lane);
    // the route's thresholds and V' need no state
    const int qk = lane & 3, qj = lane >> 2;
    uint32_t vr[SH::RG > 0 ? SH::RG : 1][Fast<N>::QW];
    load_vrows<SH>(vr, y, lane);
    wave_sync();
    uint32_t qbw[Fast<N>::QW];
    float rho;
    if constexpr (GROUP) {
        quad_share<N>(qbw, q, qk);
        rho = group_rho<N>(qbw, y.r2b, y.rms_eps);
    } else {
        rho = below_and_rho<N>(qbw, q, y.rms_eps, lane);
    }
    const float *thr = y.thr + (size_t)x * y.thr_stride;
    int ix = 1, base = 0, d0 = 0;
    for (int rd = 0; rd < m.n_rounds; rd++) {
        const int h = (m.round_pack >> (4 * rd)) & 15, nn = (1 << h) - 1, slot = base + ((ix - (1 << d0)) << h) + qj;
        uint32_t wv[Fast<N>::QW];
        float th = 0.0f;
        int dot = 0;
        if (qj < nn) {
            quad_share<N>(wv, y.w + (size_t)slot * N, qk);
            th = thr[slot];
#pragma unroll
            for (int i = 0; i < Fast<N>::QW; i++) dot = dot4(wv[i], qbw[i], dot);
        }
        dot = sum4(dot);
        const bool right = (float)dot * rho > th;
        ix = (ix << h) + (walk_round(lane_mask(right && qk == 0 && qj < nn), h) - nn);
        base += (1 << d0) << h;
        d0 += h;
    }
    const int r = ix - m.E;
    // u's weights, in flight while the readout below and the layer input are formed
    const uint8_t *g = y.gath + (uint32_t)r * (uint32_t)y.gath_bytes;
    const int K4 = FACT ? m.K / 4 : 0, ln = lane < F::NL ? lane : F::NL - 1;
    uint32_t uw[SH::K4A][SH::C], fw[FACT ? kFactK4 : 1][SH::C];
    load_uw<SH>(uw, y, r, lane);
    int in[SH::C];
    const int16_t *tr = FACT ? (const int16_t *)(g + y.off_FB)
                             : y.table + ((uint32_t)r * (uint32_t)y.table_sr + (uint32_t)x * (uint32_t)y.table_sx);
#pragma unroll
    for (int e = 0; e < SH::C; e++) in[e] = tr[F::C * ln + e];
    float fs = 0.0f;
    if constexpr (FACT) {
        fs = *(const float *)(g + y.off_FS);
#pragma unroll
        for (int k4 = 0; k4 < kFactK4; k4++)
#pragma unroll
            for (int e = 0; e < SH::C; e++)
                fw[k4][e] = k4 < K4 ? *(const uint32_t *)(g + y.off_F + ((k4 * F::NL + ln) * F::C + e) * 4) : 0u;
    }
    layer_input_regs<SH>(zw[wave], vr, y.mv, qbw, rho, lane);
    if (readout_below) {
        readout<SH>(rw[wave], G.pw, q, scale, lane);
        wave_sync();
        if (lane < R / 4) ((uint32_t *)(c.zq + (size_t)row * c.ZQW + (l - 1) * R))[lane] = ((const uint32_t *)rw[wave])[lane];
    } else {
        wave_sync();
    }
    int d[SH::C];
    uw_products<SH>(d, uw, zw[wave]);
    if constexpr (FACT) {
        const uint32_t *vx = (const uint32_t *)(y.vt + (size_t)x * m.K);
#pragma unroll
        for (int e = 0; e < SH::C; e++) {
            int df = 0;
#pragma unroll
            for (int k4 = 0; k4 < kFactK4; k4++)
                if (k4 < K4) df = dot4(fw[k4][e], vx[k4], df);
            const float fm = fs * y.mT[F::C * ln + e];
            in[e] = wadd(cvt_rne((float)df * fm), in[e]);
        }
    }
    if (lane < F::NL) {
        int16_t *to = c.u + ((size_t)(F::C * lane / 16) * c.N + row) * 16 + F::C * lane % 16;
#pragma unroll
        for (int e = 0; e < SH::C; e++) {
            const float sc = y.mulv ? y.mulv[F::C * lane + e] : y.layer_input_scale;
            const int v = wadd(in[e], cvt_rne((float)d[e] * sc));
            to[e] = (int16_t)(v > 32767 ? 32767 : (v < -32768 ? -32768 : v));
        }
    }
    if (lane == 0) {
        c.by[l & 1].leaf[row] = r;
        c.rec[row] = (uint32_t)r * (uint32_t)y.gath_bytes;
        if (c.io.leaves) c.io.leaves[c.token_at(row) * m.L + l] = r;
    }
}

// the last layer's readouts, a wavefront per row
template <class SH> __global__ __launch_bounds__(256) void s8_last(const YggDevModel m, const ScanChunk c) {
    constexpr int N = SH::N, R = SH::R;
    __shared__ __attribute__((aligned(16))) int8_t qw[4][N], rw[4][SH::ZQ];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = m.L - 1;
    const int row = blockIdx.x * 4 + wave;
    if (row >= c.N) return;
    const int r = __builtin_amdgcn_readfirstlane(c.by[l & 1].leaf[row]);
    if (r < 0) return;
    if (lane < N / 16) *(uint4 *)(qw[wave] + 16 * lane) = *(const uint4 *)(c.q + ((size_t)lane * c.N + row) * 16);
    Gather<SH> G;
    const float scale = load_readout<SH>(G, m.layers[l], r, lane);
    wave_sync();
    readout<SH>(rw[wave], G.pw, qw[wave], scale, lane);
    wave_sync();
    if (lane < R / 4) ((uint32_t *)(c.zq + (size_t)row * c.ZQW + l * R))[lane] = ((const uint32_t *)rw[wave])[lane];
}

// The recurrence of layer l: 16 lanes per stream and block of 16 coordinates, lane i row i, four streams of one block per
// wavefront (past the last stream its duplicates, whose equal stores change nothing); the A16 rows and inputs of the next
// PD tokens loaded ahead and the records' offsets PD further. Every lane holds the block's 16 state bytes (qv). One
// wavefront on a SIMD issues an instruction every 4 cycles, so a step is kept to about 25: two chains of four dot4, the
// saturation, the exchange of the new bytes (a byte permute to the lane's place, two ORs over the quad, four row
// broadcasts), four loads at immediate offsets and a byte store. Loads run past a stream's end without a look (the rows
// behind it, or kPad more): what they bring is never used. Layer 0 (L0) takes its inputs from the token's table row.
// PD 16 for few wavefronts, whose loads nothing else hides: one stream of 1001 tokens at n = 256 took 122 us per layer
// with 8 ahead and 70 instructions a step.
template <int N, int PD, bool L0>
__global__ __launch_bounds__(64) void s8_scan(const YggDevModel m, const ScanChunk c, int l) {
    using F = Fast<N>;
    constexpr int NB = N / 16;
    const YggDevLayer &y = m.layers[l];
    const int g = blockIdx.x % NB, lane = threadIdx.x & 63, i = lane & 15, ci = 16 * g + i;
    const int sw = blockIdx.x / NB * 4 + (lane >> 4), s = sw < c.Bc ? sw : c.Bc - 1;
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
    int8_t *st = c.state + ((size_t)(c.s0 + s) * m.L + l) * N + ci;
    const size_t row0 = (size_t)s * c.Tc;
    const uint32_t *rec = c.rec + row0;
    const int *xs = c.x + row0;
    const int16_t *us = c.u + ((size_t)g * c.N + row0) * 16 + i;
    int8_t *qs = c.q + ((size_t)g * c.N + row0) * 16 + i;
    // the row's 16 hi and 16 lo bytes in a record (ygg_layout.h)
    const uint32_t part = (2 * (ci % F::C) * F::NL + ci / F::C) * 16;
    const int half = 1 << (m.shift - 1), shift = m.shift;
    const uint32_t place = 0x0c0c0c0cu & ~(0xffu << (8 * (i & 3)));     // byte 0 to byte i % 4, zeros elsewhere
    int qo = *st;
    // with many wavefronts the stores are the states of 16 tokens at once, 16 bytes a lane
    constexpr bool WIDE = PD == 8;
    uint32_t qv[4], out[4] = {0u, 0u, 0u, 0u};
    auto exchange = [&]() {
        int w = (int)__builtin_amdgcn_perm(0u, (uint32_t)qo, place);
        w |= __builtin_amdgcn_update_dpp(0, w, 0xB1, 0xF, 0xF, true);
        w |= __builtin_amdgcn_update_dpp(0, w, 0x4E, 0xF, 0xF, true);
        qv[0] = __builtin_amdgcn_update_dpp(0, w, 0x150, 0xF, 0xF, true);
        qv[1] = __builtin_amdgcn_update_dpp(0, w, 0x154, 0xF, 0xF, true);
        qv[2] = __builtin_amdgcn_update_dpp(0, w, 0x158, 0xF, 0xF, true);
        qv[3] = __builtin_amdgcn_update_dpp(0, w, 0x15C, 0xF, 0xF, true);
    };
    exchange();
    uint4 hi[PD], lo[PD];
    int u[PD], xt[L0 ? PD : 1];
    uint32_t ro[PD];
    auto fetch = [&](int k, int d) {       // the token d rows on, whose record's offset is in ro[k], into slot k
        // (the offset is used here and no earlier: hoisted, its use waits for every load up to its own, PD tokens early)
        if constexpr (L0) asm volatile("" : "+v"(ro[k]), "+v"(xt[k]));
        else asm volatile("" : "+v"(ro[k]));
        const uint8_t *a = y.gath + (ro[k] + part);
        hi[k] = *(const uint4 *)a;
        lo[k] = *(const uint4 *)(a + F::NL * 16);
        if constexpr (L0) u[k] = y.table[(uint32_t)((xt[k] < 0 ? 0 : xt[k]) * N + ci)];
        else u[k] = us[d * 16];
    };
    auto offset = [&](int k, int d) {
        ro[k] = rec[d];
        if constexpr (L0) xt[k] = xs[d];
    };
#pragma unroll
    for (int k = 0; k < PD; k++) offset(k, k);
    // (in the loop's order: the waits at its top are those of the worse of the two ways in)
#pragma unroll
    for (int k = 0; k < PD; k++) {
        fetch(k, k);
        offset(k, PD + k);
    }
    auto run16 = [&](auto tail, int left) {
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int k = j % PD;
            int ah = dot4(hi[k].x, qv[0], 0), al = dot4(lo[k].x, qv[0], half);
            ah = dot4(hi[k].y, qv[1], ah);
            al = dot4(lo[k].y, qv[1], al);
            ah = dot4(hi[k].z, qv[2], ah);
            al = dot4(lo[k].z, qv[2], al);
            ah = dot4(hi[k].w, qv[3], ah);
            al = dot4(lo[k].w, qv[3], al);
            const int qn = sat8(((int)(((uint32_t)ah << 8) + (uint32_t)al) >> shift) + u[k]);
            qo = !decltype(tail)::value || j < left ? qn : qo;
            if (!WIDE && (!decltype(tail)::value || j < left)) qs[j * 16] = (int8_t)qn;
            exchange();
            if (WIDE && i == j)
#pragma unroll
                for (int e = 0; e < 4; e++) out[e] = qv[e];
            fetch(k, j + PD);
            offset(k, j + 2 * PD);
        }
        // lane i holds the states after token i
        if (WIDE && i < left) *(uint4 *)(qs + i * 15) = make_uint4(out[0], out[1], out[2], out[3]);
        rec += 16;
        if constexpr (L0) xs += 16;
        us += 256;
        qs += 256;
    };
    int t0 = 0;
    for (; t0 + 16 <= least; t0 += 16) run16(std::false_type(), 16);
    for (; t0 < most; t0 += 16) run16(std::true_type(), len - t0);
    *st = (int8_t)qo;
}

// the current layer's states row by row (a thread per 16 bytes)
template <int N> __global__ __launch_bounds__(256) void s8_rows(const ScanChunk c) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    constexpr int NB = N / 16;
    const size_t row = i / NB, b = i % NB;
    if (row < (size_t)c.N) *(uint4 *)(c.qr + row * N + b * 16) = *(const uint4 *)(c.q + (b * c.N + row) * 16);
}

// The logits (cpu/ygg.cpp:421-435, in layer order): 16 rows per workgroup, a wavefront per 64 classes; per layer and 16
// classes an int8 matrix product of Q with the rows' zq, Q held in registers over the workgroup's tiles. Lane's classes are
// 16 t + 4 kk .. + 3 of its wavefront's 64, of row lane % 16. SCORE: the rows' NLL terms instead (token_nll's), a wavefront
// per 4 rows, from LDS. SQ: per-class scales.
template <int R, int L, bool SCORE, bool SQ>
__global__ __launch_bounds__(256) void s8_logits(const YggDevModel m, const ScanChunk c) {
    __shared__ float lgs[SCORE ? 16 : 1][SCORE ? 260 : 1];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), V = m.V;
    const int cl = lane & 15, kk = lane >> 4, c0 = 64 * wave;
    long Q[L][4];
    float bias[4][4], sq[SQ ? L : 1][4][4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
#pragma unroll
        for (int l = 0; l < L; l++) {
            const int row = c0 + 16 * t + cl;
            Q[l][t] = row < m.VP && 8 * kk < R ? *(const long *)(m.layers[l].Q + (size_t)row * R + 8 * kk) : 0;
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int cls = c0 + 16 * t + 4 * kk + e;
            bias[t][e] = cls < m.VP ? m.output_bias[cls] : 0.0f;
            if constexpr (SQ)
#pragma unroll
                for (int l = 0; l < L; l++)
                    sq[l][t][e] = cls >= m.VP ? 0.0f : (m.layers[l].sqv ? m.layers[l].sqv[cls] : m.layers[l].unembed_scale);
        }
    }
    for (int r0 = blockIdx.x * 16; r0 < c.N; r0 += gridDim.x * 16) {
        const int row = r0 + cl < c.N ? r0 + cl : c.N - 1;
        const bool live = r0 + cl < c.N && c.x[row] >= 0;
        const int8_t *zq = c.zq + (size_t)row * c.ZQW + 8 * kk;
        long z[L];
#pragma unroll
        for (int l = 0; l < L; l++) z[l] = 8 * kk < R ? *(const long *)(zq + l * R) : 0;
        float *out = SCORE ? nullptr : c.io.logits + c.token_at(row) * V;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            float lg[4];
#pragma unroll
            for (int e = 0; e < 4; e++) lg[e] = bias[t][e];
#pragma unroll
            for (int l = 0; l < L; l++) {
                const v4i32 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(Q[l][t], z[l], v4i32{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; e++) lg[e] = lg[e] + (float)d[e] * (SQ ? sq[SQ ? l : 0][t][e] : m.layers[l].unembed_scale);
            }
            const int cls = c0 + 16 * t + 4 * kk;
            if constexpr (SCORE) {
#pragma unroll
                for (int e = 0; e < 4; e++) lgs[cl][cls + e] = lg[e];
            } else if (live && cls < V) {
                if ((V & 3) == 0) {
                    *(float4 *)(out + cls) = make_float4(lg[0], lg[1], lg[2], lg[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (cls + e < V) out[cls + e] = lg[e];
                }
            }
        }
        if constexpr (SCORE) {
            __syncthreads();
            for (int k = 4 * wave; k < 4 * wave + 4 && r0 + k < c.N; k++) {
                double se = 0.0, lin = 0.0;
                if (__builtin_amdgcn_readfirstlane(c.x[r0 + k]) >= 0) {
                    const int y = __builtin_amdgcn_readfirstlane(c.io.targets[c.token_at(r0 + k)]);
                    float lg[4];
                    load_words<4, 16>((uint32_t(&)[4])lg, &lgs[k][4 * lane]);
                    if (y >= 0 && y < V) nll_terms(se, lin, lg, V, y, lane);
                    else if (lane == 0) atomicOr(m.err, 2u);
                }
                if (lane == 0) c.terms[r0 + k] = make_double2(se, lin);
            }
            __syncthreads();
        }
    }
}

// The same for at most 32 classes: a thread per row. Its sum of exponentials pairs the classes as nll_terms' lanes do:
// four classes in order per lane, then lanes 4, 2 and 1 apart (the lanes past the classes add zeros).
template <int R, int L, bool SCORE>
__global__ __launch_bounds__(256) void s8_logits_few(const YggDevModel m, const ScanChunk c) {
    constexpr int RW = R / 4, MV = 32;
    const int row = blockIdx.x * 256 + threadIdx.x, V = m.V;
    if (row >= c.N) return;
    if (c.x[row] < 0) {
        if (SCORE) c.terms[row] = make_double2(0.0, 0.0);
        return;
    }
    uint32_t zw[L * RW];
    load_words<L * RW, 8>(zw, c.zq + (size_t)row * c.ZQW);
    const size_t at = c.token_at(row);
    int y = SCORE ? c.io.targets[at] : 0;
    float lg[SCORE ? MV : 1], mx = -__builtin_huge_valf(), ly = 0.0f;
#pragma unroll
    for (int k = 0; k < MV; k++) {
        if (k < V) {
            float v = m.output_bias[k];
#pragma unroll
            for (int l = 0; l < L; l++) {
                const YggDevLayer &w = m.layers[l];
                int d = 0;
#pragma unroll
                for (int i = 0; i < RW; i++) d = dot4(*(const uint32_t *)(w.Q + k * R + 4 * i), zw[l * RW + i], d);
                v = v + (float)d * (w.sqv ? w.sqv[k] : w.unembed_scale);
            }
            if constexpr (SCORE) {
                lg[k] = v;
                mx = fmaxf(mx, v);
                ly = k == y ? v : ly;
            } else {
                c.io.logits[at * V + k] = v;
            }
        }
    }
    if constexpr (SCORE) {
        if (y < 0 || y >= V) {
            atomicOr(m.err, 2u);
            c.terms[row] = make_double2(0.0, 0.0);
            return;
        }
        ConstF64 e = (ConstF64)kExpNeg;
        asm volatile("" : "+s"(e));
        double s[MV / 4];
#pragma unroll
        for (int j = 0; j < MV / 4; j++) {
            s[j] = 0.0;
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (4 * j + u < V) s[j] += exp_neg((double)lg[4 * j + u] - (double)mx, e);
        }
        const double se = ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));
        c.terms[row] = make_double2(se, (double)mx - (double)ly);
    }
}

// A thread per stream: its rows' terms in order into its NLL (NllSum's additions), and at the call's end the NLL
__global__ __launch_bounds__(64) void s8_nll(const ScanChunk c) {
    const int s = blockIdx.x * 64 + threadIdx.x;
    if (s >= c.Bc) return;
    const double4 was = c.t0 ? c.sums[s] : make_double4(0.0, 1.0, 0.0, 0.0);
    double lin = was.x, pm = was.y;
    int pe = (int)was.z;
    const double2 *terms = c.terms + (size_t)s * c.Tc;
    const int len = c.len(s);
    for (int t0 = 0; t0 < len; t0 += 8) {
        double2 v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = terms[t0 + k < len ? t0 + k : len - 1];
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (t0 + k < len && v[k].x != 0.0) {
                lin = lin + v[k].y;
                int e;
                pm = frexp(pm * v[k].x, &e);
                pe += e;
            }
    }
    if (c.t0 + c.Tc >= c.Tn) {
        NllSum sum;
        sum.lin = lin, sum.pm = pm, sum.pe = pe;
        c.io.nll[c.s0 + s] += sum.value();
    } else {
        c.sums[s] = make_double4(lin, pm, (double)pe, 0.0);
    }
}

// ------------------------------------------------------------------------------------------------------ host side
// Are a chunk's N rows sorted? A sort costs about 28 us a layer and saves the experts' second reading: per row and layer
// 0.25 + 0.14 K against 0.1 + 0.085 K ns, K the KiB of the row's A16, U', U_r and P. Measured break-even: the small,
// medium and large trained shapes at 65k, 50k and 11k rows of 1024 experts, the medium one factored 16k, configuration
// 3's model (8192 experts) 100k, configuration 4's (16384) 300k.
bool sort_pays(const YggDevModel &m, int64_t N) {
    const int64_t E = std::max(m.E, m.V), w = (int64_t)m.N * (m.R + m.R2 + m.K);
    return E <= kSortLeaves && N >= 12 * E && N * std::max<int64_t>(w, 4096) >= 240000000;
}

struct ScanPlan {
    int64_t fixed, per_row;      // workspace bytes besides the rows' and the sorts', and per row (arrays rounded up apart)
    int E, ZLW, ZQW;
};

ScanPlan scan_plan(const YggDevModel &m, int64_t B, bool score) {
    ScanPlan p{};
    p.E = m.E > m.V ? m.E : m.V;
    p.ZLW = (m.R2 + 15) / 16 * 16;
    p.ZQW = m.L * m.R;
    p.per_row = 4 * (int64_t)m.N + p.ZLW + p.ZQW + 8 + 2 * kSortRowBytes + (score ? 16 : 0);
    p.fixed = 256 * 12 + B * 4 + (score ? B * 32 : 0) + kPad * (8 + 32);
    return p;
}
// workspace bytes of a chunk of N rows, more for more rows
int64_t scan_bytes(const YggDevModel &m, const ScanPlan &p, int64_t N, bool sort) {
    return p.fixed + p.per_row * N + 2 * sort_fixed_bytes(N, p.E, sort || sort_pays(m, N));
}

template <int N, int R, int R2>
void scan_layers(const YggDevModel &m, const ScanChunk &c, bool group, bool sorted, hipStream_t st) {
    using SH = Shape<N, R, R2>;
    const bool fact = m.layers[1].vt != nullptr;
    auto scan = [&](int l) {
        const int waves = (c.Bc + 3) / 4 * (N / 16);
        auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(waves), dim3(64), 0, st, m, c, l); };
        // (at most two wavefronts per SIMD: the registers of 16 tokens ahead cost no residency)
        if (waves <= 2048) l ? go(s8_scan<N, 16, false>) : go(s8_scan<N, 16, true>);
        else l ? go(s8_scan<N, 8, false>) : go(s8_scan<N, 8, true>);
    };
    auto tiles = [&](int l, bool in, int lz, bool rd) {
        auto waves = [&](const Sort &s) { return std::min(s.max_tiles, 16384); };
        const int a = in ? (waves(c.by[l & 1]) + 3) / 4 * 4 : 0, b = rd ? waves(c.by[lz & 1]) : 0;
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((a + b + 3) / 4), dim3(256), 0, st, m, c, l, a, lz, b);
        };
        if (fact) go(s8_tiles<N, true>);
        else go(s8_tiles<N, false>);
    };
    const bool read = c.io.logits || c.io.nll;
    hipLaunchKernelGGL(s8_begin, dim3(c.Bc), dim3(256), 0, st, m, c);
    scan(0);
    if (!sorted) {
        const dim3 grid((c.N + 3) / 4);
        for (int l = 1; l < m.L; l++) {
            auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, m, c, l, (int)read); };
            if constexpr (N != 96) {
                if (group) fact ? go(s8_row<SH, true, true>) : go(s8_row<SH, true, false>);
                else fact ? go(s8_row<SH, false, true>) : go(s8_row<SH, false, false>);
            } else {
                fact ? go(s8_row<SH, false, true>) : go(s8_row<SH, false, false>);
            }
            scan(l);
        }
        if (read) hipLaunchKernelGGL(s8_last<SH>, grid, dim3(256), 0, st, m, c);
        return;
    }
    for (int l = 1; l < m.L; l++) {
        const dim3 grid((c.N + 63) / 64);
        if constexpr (N != 96) {
            if (group) hipLaunchKernelGGL((s8_route<N, true>), grid, dim3(256), 0, st, m, c, l);
            else hipLaunchKernelGGL((s8_route<N, false>), grid, dim3(256), 0, st, m, c, l);
        } else {
            hipLaunchKernelGGL((s8_route<N, false>), grid, dim3(256), 0, st, m, c, l);
        }
        launch_sort(c.by[l & 1], c.by[0], l == 1 && read, st);
        tiles(l, true, l - 1, read);
        scan(l);
    }
    if (read) {
        hipLaunchKernelGGL(s8_rows<N>, dim3((unsigned)(((int64_t)c.N * (N / 16) + 255) / 256)), dim3(256), 0, st, c);
        tiles(0, false, m.L - 1, true);
    }
}

template <int R, int L> void scan_logits(const YggDevModel &m, const ScanChunk &c, hipStream_t st) {
    auto go = [&](auto kernel, int grid) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, st, m, c); };
    if (m.V <= 32) {
        const int grid = (c.N + 255) / 256;
        c.io.nll ? go(s8_logits_few<R, L, true>, grid) : go(s8_logits_few<R, L, false>, grid);
        return;
    }
    bool sq = false;
    for (int l = 0; l < L; l++) sq = sq || m.layers[l].sqv;
    const int grid = std::min((c.N + 15) / 16, 2048);
    if (c.io.nll) sq ? go(s8_logits<R, L, true, true>, grid) : go(s8_logits<R, L, true, false>, grid);
    else sq ? go(s8_logits<R, L, false, true>, grid) : go(s8_logits<R, L, false, false>, grid);
}

template <int R> void scan_logits_of(const YggDevModel &m, const ScanChunk &c, hipStream_t st) {
    if (m.L == 2) scan_logits<R, 2>(m, c, st);
    else if (m.L == 3) scan_logits<R, 3>(m, c, st);
    else if (m.L == 4) scan_logits<R, 4>(m, c, st);
    else scan_logits<R, 5>(m, c, st);
}

}  // namespace

bool scan_pays(const YggDevModel &m, int64_t B, int64_t T, ScanCall call, TokenKernel token) {
    // K: KiB of an expert's A16, U', U_r and P; hot: a layer's of these fit an XCD's L2
    const double L = m.L, P = m.n_rounds, N = (double)B * T, n = m.N, K = n * (32 + m.R + m.R2 + m.K) / 1024;
    const double score = call == ScanCall::score, out = call != ScanCall::state;
    const bool hot = m.E * K <= 4096;
    // token by token: a stream's tokens one after the other while the streams do not fill the chip, then all rows
    double alone, rows;
    if (m.K) {
        alone = L * (1.3 + T * (0.52 + 0.086 * K + 0.51 * P + 0.43 * score));
        rows = 1e-3 * N * L * ((hot ? 0.088 : 0.137) * K + 0.09 * score);
    } else if (token == TokenKernel::flow) {
        const double whole = !flow_split_build(m.N, m.R, m.R2, m.L, call == ScanCall::score ? kModeScore : kModeRun);
        alone = 5.1 * L + T * (0.52 + 0.62 * whole + 0.0086 * L * K + 0.52 * score);
        rows = 1e-3 * N * L * ((hot ? 0.12 : 0.095) * K + 0.35 + 0.55 * whole + 0.5 * score);
        alone *= alone, rows *= rows;      // (few calls between the two: nearer their maximum than the others)
    } else if (token == TokenKernel::pipe) {
        alone = L * (1.6 + 0.24 * P) + T * (0.8 + 0.31 * P + 0.019 * L * K + 1.2 * score);
        rows = 3.3 + 1e-3 * N * L * ((hot ? 0.034 : 0.053) * K + 0.134 * P + 0.23 * score);
    } else {
        alone = L * (2.1 + T * (0.74 + 0.0069 * K + 0.27 * P + 0.27 * score));
        rows = 1e-3 * N * L * ((hot ? 0.052 : 0.1) * K + 0.18 * score);
    }
    double by_token = std::hypot(alone, rows);
    if (!m.K && token == TokenKernel::flow) by_token = std::sqrt(by_token);
    // layer by layer: the launches, the recurrence's steps (whole runs of 16 tokens), its loads past each stream's end, the
    // rows (past 4 MB of A16 an XCD's blocks outgrow its L2), the logits or the NLL
    const double steps = (T + 15) / 16 * 16;
    double scan = 3.3e-7 * B * L * n * n;
    if (sort_pays(m, B * T)) {
        const double E = std::max(m.E, m.V), miss = (double)m.E * n * 4 > 6e6 ? 2.5 : 1.0;
        scan += L * (18.6 + 0.057 * steps + 0.0022 * E) + 1e-3 * N * ((L - 1) * 0.037 * K + 2.1e-3 * L * n * miss);
        scan += out * (10.6 + N * (7e-5 + 1.4e-6 * m.V)) + score * (13 + 0.06 * T + 1.7e-4 * N);
    } else {
        scan += L * (8.5 + steps * (0.046 + 0.00016 * n)) + 1e-3 * N * (L - 1) * 0.145 * K;
        scan += out * (9 + 2.1e-6 * N * m.V) + score * (5.5 + 0.054 * T + 2.4e-4 * N);
    }
    return scan < by_token;
}

int64_t scan_scratch_bytes(const YggDevModel &m, int64_t B, int64_t T, bool score, bool sort, int64_t cap) {
    const ScanPlan p = scan_plan(m, B, score);
    cap = std::max(cap, scan_bytes(m, p, 64, sort));
    return (int64_t)up256((size_t)std::min(scan_bytes(m, p, B * T, sort), cap));
}

hipError_t launch_scan(const YggDevModel &m, const int32_t *tokens, int B, int T, int8_t *state, const YggIO &io,
                       bool group, bool sort, void *ws, int64_t bytes, hipStream_t st) {
    const bool score = io.nll != nullptr;
    const ScanPlan p = scan_plan(m, B, score);
    // a chunk's rows; whole calls where they fit, else runs of at least 128 tokens of as many streams as fit
    const int64_t rows = rows_that_fit((int64_t)B * T, bytes, [&](int64_t N) { return scan_bytes(m, p, N, sort); });
    if (rows < 1) return hipErrorInvalidValue;
    int64_t Tc = T, Bc = B;
    if ((int64_t)B * T > rows) {
        Tc = std::min<int64_t>(std::min<int64_t>(std::max<int64_t>(rows / B, 128), T), rows);
        Bc = std::min<int64_t>(rows / Tc, B);
    }
    for (int s0 = 0; s0 < B; s0 += (int)Bc)
        for (int t0 = 0; t0 < T; t0 += (int)Tc) {
            ScanChunk c{};
            c.tokens = tokens;
            c.Tn = T;
            c.s0 = s0;
            c.Bc = (int)std::min<int64_t>(B - s0, Bc);
            c.t0 = t0;
            c.Tc = (int)std::min<int64_t>(T - t0, Tc);
            c.N = c.Bc * c.Tc;
            c.ZLW = p.ZLW;
            c.ZQW = p.ZQW;
            c.state = state;
            c.io = io;
            const bool sorted = sort || sort_pays(m, c.N);
            uint8_t *w = (uint8_t *)ws;
            auto take = [&](size_t k) {
                uint8_t *q = w;
                w += up256(k);
                return q;
            };
            const size_t N = (size_t)c.N;
            c.stop = (int *)take((size_t)B * 4);
            if (score) c.sums = (double4 *)take((size_t)B * 32);
            for (int k = 0; k < 2; k++) lay_out(c.by[k], c.N, p.E, sorted, take);
            if (score) c.terms = (double2 *)take(N * 16);
            c.x = (int *)take((N + kPad) * 4);
            c.rec = (uint32_t *)take((N + kPad) * 4);
            c.zl = (int8_t *)take(N * p.ZLW);
            c.zq = (int8_t *)take(N * p.ZQW);
            c.qr = (int8_t *)take(N * m.N);
            c.q = (int8_t *)take(N * m.N);
            c.u = (int16_t *)take(N * m.N * 2 + kPad * 32);
            if (w - (uint8_t *)ws > bytes) return hipErrorInvalidValue;
#define YGG_S(N_, R_, R2_) \
            if (m.N == N_ && m.R == R_ && m.R2 == R2_) scan_layers<N_, R_, R2_>(m, c, group, sorted, st);
            YGG_SHAPES(YGG_S)
#undef YGG_S
            if (io.logits || score) {
                if (m.R == 8) scan_logits_of<8>(m, c, st);
                else if (m.R == 16) scan_logits_of<16>(m, c, st);
                else scan_logits_of<32>(m, c, st);
                if (score) hipLaunchKernelGGL(s8_nll, dim3((c.Bc + 63) / 64), dim3(64), 0, st, c);
            }
        }
    return hipGetLastError();
}

}  // namespace ygg
