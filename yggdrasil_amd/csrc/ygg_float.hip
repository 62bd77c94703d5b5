// The float step of Yggdrasil (yggdrasil/inference.py:42-74): the inference model of a float checkpoint, in f32 for
// serving (the role of the Triton backend, yggdrasil/inference_triton.py) or f64 (the precision cpu/export.py
// calibrates in, cpu/export.py:101-153). One workgroup of 256 threads runs one stream through every layer of every
// token of a launch; the states of all layers stay in LDS.
//
// Per token x and layer l (expert r = x in the token layer, else the router's leaf):
//   route:   node = 1 .. 2^D - 1 (heap), right iff [router_embed[x]; rms(h_below)] . W[node] + b[node] > 0
//   update:  h = T_r[x];  h += U'_r (V' rms(h_below));  h += A_r h_old   (A_r block-diagonal)
//   readout: z = P_r h;   logits += Q z
// and rms(h) = h / sqrt(mean(h^2) + 1e-6) feeds the next layer.
// Work split: the router descends in rounds of up to 4 levels, 16 groups of 16 threads each forming one node's dot of
// the round's subtree (every load of a round issued at once, the input row held in registers for the layer); for the
// layer input wavefront q sums its quarter of the coordinates for row k = lane of V'; thread i owns coordinate i of
// the update (its table entry, U' column and A row loaded together); the readout takes 256 / R threads per row of P;
// thread c owns class c of the logits. The reference's trained shapes have f32 builds of their own (float_step).
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "ygg_float.h"

using namespace ygg::flt;

namespace {

constexpr int kFThreads = 256;

template <typename T> __device__ __forceinline__ T wave_sum(T v) {
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

template <typename T> __device__ __forceinline__ T wave_max(T v) {
    for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}

// the sum over aligned groups of G lanes (G a power of 2, at most 64), in every lane of the group
template <int G, typename T> __device__ __forceinline__ T group_sum(T v) {
    for (int o = G / 2; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
template <typename T> __device__ __forceinline__ T group_sum_n(T v, int g) {
    for (int o = g / 2; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
template <typename T> __device__ __forceinline__ T group_max_n(T v, int g) {
    for (int o = g / 2; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}

// atomic max of a non-negative double (its bit pattern orders as an unsigned integer)
__device__ __forceinline__ void atomic_max_nonneg(double *p, double v) {
    atomicMax((unsigned long long *)p, (unsigned long long)__double_as_longlong(v));
}

// the sum of v over the workgroup (red: 4 slots of LDS; two barriers)
template <typename T> __device__ __forceinline__ T block_sum(T v, T *red, int tid) {
    v = wave_sum(v);
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    const T s = (red[0] + red[1]) + (red[2] + red[3]);
    __syncthreads();
    return s;
}

constexpr int kRouteGroup = 16;                           // threads per node of a router round
constexpr int kRouteElems = (kMaxF + kMaxN) / kRouteGroup; // router inputs per thread at most

// The f32 step of the reference's trained shapes: 4 N threads per stream (its 1024 threads at n = 256 are a CU's), so that
// a layer's loads are many threads' and short. Per layer, for G = 32 lanes a node at n = 256, 16 at 128, 8 at 64:
//   route    rounds of 5 levels, the 31 nodes of a subtree on G lanes each; a round's decisions are bits of one LDS word
//   V' h     thread (k, part): row k over a sixteenth of the coordinates; the parts are summed after the first round
//   update   thread (i, quarter): a quarter of coordinate i's U' and A terms; the quarters are summed by thread i
//   readout  32 lanes per row of P; logits: thread (class, part) 8 ranks of the class, its parts summed once per token
// The next layer's V', first round and token part are loaded behind the current one's update, so a layer waits for two
// dependent loads, its second round and its expert's record, and meets five barriers: latency bounds it until the streams
// fill the chip. Depth 10, 5 layers, 4 tokens of 1 / 16 / 256 / 1024 streams (us; before, on 256 threads with three rounds
// of 4 levels and 13 barriers a layer): n = 64 54 / 55 / 58 / 71 (132 / 134 / 135 / 531), n = 128 57 / 58 / 76 / 152
// (148 / 151 / 161 / 629), n = 256 87 / 93 / 121 / 455 (189 / 193 / 219 / 837).
template <int G> __device__ __forceinline__ float lanes_sum(float v) {
    auto move = [&](auto ctrl) {
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), decltype(ctrl)::value, 0xf, 0xf, true));
    };
    v += move(std::integral_constant<int, 0xB1>());      // quad_perm 1 0 3 2
    v += move(std::integral_constant<int, 0x4E>());      // quad_perm 2 3 0 1
    if constexpr (G >= 8) v += move(std::integral_constant<int, 0x141>());     // row_half_mirror
    if constexpr (G >= 16) v += move(std::integral_constant<int, 0x140>());    // row_mirror
    if constexpr (G >= 32) v += __shfl_xor(v, 16);
    return v;
}

// base[i], its offset in 32 bits beside a uniform base (a 64-bit address per thread and array does not fit the registers)
__device__ __forceinline__ const float *from(const float *base, uint32_t i) {
    return (const float *)((const char *)base + i * 4u);
}

// The step. ANY: models of these sizes with a token part past kStepF entries (the rest loaded where it is added) or without
// transitions, and calls with the calibration maxima, kept in LDS by the threads that form the values. A build of its own:
// the plain one keeps its registers. One token of one stream, n = 64 / 128 / 256 (us; the plain build 16 / 17 / 22, the
// general kernel 110 to 130): a token part of 64 20 / 20 / 25, no transitions 17 / 18 / 23, with the maxima 21 / 21 / 27; of
// 256 streams 21 / 24 / 34, 18 / 20 / 31 and 40 / 41 / 47, these last bound by the maxima's additions in memory.
template <int N, int R, int R2, bool ANY>
__device__ __forceinline__ void float_step(const FloatDevModel<float> &m, const int32_t *__restrict__ tokens, int Tn,
                                           float *__restrict__ state, float *__restrict__ logits,
                                           int32_t *__restrict__ leaves, double *__restrict__ stats) {
    constexpr int NT = 4 * N, G = N / 8, PARTS = NT / R2, VC = N / PARTS, UK = R2 / 4,
                  PL = 32, PE = N / PL, FE = kStepF / G, QP = NT / 256, RQ = R / QP;
    static_assert(NT / R == PL && PARTS == 16 && RQ == 8, "the trained shapes' proportions");
    __shared__ float hs[YGG_MAX_LAYERS][N];   // states
    __shared__ float bl[N], hn[N];            // rms(h) of the layer below; the new state
    __shared__ float zp[PARTS][R2 + 1], zl[R2], up[4][N], zs[R], red[N / 64], lgp[QP][256];
    __shared__ uint32_t dec[4];               // a round's decisions, a bit per node of its subtree
    // (ANY) maxima of |h| per 16 coordinates, |zl| and |z| per row
    constexpr int NM = ANY ? N / 16 + R2 + R : 1;
    __shared__ float top[ANY ? YGG_MAX_LAYERS : 1][NM];
    const int s = blockIdx.x, tid = threadIdx.x, lane = tid & 63, L = m.L, V = m.V, C = m.classes, F = m.F, D = m.D;
    const bool rs = m.router_state != 0;
    float *st = state + (size_t)s * L * N;
    for (int i = tid; i < L * N; i += NT) hs[i / N][i % N] = st[i];
    if (tid < 4) dec[tid] = 0u;
    if constexpr (ANY)
        for (int i = tid; i < L * NM; i += NT) top[i / NM][i % NM] = 0.0f;
    __syncthreads();
    const int32_t *tok = tokens + (size_t)s * Tn;
    for (int t = 0; t < Tn; t++) {
        const int x = __builtin_amdgcn_readfirstlane(tok[t]);
        if (x < 0 || x >= V) {
            if (tid == 0) atomicOr(m.err, 1u);
            break;
        }
        float lg = 0.0f, vv[VC], w[N / G], wt[FE], emb[FE], bias = 0.0f;
        int rg = 0, rl = 0, vk = 0, vp = 0, ui = 0, uq = 0, qc = 0, qp = 0, kdep = 0, path = 0;
        // this thread's places, computed again in each layer (hidden from the compiler: every array's offset kept over
        // the loop does not fit the registers at n = 256, 26 of them spilled)
        auto places = [&] {
            int i = tid;
            asm volatile("" : "+v"(i));
            i &= NT - 1;
            rg = i / G, rl = i % G, vk = i % R2, vp = i / R2, ui = i % N, uq = i / N, qc = i & 255, qp = i >> 8;
            kdep = 31 - __builtin_clz(rg + 1), path = rg + 1 - (1 << kdep);     // node rg of a subtree
        };
        // layer l's V', token part and the rows of its round from node `root` (heap order) of h levels
        auto load_below = [&](int l) {
            const float *v = from(m.layers[l].Vd, vp * VC * R2 + vk);
#pragma unroll
            for (int i = 0; i < VC; i++) vv[i] = v[i * R2];
            const float *e = m.layers[l].emb + (size_t)x * F;
#pragma unroll
            for (int k = 0; k < FE; k++) emb[k] = *from(e, min(rl + G * k, F - 1));
        };
        // the row of this thread's node of a round (lanes past the round's nodes: a row that nobody reads)
        auto node_of = [&](int root, int h) { return rg < (1 << h) - 1 ? ((root + 1) << kdep) - 1 + path : 0; };
        auto load_round = [&](int l, int root, int h) {
            const int at = node_of(root, h);
            const uint32_t row = (uint32_t)at * (F + (rs ? N : 0));      // (at most 2^20 rows of 512)
#pragma unroll
            for (int k = 0; k < FE; k++) wt[k] = *from(m.layers[l].W, row + min(rl + G * k, F - 1));
            const float *ws = rs ? from(m.layers[l].W, row + F + rl) : from(m.layers[l].P, rl);   // (P: not used)
#pragma unroll
            for (int k = 0; k < N / G; k++) w[k] = ws[G * k];
            bias = *from(m.layers[l].bias, at);
        };
        for (int l = 0; l < L; l++) {
            const FloatLayerDev<float> &y = m.layers[l];
            int r = x;
            places();
            // 8 ranks of class qc's column of Q^T
            float qw[RQ];
#pragma unroll
            for (int j = 0; j < RQ; j++) qw[j] = *from(y.Q + j * C, qp * RQ * C + min(qc, C - 1));
            if (l > 0) {
                float f[N / G];
#pragma unroll
                for (int k = 0; k < N / G; k++) f[k] = bl[rl + G * k];
                float z = 0.0f;
#pragma unroll
                for (int i = 0; i < VC; i++) z = fmaf(vv[i], bl[vp * VC + i], z);
                zp[vp][vk] = z;
                int root = 0;
                for (int d0 = 0, rd = 0; d0 < D; d0 += 5, rd++) {
                    const int h = D - d0 < 5 ? D - d0 : 5;
                    if (rd) load_round(l, root, h);
                    float p = 0.0f;
#pragma unroll
                    for (int k = 0; k < FE; k++) p = rl + G * k < F ? fmaf(emb[k], wt[k], p) : p;
                    if constexpr (ANY) {
                        const float *e = y.emb + (size_t)x * F, *wr = y.W + (size_t)node_of(root, h) * (F + (rs ? N : 0));
                        for (int k = kStepF + rl; k < F; k += G) p = fmaf(e[k], wr[k], p);
                    }
                    if (rs) {
#pragma unroll
                        for (int k = 0; k < N / G; k++) p = fmaf(f[k], w[k], p);
                    }
                    p = lanes_sum<G>(p);
                    if (rl == 0 && rg < (1 << h) - 1 && p + bias > 0.0f) atomicOr(&dec[rd], 1u << rg);
                    __syncthreads();
                    if (rd == 0 && tid < R2) {
                        float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int q = 0; q < PARTS; q++) a[q % 4] += zp[q][tid];
                        zl[tid] = (a[0] + a[1]) + (a[2] + a[3]);
                        if constexpr (ANY) top[l][N / 16 + tid] = fmaxf(top[l][N / 16 + tid], fabsf(zl[tid]));
                    }
                    const uint32_t bits = dec[rd];
                    int j = 0;
                    for (int k = 0; k < h; k++) j = 2 * j + 1 + ((bits >> j) & 1u);
                    root = ((root + 1) << h) - 1 + (j - ((1 << h) - 1));
                }
                r = __builtin_amdgcn_readfirstlane(root - ((1 << D) - 1));
                if (D <= 5) __syncthreads();        // (zl, where no second round's barrier follows it)
            }
            // the expert's record: this thread's share of U', A and P; then the next layer's loads behind it
            float uw[UK], pw[PE], tab = 0.0f;
            if (l > 0) {
                const float *u = from(y.Up + (size_t)r * R2 * N, uq * UK * N + ui);
#pragma unroll
                for (int k = 0; k < UK; k++) uw[k] = u[k * N];
            }
            float4 aw = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (!ANY || y.A)
                aw = *(const float4 *)from(y.A + (size_t)r * N * 16, (ui / 16) * 256 + a_index<float>(16, ui % 16, 4 * uq));
            if (uq == 0) tab = *from(y.table + (l == 0 ? (size_t)x : (size_t)r * V + x) * N, ui);
            const int prow = (uq * N + ui) / PL, pu = ui % PL;
            const float *pr = from(y.P + (size_t)r * R * N, prow * N + pu);
#pragma unroll
            for (int e = 0; e < PE; e++) pw[e] = pr[PL * e];
            if (l + 1 < L) {
                load_below(l + 1);
                load_round(l + 1, 0, D < 5 ? D : 5);
            }
            float a = 0.0f, b = 0.0f;
            if (l > 0) {
#pragma unroll
                for (int k = 0; k < UK; k++) a = fmaf(uw[k], zl[uq * UK + k], a);
            }
            const float *ho = hs[l] + (ui & ~15) + 4 * uq;
            if (!ANY || y.A) {
                b = fmaf(aw.x, ho[0], b);
                b = fmaf(aw.y, ho[1], b);
                b = fmaf(aw.z, ho[2], b);
                b = fmaf(aw.w, ho[3], b);
            }
            up[uq][ui] = a + b;
            __syncthreads();
            if (tid < N) {
                const float h = tab + ((up[0][ui] + up[1][ui]) + (up[2][ui] + up[3][ui]));
                hn[ui] = h;
                hs[l][ui] = h;
                const float ss = wave_sum(h * h);
                if (lane == 0) red[tid >> 6] = ss;
                if constexpr (ANY) {
                    const float g = group_max_n(fabsf(h), 16);
                    if ((ui & 15) == 0) top[l][ui / 16] = fmaxf(top[l][ui / 16], g);
                }
            }
            if (tid < 4) dec[tid] = 0u;
            __syncthreads();
            float ss = 0.0f;
#pragma unroll
            for (int k = 0; k < N / 64; k++) ss += red[k];
            if (tid < N) bl[ui] = hn[ui] * (1.0f / sqrtf(ss / (float)N + (float)kRmsEps));
            float z = 0.0f;
#pragma unroll
            for (int e = 0; e < PE; e++) z = fmaf(pw[e], hn[pu + PL * e], z);
            z = lanes_sum<PL>(z);
            if (pu == 0) {
                zs[prow] = z;
                if constexpr (ANY) top[l][N / 16 + R2 + prow] = fmaxf(top[l][N / 16 + R2 + prow], fabsf(z));
            }
            __syncthreads();
            float q = 0.0f;
#pragma unroll
            for (int j = 0; j < RQ; j++) q = fmaf(qw[j], zs[qp * RQ + j], q);
            lg += q;
            if (leaves && tid == 0) leaves[((size_t)s * Tn + t) * L + l] = r;
        }
        if (logits) {
            lgp[qp][qc] = lg;
            __syncthreads();
            if (tid < C) {
                float v = lgp[0][tid];
#pragma unroll
                for (int k = 1; k < QP; k++) v += lgp[k][tid];
                logits[((size_t)s * Tn + t) * C + tid] = m.output_bias[tid] + v;
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < L * N; i += NT) st[i] = hs[i / N][i % N];
    if constexpr (ANY) {
        if (stats && tid < 64)
            for (int l = 0; l < L; l++) {
                double *to = stats + (size_t)l * (3 + N / 16 + R);
                const float h = lane < N / 16 ? top[l][lane] : 0.0f, v = lane < R2 ? top[l][N / 16 + lane] : 0.0f,
                            z = lane < R ? top[l][N / 16 + R2 + lane] : 0.0f;
                const double ha = wave_max(h), va = wave_max(v), za = wave_max(z);
                if (lane == 0) {
                    atomic_max_nonneg(to, ha);
                    atomic_max_nonneg(to + 1, va);
                    atomic_max_nonneg(to + 2, za);
                }
                if (lane < N / 16) atomic_max_nonneg(to + 3 + lane, h);
                if (lane < R) atomic_max_nonneg(to + 3 + N / 16 + lane, z);
            }
    }
}

template <int N, int R, int R2>
__global__ __launch_bounds__(4 * N) __attribute__((amdgpu_waves_per_eu(N / 64, 8))) void float_any_kernel(
    const FloatDevModel<float> m, const int32_t *__restrict__ tokens, int Tn, float *__restrict__ state,
    float *__restrict__ logits, int32_t *__restrict__ leaves, double *__restrict__ stats) {
    float_step<N, R, R2, true>(m, tokens, Tn, state, logits, leaves, stats);
}

// stats (calibration maxima, cpu/export.py:127-153), per layer: [|h|, |V' rms(h_below)|, |P_r h|, |h| per 16
// coordinates (n/16), |P_r h| per row (R)]
// NS, RS, R2S, BS: the state width, readout rank, layer-input rank and block size of a float_step build (the reference's
// trained shapes, as step_whole and without stats), or 0 for the model's (any shape the loader takes)
// (one wavefront per SIMD: the unrolled row loads of a thread are its registers)
template <typename T, int NS = 0, int RS = 0, int R2S = 0, int BS = 0>
__global__ __launch_bounds__(NS ? 4 * NS : kFThreads)
__attribute__((amdgpu_waves_per_eu(NS ? NS / 64 : 1, NS ? 8 : 1))) void float_kernel(
    const FloatDevModel<T> m, const int32_t *__restrict__ tokens, int Tn, T *__restrict__ state,
    T *__restrict__ logits, int32_t *__restrict__ leaves, double *__restrict__ stats) {
    if constexpr (NS != 0) {
        float_step<NS, RS, R2S, false>(m, tokens, Tn, state, logits, leaves, nullptr);
        return;
    } else {
    constexpr int MN = kMaxN, MR = kMaxR, MR2 = kMaxR2, MB = kMaxB;
    __shared__ T hs[YGG_MAX_LAYERS][kMaxN];   // states
    __shared__ T bl[kMaxN];                   // rms(h) of the layer below
    __shared__ T hn[kMaxN];                   // the new state of the current layer
    __shared__ T zl[kMaxR2];
    __shared__ T zs[kMaxR];
    __shared__ T zp[4][kMaxR2];               // the layer input's partial sums, per quarter of the coordinates
    __shared__ T red[4];
    __shared__ int dec[16];                   // a router round's decisions, by breadth-first node of its subtree
    __shared__ double gmax[YGG_MAX_LAYERS][kMaxN / 16];

    constexpr int PE = MN / 4;   // readout coordinates per thread
    const int s = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int L = m.L, n = m.n, b = m.b, V = m.V, C = m.classes, R = m.R, R2 = m.R2, F = m.F;
    const int width = F + (m.router_state ? n : 0);
    // readout: TPR threads per row of P (a power of 2 of at most 64 lanes), its coordinates u, u + TPR, ...
    int Rp = 1;
    while (Rp < R) Rp <<= 1;
    const int TPR = kFThreads / Rp > 64 ? 64 : kFThreads / Rp;
    const int prow = tid / TPR, pu = tid % TPR;
    // layer input: wave q takes the quarter q of the coordinates, lane k row k of V'
    const int vrow = lane, vq = tid >> 6, vlen = n / 4;
    // router rounds: group g of kRouteGroup threads forms node g of the round's subtree
    const int rg = tid / kRouteGroup, rl = tid % kRouteGroup;

    T *st = state + (size_t)s * L * n;
    for (int l = 0; l < L; l++)
        for (int i = tid; i < n; i += kFThreads) hs[l][i] = st[(size_t)l * n + i];
    for (int l = 0; l < L; l++)
        for (int g = tid; g < n / 16; g += kFThreads) gmax[l][g] = 0.0;
    // per-thread maxima (calibration runs only): |h| (thread i's coordinate), |zl| (row vrow's reducer), |z| (row
    // prow's reducer)
    double smax[YGG_MAX_LAYERS], vmax[YGG_MAX_LAYERS], zmax[YGG_MAX_LAYERS];
    for (int l = 0; l < YGG_MAX_LAYERS; l++) smax[l] = vmax[l] = zmax[l] = 0.0;
    const int sstride = 3 + n / 16 + R;
    __syncthreads();

    const int32_t *tok = tokens + (size_t)s * Tn;
    for (int t = 0; t < Tn; t++) {
        const int x = __builtin_amdgcn_readfirstlane(tok[t]);
        if (x < 0 || x >= V) {
            if (tid == 0) atomicOr(m.err, 1u);
            break;
        }
        T lg = tid < C ? m.output_bias[tid] : T(0);
        for (int l = 0; l < L; l++) {
            const FloatLayerDev<T> &y = m.layers[l];
            int r = x;
            // the layer's constants: class c's column of Q^T (thread c) and this thread's share of V' (wave q's quarter
            // of the coordinates of row k = lane)
            T qw[MR], vv[MN / 4];
            auto load_q = [&]() {
                if (tid < C) {
                    const T *q = y.Q + tid;
#pragma unroll
                    for (int j = 0; j < MR; j++) qw[j] = j < R ? q[(size_t)j * C] : T(0);
                }
            };
            const bool vlive = l > 0 && y.Vd != nullptr && vrow < R2;
            auto load_v = [&]() {
                if (vlive) {
                    const T *vc = y.Vd + (size_t)(vq * vlen) * R2 + vrow;
#pragma unroll
                    for (int i = 0; i < MN / 4; i++) vv[i] = i < vlen ? vc[(size_t)i * R2] : T(0);
                }
            };
            if (l > 0) {
                // router descent over f = [router_embed[x]; rms(h_below)], in rounds of up to 4 levels
                T f[kRouteElems];
                const T *e = y.emb + (size_t)x * F;
#pragma unroll
                for (int k = 0; k < kRouteElems; k++) {
                    const int i = rl + kRouteGroup * k;
                    f[k] = i < F ? e[i] : (i < width ? bl[i - F] : T(0));
                }
                int root = 0;
                for (int d0 = 0; d0 < m.D; d0 += 4) {
                    const int h = m.D - d0 < 4 ? m.D - d0 : 4;
                    const int nn = (1 << h) - 1;
                    // node rg of the subtree: depth k = floor(log2(rg + 1)), path p = rg + 1 - 2^k
                    const int kdep = 31 - __builtin_clz(rg + 1), path = rg + 1 - (1 << kdep);
                    const int node = ((root + 1) << kdep) - 1 + path;
                    T p = T(0);
                    if (rg < nn) {
                        const T *w = y.W + (size_t)node * width;
                        T wl[kRouteElems];
#pragma unroll
                        for (int k = 0; k < kRouteElems; k++) {
                            const int i = rl + kRouteGroup * k;
                            wl[k] = i < width ? w[i] : T(0);
                        }
#pragma unroll
                        for (int k = 0; k < kRouteElems; k++) p += f[k] * wl[k];
                    }
                    p = group_sum<kRouteGroup>(p);
                    if (rg < nn && rl == 0) dec[rg] = (p + y.bias[node]) > T(0) ? 1 : 0;
                    __syncthreads();
                    int q = 0;
                    for (int k = 0; k < h; k++) q = 2 * q + dec[(1 << k) - 1 + q];
                    root = ((root + 1) << h) - 1 + q;
                    __syncthreads();
                }
                r = root - ((1 << m.D) - 1);
                // the layer input zl = V' rms(h_below): each wave's partial sum for row k = lane over its quarter of
                // the coordinates, the four partials then added in quarter order
                if (y.Vd) {
                    load_v();
                    if (vlive) {
                        T a = T(0);
#pragma unroll
                        for (int i = 0; i < MN / 4; i++)
                            if (i < vlen) a += vv[i] * bl[vq * vlen + i];
                        zp[vq][vrow] = a;
                    }
                    __syncthreads();
                    if (tid < R2) {
                        const T z = ((zp[0][tid] + zp[1][tid]) + zp[2][tid]) + zp[3][tid];
                        zl[tid] = z;
                        if (stats) vmax[l] = fmax(vmax[l], (double)fabs(z));
                    }
                    __syncthreads();
                }
            }
            // expert r's P row share for the readout: TPR threads per row, coordinates pu, pu + TPR, ...
            T pw[PE];
            auto load_p = [&]() {
                if (prow < R) {
                    const T *pr = y.P + ((size_t)r * R + prow) * n;
#pragma unroll
                    for (int e = 0; e < PE; e++) pw[e] = pu + TPR * e < n ? pr[pu + TPR * e] : T(0);
                }
            };
            // h = T_r[x] + U'_r zl + A_r h_old, thread i for coordinate i
            T hv = T(0);
            if (tid < n) {
                // (the table entry, U' column and A row of coordinate i loaded together; sums in index order)
                const int i = tid;
                const T *trow = l == 0 ? y.table + (size_t)x * n : y.table + ((size_t)r * V + x) * n;
                const bool up = l > 0 && y.Up != nullptr, ta = y.A != nullptr;
                const int g = i / b, ii = i % b;
                const T *u = up ? y.Up + (size_t)r * R2 * n + i : nullptr;                    // column i
                const T *ablk = ta ? y.A + ((size_t)r * (n / b) + g) * b * b : nullptr;       // block g
                T uw[MR2], aw[MB];
#pragma unroll
                for (int k = 0; k < MR2; k++) uw[k] = (up && k < R2) ? u[(size_t)k * n] : T(0);
                // (a_index: in f32 whole 16-byte chunks of row ii for b = 16; in f64 they spilled 28 registers more beside the
                // other layout's loads, 3 to 8% of a token, so there either layout's entries are loaded by strides)
                constexpr int VE = 16 / (int)sizeof(T);
                if (sizeof(T) == 4 && ta && b == 16) {
                    struct alignas(16) Chunk { T v[VE]; };
#pragma unroll
                    for (int j = 0; j < MB / VE; j++) {
                        const Chunk w = *(const Chunk *)(ablk + a_index<T>(16, ii, j * VE));
#pragma unroll
                        for (int e = 0; e < VE; e++) aw[j * VE + e] = w.v[e];
                    }
                } else {
                    const bool chunks = sizeof(T) == 8 && b == 16;
                    const T *arow = ta ? ablk + (chunks ? ii * VE : ii) : nullptr;
                    const int chunk = VE * b, next = chunks ? 1 : b;
#pragma unroll
                    for (int j = 0; j < MB; j++) aw[j] = (ta && j < b) ? arow[j / VE * chunk + j % VE * next] : T(0);
                }
                T h = trow[i];
                if (up) {
                    T a = T(0);
#pragma unroll
                    for (int k = 0; k < MR2; k++)
                        if (k < R2) a += uw[k] * zl[k];
                    h = h + a;
                }
                if (ta) {
                    T a = T(0);
#pragma unroll
                    for (int j = 0; j < MB; j++)
                        if (j < b) a += aw[j] * hs[l][g * b + j];
                    h = h + a;
                }
                hv = h;
                if (stats) smax[l] = fmax(smax[l], (double)fabs(h));
            }
            // (every thread has read hs[l] before it is overwritten below)
            const T ss = block_sum(tid < n ? hv * hv : T(0), red, tid);
            if (tid < n) {
                hn[tid] = hv;
                hs[l][tid] = hv;
            }
            if (stats && tid < n) {
                // |h| per 16 coordinates: 16 consecutive threads
                const double a = group_max_n((double)fabs(hv), 16);
                if ((tid & 15) == 0) gmax[l][tid >> 4] = fmax(gmax[l][tid >> 4], a);
            }
            const T rinv = T(1) / sqrt(ss / T(n) + T(kRmsEps));
            if (tid < n) bl[tid] = hv * rinv;
            __syncthreads();
            // z = P_r h (every load issued at once)
            load_p();
            if (prow < R) {
                T a = T(0);
#pragma unroll
                for (int e = 0; e < PE; e++)
                    if (pu + TPR * e < n) a += pw[e] * hn[pu + TPR * e];
                a = group_sum_n(a, TPR);
                if (pu == 0) {
                    zs[prow] = a;
                    if (stats) zmax[l] = fmax(zmax[l], (double)fabs(a));   // row prow's reducer holds its maximum
                }
            }
            __syncthreads();
            // logits += Q z, thread c for class c
            load_q();
            if (tid < C) {
                T a = T(0);
#pragma unroll
                for (int j = 0; j < MR; j++)
                    if (j < R) a += qw[j] * zs[j];
                lg = lg + a;
            }
            if (leaves && tid == 0) leaves[((size_t)s * Tn + t) * L + l] = r;
            __syncthreads();
        }
        if (logits && tid < C) logits[((size_t)s * Tn + t) * C + tid] = lg;
    }
    __syncthreads();
    for (int l = 0; l < L; l++)
        for (int i = tid; i < n; i += kFThreads) st[(size_t)l * n + i] = hs[l][i];
    if (stats) {
        for (int l = 0; l < L; l++) {
            const double a = wave_max(smax[l]), v = wave_max(vmax[l]), z = wave_max(zmax[l]);
            if (lane == 0) {
                atomic_max_nonneg(&stats[(size_t)l * sstride + 0], a);
                atomic_max_nonneg(&stats[(size_t)l * sstride + 1], v);
                atomic_max_nonneg(&stats[(size_t)l * sstride + 2], z);
            }
            for (int g = tid; g < n / 16; g += kFThreads)
                atomic_max_nonneg(&stats[(size_t)l * sstride + 3 + g], gmax[l][g]);
            if (prow < R && pu == 0) atomic_max_nonneg(&stats[(size_t)l * sstride + 3 + n / 16 + prow], zmax[l]);
        }
    }
    }
}

}  // namespace

namespace ygg::flt {
int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    return ygg::set_error(code, buf);
}
}  // namespace ygg::flt

namespace {

template <typename T> int upload(const ygg_float_desc *d, int device, ygg_fmodel *fm, FloatDevModel<T> &m) {
    const int L = d->n_layers, n = d->d_state, b = d->block_size, V = d->vocab, C = d->classes, D = d->router_depth,
              R = d->readout_rank, R2 = d->layer_input_rank, F = d->router_token_dim;
    const int64_t E = (int64_t)1 << D, nodes = E - 1, width = F + (d->router_state ? n : 0);
    // a part is `outer` matrices of rows x cols, stored as given (rows = 0), each transposed, or (block) as a_index
    // places a transition block
    struct Part { const double *src; int64_t count; size_t off; int64_t outer, rows, cols; bool block; };
    std::vector<Part> parts;
    size_t total = 256;   // the error word first
    auto add = [&](const double *src, int64_t count, int64_t rows = 0, int64_t cols = 0, bool block = false) -> int {
        if (!src || count <= 0) return -1;
        parts.push_back({src, count, total, rows ? count / (rows * cols) : 0, rows, cols, block});
        total += ((size_t)count * sizeof(T) + 255) / 256 * 256;
        return (int)parts.size() - 1;
    };
    const int ob = add(d->output_bias, C);
    if (ob < 0) return fail(YGG_ERR_ARG, "float model: output_bias is NULL");
    struct Idx { int table, A, P, Q, emb, W, bias, Vd, Up; };
    std::vector<Idx> idx(L);
    // the layers' transposed unembeddings one after the other: [L R][classes]
    for (int l = 0; l < L; l++) {
        idx[l].Q = add(d->layers[l].unembed, (int64_t)C * R, C, R);
        if (idx[l].Q >= 0) total = parts.back().off + (size_t)C * R * sizeof(T);
    }
    total = (total + 255) / 256 * 256;
    for (int l = 0; l < L; l++) {
        const ygg_float_layer &y = d->layers[l];
        const int64_t El = l == 0 ? V : E;
        Idx &k = idx[l];
        k.table = add(y.table, l == 0 ? (int64_t)V * n : El * V * n);
        k.A = add(y.transition, El * n * b, b, b, true);
        k.P = add(y.readout, El * R * n);
        k.emb = l ? add(y.router_embed, (int64_t)V * F) : -1;
        k.W = l ? add(y.router_weight, nodes * width) : -1;
        k.bias = l ? add(y.router_bias, nodes) : -1;
        k.Vd = (l && R2) ? add(y.layer_input_down, (int64_t)R2 * n, R2, n) : -1;
        k.Up = (l && R2) ? add(y.layer_input_proj, El * n * R2, n, R2) : -1;
        if (k.table < 0 || k.P < 0 || k.Q < 0 || (l && (k.emb < 0 || k.W < 0 || k.bias < 0)) ||
            (l && R2 && (k.Vd < 0 || k.Up < 0)))
            return fail(YGG_ERR_ARG, "float model: layer %d lacks an array", l);
    }
    // the description is checked before any device is touched
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return fail(YGG_ERR_DEVICE, "no HIP device");
    if (device < 0 || device >= ndev) return fail(YGG_ERR_ARG, "device %d out of range", device);
    std::vector<uint8_t> host;
    try {
        host.assign(total, 0);
    } catch (const std::bad_alloc &) {
        return fail(YGG_ERR_NOMEM, "float model: %zu bytes of host staging", total);
    }
    for (const Part &p : parts) {
        T *dst = (T *)(host.data() + p.off);
        if (!p.rows) {
            for (int64_t i = 0; i < p.count; i++) dst[i] = (T)p.src[i];
            continue;
        }
        const int64_t mat = p.rows * p.cols;
        for (int64_t o = 0; o < p.outer; o++)
            for (int64_t r = 0; r < p.rows; r++)
                for (int64_t c = 0; c < p.cols; c++)
                    dst[o * mat + (p.block ? a_index<T>((int)p.rows, (int)r, (int)c) : c * p.rows + r)] =
                        (T)p.src[o * mat + r * p.cols + c];
    }
    DeviceGuard g;
    HIP_TRY(g.set(device));
    void *arena = nullptr;
    HIP_TRY(hipMalloc(&arena, total));
    hipError_t e = hipMemcpy(arena, host.data(), total, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(arena);
        return fail(YGG_ERR_DEVICE, "upload failed: %s", hipGetErrorString(e));
    }
    uint8_t *A = (uint8_t *)arena;
    auto at = [&](int i) -> const T * { return i < 0 ? nullptr : (const T *)(A + parts[i].off); };
    m.L = L; m.n = n; m.b = b; m.V = V; m.classes = C; m.D = D; m.R = R; m.R2 = R2; m.F = F;
    m.router_state = d->router_state;
    m.output_bias = at(ob);
    m.err = (uint32_t *)arena;
    for (int l = 0; l < L; l++) {
        const Idx &k = idx[l];
        m.layers[l] = FloatLayerDev<T>{at(k.table), at(k.A), at(k.P), at(k.Q), at(k.emb), at(k.W), at(k.bias),
                                       at(k.Vd), at(k.Up)};
    }
    fm->arena = arena;
    fm->arena_bytes = total;
    return YGG_OK;
}

}  // namespace

extern "C" {

int ygg_float_load(const ygg_float_desc *d, int precision, int device, ygg_fmodel **out) {
    if (!out) return fail(YGG_ERR_ARG, "out is NULL");
    *out = nullptr;
    if (!d) return fail(YGG_ERR_ARG, "desc is NULL");
    if (precision != 32 && precision != 64) return fail(YGG_ERR_ARG, "precision %d: 32 or 64", precision);
    const int L = d->n_layers, n = d->d_state, b = d->block_size;
    if (L < 1 || L > YGG_MAX_LAYERS || n < 16 || n > kMaxN || n % 16 || b < 1 || b > kMaxB || n % b || d->vocab < 1 ||
        d->classes < 1 || d->classes > kMaxClasses || d->readout_rank < 1 || d->readout_rank > kMaxR ||
        d->layer_input_rank < 0 || d->layer_input_rank > kMaxR2 || (L > 1 && (d->router_depth < 1 ||
        d->router_depth > 20 || d->router_token_dim < 0 || d->router_token_dim > kMaxF)))
        return fail(YGG_ERR_LIMITS, "float model: unsupported shape (L %d, n %d, b %d, classes %d, R %d, R2 %d, D %d)",
                    L, n, b, d->classes, d->readout_rank, d->layer_input_rank, d->router_depth);
    ygg_fmodel *fm = new ygg_fmodel();
    fm->device = device;
    fm->precision = precision;
    const int rc = precision == 32 ? upload<float>(d, device, fm, fm->m32) : upload<double>(d, device, fm, fm->m64);
    if (rc != YGG_OK) {
        delete fm;
        return rc;
    }
    *out = fm;
    return YGG_OK;
}

int ygg_float_run(const ygg_fmodel *m, const int32_t *d_tokens, int B, int T, void *d_state, void *d_logits,
                  int32_t *d_leaves, double *d_stats, void *stream) {
    if (!m) return fail(YGG_ERR_ARG, "model is NULL");
    if (B < 0 || T < 0) return fail(YGG_ERR_ARG, "negative B (%d) or T (%d)", B, T);
    if (B == 0) return YGG_OK;
    if (!d_state || (T > 0 && !d_tokens)) return fail(YGG_ERR_ARG, "tokens or state is NULL");
    DeviceGuard g;
    HIP_TRY(g.set(m->device));
    if (m->precision == 32) {
        // the reference's trained shapes (configs/*/{small,medium,large}.yaml: block 16) have builds of their own
        const FloatDevModel<float> &fm = m->m32;
        auto go = [&](auto kernel, int threads) {
            hipLaunchKernelGGL(kernel, dim3(B), dim3(threads), 0, (hipStream_t)stream, fm, d_tokens, T,
                               (float *)d_state, (float *)d_logits, d_leaves, d_stats);
        };
        const bool any = d_stats || !step_whole(fm);
        if (!float_steps(fm)) go(float_kernel<float>, kFThreads);
        else if (fm.n == 64) any ? go(float_any_kernel<64, 8, 16>, 256) : go(float_kernel<float, 64, 8, 16, 16>, 256);
        else if (fm.n == 128) any ? go(float_any_kernel<128, 16, 32>, 512) : go(float_kernel<float, 128, 16, 32, 16>, 512);
        else any ? go(float_any_kernel<256, 32, 64>, 1024) : go(float_kernel<float, 256, 32, 64, 16>, 1024);
    } else
        hipLaunchKernelGGL(float_kernel<double>, dim3(B), dim3(kFThreads), 0, (hipStream_t)stream, m->m64, d_tokens, T,
                           (double *)d_state, (double *)d_logits, d_leaves, d_stats);
    HIP_TRY(hipGetLastError());
    return YGG_OK;
}

int ygg_float_take_errors(const ygg_fmodel *m, void *stream, uint32_t *errors) {
    if (!m || !errors) return fail(YGG_ERR_ARG, "NULL argument");
    DeviceGuard g;
    HIP_TRY(g.set(m->device));
    HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
    uint32_t v = 0;
    HIP_TRY(hipMemcpy(&v, m->arena, 4, hipMemcpyDeviceToHost));
    if (v) {
        const uint32_t zero = 0;
        HIP_TRY(hipMemcpy(m->arena, &zero, 4, hipMemcpyHostToDevice));
    }
    *errors = v;
    return YGG_OK;
}

void ygg_float_free(ygg_fmodel *m) {
    if (!m) return;
    DeviceGuard g;
    if (g.set(m->device) == hipSuccess) (void)hipFree(m->arena);
    delete m;
}

}  // extern "C"
