// The float model on the device, shared by its two forms: the per-stream step (ygg_float.hip) and the layer-by-layer
// form for many known tokens (ygg_float_scan.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/ygg_hip.h"
#include "ygg_layout.h"

namespace ygg {
int set_error(int code, const char *msg);
}

namespace ygg::flt {

constexpr int kMaxN = 256, kMaxR = 64, kMaxR2 = 64, kMaxClasses = 256, kMaxF = 256, kMaxB = 16;
constexpr double kRmsEps = 1e-6;   // yggdrasil/config.py:8

// Device layouts: the arrays a thread reads a row of at each step of a dot are stored transposed from the checkpoint's,
// so that the lanes of a wavefront read consecutive addresses at every step.
template <typename T> struct FloatLayerDev {
    const T *table;          // token layer [V][n] (T_x[x]); routed [E][V][n]
    const T *A;              // [E][n/b] blocks of b x b (a_index) or null
    const T *P;              // [E][R][n]
    const T *Q;              // [R][classes] (transposed); the layers' lie one after the other, so layer 0's is [L R][classes]
    const T *emb;            // routed: [V][F]
    const T *W;              // routed: [nodes][F + n] (router_state) or [nodes][F]
    const T *bias;           // routed: [nodes]
    const T *Vd;             // [n][R2] (transposed) or null
    const T *Up;             // [E][R2][n] (each expert's matrix transposed) or null
};

// The place of entry (row i, column j) of a transition block: for b = 16, 16-byte chunks of a row's columns, interleaved
// by row, so that 16 lanes that take a row each read a block in whole lines; otherwise transposed.
template <typename T> __host__ __device__ constexpr int a_index(int b, int i, int j) {
    constexpr int VE = 16 / (int)sizeof(T);
    return b == 16 ? (j / VE) * 16 * VE + i * VE + j % VE : j * b + i;
}

template <typename T> struct FloatDevModel {
    int L, n, b, V, classes, D, R, R2, F, router_state;
    const T *output_bias;    // [classes]
    uint32_t *err;
    FloatLayerDev<T> layers[YGG_MAX_LAYERS];
};

// Whether a model has the f32 step of the trained shapes.
inline bool float_steps(const FloatDevModel<float> &m) {
    return m.b == 16 && ((m.n == 64 && m.R == 8 && m.R2 == 16) || (m.n == 128 && m.R == 16 && m.R2 == 32) ||
                         (m.n == 256 && m.R == 32 && m.R2 == 64));
}
inline bool float_steps(const FloatDevModel<double> &) { return false; }
// Whether that step's plain build takes it (calls without maxima): with transitions, and at most 32 token entries in a
// router's input (a lane's loads of a node's row are one of these and 8 of the state's).
constexpr int kStepF = 32;
inline bool step_whole(const FloatDevModel<float> &m) {
    if (m.L > 1 && m.F > kStepF) return false;
    for (int l = 0; l < m.L; l++)
        if (!m.layers[l].A) return false;
    return true;
}

int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));

struct DeviceGuard {
    int prev = -1;
    hipError_t set(int dev) {
        hipError_t e = hipGetDevice(&prev);
        if (e != hipSuccess) { prev = -1; return e; }
        return hipSetDevice(dev);
    }
    ~DeviceGuard() {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

}  // namespace ygg::flt

#define HIP_TRY(expr)                                                                                             \
    do {                                                                                                          \
        hipError_t e_ = (expr);                                                                                   \
        if (e_ != hipSuccess) return ygg::flt::fail(YGG_ERR_DEVICE, "%s: %s", #expr, hipGetErrorString(e_));      \
    } while (0)

struct ygg_fmodel {
    int device = 0, precision = 32;
    void *arena = nullptr;
    size_t arena_bytes = 0;
    ygg::flt::FloatDevModel<float> m32{};
    ygg::flt::FloatDevModel<double> m64{};
};
