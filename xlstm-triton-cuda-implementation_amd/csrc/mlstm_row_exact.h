// Rows of the fp32 row kernels from their definition, shared by mlstm_row.hip and mlstm_rowf.hip.
#pragma once
#include "mlstm_device.h"
#include "mlstm_kernels.h"

namespace mlstm {

constexpr int ROW_MODE_FWD = 0, ROW_MODE_DQ = 1;

// One row by one wave from its definition, in fp32 multiply-adds straight from memory (see not_finite in mlstm_device.h): the keys
// of the row's own chunk one after the other and the state before it, columns lane and lane + 64.  Positions count from the
// chunk's first one, as in the kernel.
template <int D, int MODE>
__device__ __forceinline__ void row_exact(const RowArgs& a, int bh, int chunk, int t, int S, size_t hoff, size_t poff, size_t goff, const float* x,
                                          const float* Y1, const float* Y2, size_t rsA, size_t offA, size_t offO, size_t offB, size_t rsO, size_t rsB,
                                          float inv_n, float db) {
    constexpr int NC = D / 64;
    const int lane = threadIdx.x & 63;
    const double G = a.G2[goff + t / GRAN];
    const float crow = -0.5f * __log2f((float)D) - a.beta2[poff + t];
    float xv[NC], o[NC], b = 0.f;
#pragma unroll
    for (int n = 0; n < NC; n++) { xv[n] = x[lane + 64 * n]; o[n] = 0.f; }
    if (chunk > 0) {
        const size_t st = (size_t)bh * a.n_states + chunk - 1;
        const float* C = reinterpret_cast<const float*>(a.Cst) + st * D * D;
        const float* nst = a.Nst + st * D;
        for (int k = 0; k < D; k++) {   // (row k of the state lies where the tile kernels' transposing reads want it: mlstm_chunk.hip)
            const float xk = x[k];
            const int at = (k & ~12) | ((k & 4) << 1) | ((k & 8) >> 1);
#pragma unroll
            for (int n = 0; n < NC; n++) o[n] += xk * C[(size_t)at * D + lane + 64 * n];
            if constexpr (MODE == ROW_MODE_FWD) b += xk * nst[k];
        }
        const float dec = fast_exp2(a.beta2[poff - 1] - a.beta2[poff + t] + (float)(G - a.G2[goff - 1]));
        if constexpr (MODE == ROW_MODE_FWD) {
            b *= dec;
#pragma unroll
            for (int n = 0; n < NC; n++) o[n] *= dec;
        } else {
            const float* q = reinterpret_cast<const float*>(a.Qrow) + offA + (size_t)t * rsA;
            float rp = 0.f;
#pragma unroll
            for (int n = 0; n < NC; n++) {
                o[n] = o[n] * (dec * inv_n) + dec * db * nst[lane + 64 * n];
                rp += o[n] * q[lane + 64 * n];
            }
            rp = wave_reduce<OpAdd>(rp);
            if (lane == (t & 31)) a.rowinter[hoff + t] = rp;
        }
    }
    for (int j = 0; j <= t; j++) {
        float s = 0.f;
#pragma unroll
        for (int n = 0; n < NC; n++) s += xv[n] * Y1[(size_t)j * rsA + lane + 64 * n];
        s = wave_reduce<OpAdd>(s);
        const float e = fast_exp2(a.alpha2[poff + j] + (crow + (float)(G - a.G2[goff + j / GRAN])));
        const float p = MODE == ROW_MODE_FWD ? s * e : (s * inv_n + db) * e;
        b += p;
#pragma unroll
        for (int n = 0; n < NC; n++) o[n] += p * Y2[(size_t)j * rsA + lane + 64 * n];
    }
    float onorm = 1.0f;
    if constexpr (MODE == ROW_MODE_FWD) {
        onorm = 1.0f / (fmaxf(fabsf(b), __expf(-a.M[hoff + t])) + 1e-6f);
        if (lane == (t & 31)) a.Bsum[hoff + t] = b;
    }
#pragma unroll
    for (int n = 0; n < NC; n++) {
        const int d = lane + 64 * n;
        reinterpret_cast<float*>(a.out)[offO + (size_t)t * rsO + d] = o[n] * onorm;
        if constexpr (MODE == ROW_MODE_FWD) {
            if (a.O) {
                const size_t at = offB + (size_t)t * rsB + d;
                reinterpret_cast<float*>(a.out_gated)[at] = o[n] * onorm * silu(reinterpret_cast<const float*>(a.O)[at]);
            }
        }
    }
}

}  // namespace mlstm
