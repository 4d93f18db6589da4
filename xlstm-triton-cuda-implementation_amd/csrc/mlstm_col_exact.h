// Keys of the fp32 column kernels from their definition, shared by mlstm_col.hip and mlstm_colf.hip.
#pragma once
#include "mlstm_device.h"
#include "mlstm_kernels.h"

namespace mlstm {

// KEYS keys from key0 on, of the granule jt, by their workgroup from the definitions, in fp32 multiply-adds straight from memory (see not_finite in mlstm_device.h):
// dK, dV and the column sums a key per wave, over the queries of the key's own chunk and the reverse state behind it, columns
// lane and lane + 64; then the row partials
// (slice: [S]) a query per wave and a key per lane.
template <int D, int KEYS>
__device__ __forceinline__ void col_exact(const ColArgs& a, int bh, int key0, int chunk, int NGe, bool has_state, const float* Q, const float* dH, const float* K,
                                          const float* V, size_t rsA, size_t rsB, size_t offA, float* slice) {
    constexpr int NC = D / 64;
    const int jt = key0 / GRAN;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, S = a.S, end = GRAN * NGe < S ? GRAN * NGe : S;
    const size_t hoff = (size_t)bh * S, poff = (size_t)bh * a.NG * GRAN, goff = (size_t)bh * a.NG;
    const double gj = a.G2[goff + jt];
    const float log2scale = -0.5f * __log2f((float)D);
    auto gate = [&](int t) { return log2scale - a.beta2[poff + t] + (float)(a.G2[goff + t / GRAN] - gj); };   // plus alpha2 of the key
    for (int j = key0 + wave; j < key0 + KEYS && j < S; j += 4) {
        const float al = a.alpha2[poff + j];
        float k[NC], v[NC], dk[NC], dv[NC], col = 0.f;
#pragma unroll
        for (int n = 0; n < NC; n++) { k[n] = K[(size_t)j * rsA + lane + 64 * n]; v[n] = V[(size_t)j * rsA + lane + 64 * n]; dk[n] = dv[n] = 0.f; }
        if (has_state) {   // (rows of the state: see row_exact)
            const size_t st = (size_t)bh * a.n_states + chunk;
            const float* E = reinterpret_cast<const float*>(a.Ev) + st * D * D;
            const float* g = a.gvec + st * D;
            auto at = [](int u) { return (size_t)((u & ~12) | ((u & 4) << 1) | ((u & 8) >> 1)) * D; };
            for (int u = 0; u < D; u++) {
                const float vu = V[(size_t)j * rsA + u], ku = K[(size_t)j * rsA + u];
#pragma unroll
                for (int n = 0; n < NC; n++) {
                    dk[n] += vu * E[at(u) + lane + 64 * n];
                    dv[n] += ku * E[at(lane + 64 * n) + u];
                }
            }
            const int pe = (chunk + 1) * a.chunk_len - 1;
            const float w = fast_exp2(al - a.beta2[poff + pe] + (float)(a.G2[goff + pe / GRAN] - gj));
#pragma unroll
            for (int n = 0; n < NC; n++) {
                dk[n] = (dk[n] + g[lane + 64 * n]) * w;
                dv[n] *= w;
                col += dk[n] * k[n];
            }
            col = wave_reduce<OpAdd>(col);
        }
        for (int t = j; t < end; t++) {
            float q[NC], u[NC], s = 0.f, dc = 0.f;
#pragma unroll
            for (int n = 0; n < NC; n++) {
                q[n] = Q[(size_t)t * rsA + lane + 64 * n];
                u[n] = dH[(size_t)t * rsB + lane + 64 * n];
                s += q[n] * k[n];
                dc += u[n] * v[n];
            }
            const float e = fast_exp2(al + gate(t)), inv = a.inv_n[poff + t];
            const float ct = wave_reduce<OpAdd>(s) * e, dct = wave_reduce<OpAdd>(dc) * inv + a.db[poff + t];
            col += ct * dct;
#pragma unroll
            for (int n = 0; n < NC; n++) {
                dk[n] += dct * e * q[n];
                dv[n] += ct * inv * u[n];
            }
        }
#pragma unroll
        for (int n = 0; n < NC; n++) {
            const size_t at = offA + (size_t)j * rsA + lane + 64 * n;
            reinterpret_cast<float*>(a.dK)[at] = dk[n];
            reinterpret_cast<float*>(a.dV)[at] = dv[n];
        }
        if (lane == 0) a.colsum[hoff + j] = col;
    }
    const int j = key0 + lane % KEYS, jc = j < S ? j : S - 1;
    for (int t = GRAN * jt + wave; t < end; t += 4) {
        float s = 0.f, dc = 0.f;
        for (int u = 0; u < D; u++) {
            s += Q[(size_t)t * rsA + u] * K[(size_t)jc * rsA + u];
            dc += dH[(size_t)t * rsB + u] * V[(size_t)jc * rsA + u];
        }
        const float ct = s * fast_exp2(a.alpha2[poff + j] + gate(t)), dd = ct * (dc * a.inv_n[poff + t] + a.db[poff + t]);
        const float sum = wave_reduce<OpAdd>(lane < KEYS && j <= t ? dd : 0.f);
        if (lane == 0) slice[t] = sum;
    }
}

}  // namespace mlstm
