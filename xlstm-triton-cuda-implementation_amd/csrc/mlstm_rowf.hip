// Row kernel of the fp32 tensors where few workgroups would run: the math of mlstm_row.hip and its order of operations, hence its
// bits, on 32 rows per workgroup with the work on them spread over four waves.
//
// In row_kernel a wave owns 32 rows outright: at D = 128, in chunks of 128 positions, up to 576 products of 32 cycles one after the
// other (the terms' six per 16 elements), between waits for tiles that its workgroup's four waves share.  Nothing but the accumulation
// over the keys is a chain, so here
//   phase 1   wave w = key block:      S^T = K Q^T (dQ pass: dC^T = V dH^T) of its 32 keys, gate weights, the weights' terms to LDS;
//   phase 2   wave w = column block:   H^T += V^T P^T (dQ^T += K^T G^T) of its 32 columns over the 128 keys.
// In phase 2, and for the state of the previous chunk before it, a wave reads only its own 32 columns: those come straight into
// registers, a dword per lane and row in whole 128-byte lines.  They, the rows' own operand and the keys of phase 1 (into LDS, a block
// per wave) are all requested in the first instructions of the kernel: one trip to memory per 128 keys.  (Through LDS instead, the
// state first and V into its place behind it: 17.5 us where this takes 15.5, B2 H4 S1000 D128.)
// (D = 64: waves 0 and 1 have the two column blocks.)
#include <type_traits>
#include "mlstm_device.h"
#include "mlstm_kernels.h"
#include "mlstm_row_exact.h"

namespace mlstm {

template <int D>
struct RowfCfg {
    static constexpr int ROWS = 32, KEYS = 128;
    static constexpr size_t X_BYTES = (size_t)ROWS * D * 4, K_BYTES = (size_t)KEYS * D * 4;
    static constexpr size_t P_BYTES = 4 * 2 * 3 * 64 * 16;   // [key block][16 keys][term][lane] x 16 B
    static constexpr size_t HAND_BYTES = 2 * 16 * 64 * 8;     // forward: [key block of the rows' granule][register][lane] x {product, weight}
    static constexpr size_t LDS_BYTES = X_BYTES + K_BYTES + P_BYTES + HAND_BYTES + (4 * 64 * 2 + 32 * 2 + 4 * 64 + 4 + D) * sizeof(float);
};

template <int D, int MODE>
__global__ __launch_bounds__(256, 1) void rowf_kernel(RowArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    using T = float;
    using R = Tr<float>;
    using Cfg = RowfCfg<D>;
    typedef R::frag frag;
    constexpr int KW = R::KW, NS = D / KW, NCB = D / 32;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    T* const xtile = reinterpret_cast<T*>(smem);
    char* const pbuf = smem + Cfg::X_BYTES + Cfg::K_BYTES;
    float2* const hand = reinterpret_cast<float2*>(pbuf + Cfg::P_BYTES);
    float* const part = reinterpret_cast<float*>(pbuf + Cfg::P_BYTES + Cfg::HAND_BYTES);   // [key block][lane] x {sum, row factor}
    float* const stat = part + 4 * 64 * 2;                               // [row] x {1/n, db}; then (forward) {1/n, b}
    float* const rix = stat + 32 * 2;                                    // [column block][lane]
    unsigned* const bads = reinterpret_cast<unsigned*>(rix + 4 * 64);    // [wave]
    float* const nvl = reinterpret_cast<float*>(bads + 4);               // [D] the previous chunk's vector state

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, c32 = lane & 31;
    int S = a.S, bh, rt;
    {
        const int bid = blockIdx.x, nT = 2 * a.NG;   // (the rows behind the sequence in its last granule have a tile too) heaviest row tiles first; with a multiple of 8 heads a head's tiles on one XCD
        if ((a.BH & 7) == 0) {
            const int rest = bid >> 3, ngrp = a.BH >> 3;
            bh = (rest % ngrp) * 8 + (bid & 7);
            rt = nT - 1 - rest / ngrp;
        } else {
            bh = bid % a.BH;
            rt = nT - 1 - bid / a.BH;
        }
    }
    size_t hoff = (size_t)bh * S, poff = (size_t)bh * a.NG * GRAN, goff = (size_t)bh * a.NG;
    const size_t rsA = (size_t)a.la.ss, rsB = (size_t)a.lb.ss, rsH = (size_t)a.lh.ss;
    size_t offA = a.la.head(bh), offB = a.lb.head(bh), offH = a.lh.head(bh);
    int chunk = 0;   // in chunks positions count from the chunk's first one (see mlstm_row.hip)
    if (a.chunk_len > 0) {
        chunk = (rt * 32) / a.chunk_len;
        const int p0 = chunk * a.chunk_len;
        hoff += p0; poff += p0; goff += p0 / GRAN;
        offA += (size_t)p0 * rsA; offB += (size_t)p0 * rsB; offH += (size_t)p0 * rsH;
        S -= p0; rt -= p0 / 32;
    }
    const int r0 = 32 * rt, row = r0 + c32, rowc = row < S ? row : S - 1;
    if (r0 >= S) {   // (uniform over the workgroup)
        if (MODE == ROW_MODE_DQ && tid < 32) { a.inv_n[poff + row] = 0.f; a.db[poff + row] = 0.f; }   // see mlstm_row.hip
        return;
    }
    const int nkb = rt + 1, nR = (nkb + 3) / 4;   // key blocks of 32 at or before the rows; rounds of four
    const size_t rsX = MODE == ROW_MODE_FWD ? rsA : rsB, offX = MODE == ROW_MODE_FWD ? offA : offB;
    const size_t rsO = MODE == ROW_MODE_FWD ? rsB : rsA, offO = MODE == ROW_MODE_FWD ? offB : offA;
    const T* X = reinterpret_cast<const T*>(a.X) + offX;
    const T* Y1 = reinterpret_cast<const T*>(a.Y1) + offA;
    const T* Y2 = reinterpret_cast<const T*>(a.Y2) + offA;
    const bool second = wave < NCB;   // the wave has a column block
    constexpr int SUMS = 3;           // the wave of the row sums (D = 64: it has none)
    const int col = 32 * wave + c32;

    // ---- requests: the rows' operand, the wave's first key block, its columns of the state and of the first keys
    const float beta_row = a.beta2[poff + rowc], beta_end = chunk > 0 ? a.beta2[poff - 1] : 0.f;
    const double g_row = a.G2[goff + r0 / GRAN], g_end = chunk > 0 ? a.G2[goff - 1] : 0.0;
    {
        TileDma<T, D, 32, 256> xd;
        xd.init(tid);
        if (r0 + 32 <= S) xd.issue(xtile, X + (size_t)r0 * rsX, xd.rows(tid, (unsigned)(rsX * sizeof(T))));
        else tile_dma_rolled<T, D, 32, 256>(xtile, X, r0, S, tid, rsX);
    }
    TileDma<T, D, 32, 64> kd;
    kd.init(lane);
    const auto kr = kd.rows(lane, (unsigned)(rsA * sizeof(T)));
    T* const ktile = reinterpret_cast<T*>(smem + Cfg::X_BYTES + (size_t)wave * 32 * D * sizeof(T));
    auto copy_k = [&](int kb) {
        if (32 * kb + 32 <= S) kd.issue(ktile, Y1 + (size_t)(32 * kb) * rsA, kr);
        else tile_dma_rolled<T, D, 32, 64>(ktile, Y1, 32 * kb, S, lane, rsA);
    };
    if (wave < nkb) copy_k(wave);
    // element e of group g of the wave's columns: row 16 g + 8 (e / 4) + 4 h + e % 4 (the order of Tr::from_acc)
    frag cf[NS];
    const T* const Cst = chunk > 0 ? reinterpret_cast<const T*>(a.Cst) + ((size_t)bh * a.n_states + chunk - 1) * D * D : nullptr;
    if (second && chunk > 0) {
#pragma unroll
        for (int g = 0; g < NS; g++)
#pragma unroll
            for (int e = 0; e < 8; e++) cf[g][e] = Cst[(size_t)(16 * g + 8 * (e >> 2) + 4 * h + (e & 3)) * D + col];
    }
    frag vf[8];
    auto load_v = [&](int r) __attribute__((always_inline)) {   // rows past the rows' own block are not used, past the end clamped
        const int k0 = 128 * r;
        const unsigned lane_off = (unsigned)(4 * h * rsA) + col;
#pragma unroll
        for (int g = 0; g < 8; g++) {
            if (k0 + 16 * g + 16 <= S) {
                const T* p = Y2 + (size_t)(k0 + 16 * g) * rsA;
#pragma unroll
                for (int e = 0; e < 8; e++) vf[g][e] = (p + (size_t)(8 * (e >> 2) + (e & 3)) * rsA)[lane_off];
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int pos = k0 + 16 * g + 8 * (e >> 2) + 4 * h + (e & 3);
                    vf[g][e] = Y2[(size_t)(pos < S ? pos : S - 1) * rsA + col];
                }
            }
        }
    };
    if (second) load_v(0);
    const float m_row = a.M[hoff + rowc];
    if (chunk > 0 && tid < D) nvl[tid] = a.Nst[((size_t)bh * a.n_states + chunk - 1) * D + tid];
    const float nbeta = -beta_row;
    constexpr double LOG2_SCALE = D == 64 ? -3.0 : -3.5;
    float dec = 0.f;
    if (chunk > 0) dec = fast_exp2(beta_end - beta_row + (float)(g_row - g_end));
    dma_wait();
    __syncthreads();   // the rows' operand is there
    SwzRowReader<T, D> rrd;
    rrd.init(lane);
    frag xf[NS];
    typename R::terms xt[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) { xf[s] = rrd.read(xtile, 0, s); xt[s] = R::split(xf[s]); }
    float inv_n = 0.f, dbv = 0.f;
    if constexpr (MODE == ROW_MODE_DQ) {
        if (wave == 3) {
            row_stats<T, NS>(xf, reinterpret_cast<const T*>(a.Hin) + offH + (size_t)rowc * rsH, h, a.Bin[hoff + rowc], m_row, inv_n, dbv, nullptr);
            if (h == 0) {
                *reinterpret_cast<float2*>(stat + 2 * c32) = make_float2(inv_n, dbv);
                a.inv_n[poff + row] = row < S ? inv_n : 0.f;   // (rows behind the sequence: zeros, see mlstm_row.hip)
                a.db[poff + row] = row < S ? dbv : 0.f;
            }
        }
        __syncthreads();
        const float2 st = *reinterpret_cast<const float2*>(stat + 2 * c32);
        inv_n = st.x; dbv = st.y;
    }
    f32x16 acc;
#pragma unroll
    for (int x = 0; x < 16; x++) acc[x] = 0.f;
    float bsum = 0.f;
    if (chunk > 0) {
        if (second) {
            R::template stream<NS>([&](auto n) { return cf[n]; },
                                   [&](auto n, const auto& c, auto&& between) { R::mma_between(acc, c, xt[n], between); });
        }
        if constexpr (MODE == ROW_MODE_FWD) {
            if (wave == SUMS) {
                float pt = 0.f;
#pragma unroll
                for (int s = 0; s < NS; s++)
#pragma unroll
                    for (int e = 0; e < R::EPL; e++) pt = fmaf(xf[s][e], nvl[KW * s + R::EPL * h + e], pt);
                bsum = fmaf(dec, pt, bsum);
            }
#pragma unroll
            for (int x = 0; x < 16; x++) acc[x] *= dec;
        } else if (second) {
            const float decn = dec * inv_n, rank1 = dec * dbv;
            const T* qrow = reinterpret_cast<const T*>(a.Qrow) + offA + (size_t)rowc * rsA;
            float rp = 0.f;
#pragma unroll
            for (int a4 = 0; a4 < 4; a4++) {
                const int c0 = 32 * wave + 8 * a4 + 4 * h;
                const f32x4 nv = *reinterpret_cast<const f32x4*>(nvl + c0), qv = *reinterpret_cast<const f32x4*>(qrow + c0);
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    acc[4 * a4 + c] = fmaf(rank1, nv[c], acc[4 * a4 + c] * decn);
                    rp = fmaf(acc[4 * a4 + c], qv[c], rp);
                }
            }
            rix[wave * 64 + lane] = rp;
        }
    }
    // ---- the keys, 128 at a time
    for (int r = 0; r < nR; r++) {
        const int kb = 4 * r + wave;
        if (r > 0) __syncthreads();   // phase 2 of the previous round is done with the weights
        if (kb < nkb) {
            const int k0 = 32 * kb;
            const bool fact = k0 / GRAN < r0 / GRAN;   // (row_kernel: factorised weights in the tiles of 64 keys before the rows' own)
            const double crow = LOG2_SCALE + (g_row - a.G2[goff + k0 / GRAN]);
            const float am = a.amax2[goff * 2 + kb];
            f32x4 wk[4];
#pragma unroll
            for (int a4 = 0; a4 < 4; a4++) wk[a4] = *reinterpret_cast<const f32x4*>((fact ? a.ek2 : a.alpha2) + poff + k0 + 8 * a4 + 4 * h);
            f32x16 s = {}, small = {};
            if (r > 0) dma_wait();   // (the wave's own copy)
            R::template stream<NS>([&](auto n) { return rrd.read(ktile, 0, n); },
                                   [&](auto n, const auto& kf, auto&& between) { R::mma_between(s, small, kf, xt[n], between); });
            s += small;
            if (kb + 4 < nkb) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the block's reads are over: the copies' instructions say nothing of memory)
                copy_k(kb + 4);
            }
            float blk = 0.f, er = 1.f;
            if (fact) {
                er = fast_exp2((float)((double)(am + nbeta) + crow));
#pragma unroll
                for (int x = 0; x < 16; x++) {
                    const float ek = wk[x >> 2][x & 3];
                    if constexpr (MODE == ROW_MODE_FWD) {
                        blk = fmaf(s[x], ek, blk);
                        s[x] = (s[x] * ek) * er;
                    } else {
                        s[x] = (s[x] * inv_n + dbv) * (ek * er);
                    }
                }
            } else {
#pragma unroll
                for (int x = 0; x < 16; x++) {
                    float e = fast_exp2((wk[x >> 2][x & 3] + nbeta) + (float)crow);
                    if (k0 == r0 && 8 * (x >> 2) + 4 * h + (x & 3) > c32) e = 0.f;
                    if constexpr (MODE == ROW_MODE_FWD) {
                        hand[((kb & 1) * 16 + x) * 64 + lane] = make_float2(s[x], e);
                        s[x] *= e;
                    } else {
                        s[x] = (s[x] * inv_n + dbv) * e;
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const typename R::terms p = R::split(R::from_acc(s, t));
                bf16x8* dst = reinterpret_cast<bf16x8*>(pbuf) + (wave * 2 + t) * 3 * 64 + lane;
                dst[0] = p.hi; dst[64] = p.mid; dst[128] = p.lo;
            }
            if constexpr (MODE == ROW_MODE_FWD) *reinterpret_cast<float2*>(part + (wave * 64 + lane) * 2) = make_float2(blk, er);
        }
        __syncthreads();
        const int nb = nkb - 4 * r < 4 ? nkb - 4 * r : 4;   // key blocks of this round
        float2 be[4], own[32];
        if constexpr (MODE == ROW_MODE_FWD) {
            if (wave == SUMS) {   // (requested ahead of the products, added up behind them)
#pragma unroll
                for (int t = 0; t < 4; t++) be[t] = *reinterpret_cast<const float2*>(part + (t * 64 + lane) * 2);
                if (r == nR - 1) {
#pragma unroll
                    for (int x = 0; x < 32; x++) own[x] = hand[x * 64 + lane];
                }
            }
        }
        if (second) {
            const bf16x8* p = reinterpret_cast<const bf16x8*>(pbuf) + lane;
            auto products = [&](auto groups_tag) __attribute__((always_inline)) {
                R::template stream<decltype(groups_tag)::value>([&](auto n) { return vf[n]; }, [&](auto n, const auto& v, auto&& between) {
                    const typename R::terms w = {p[(3 * n) * 64], p[(3 * n + 1) * 64], p[(3 * n + 2) * 64]};
                    R::mma_between(acc, v, w, between);
                });
            };
            switch (nb) {
                case 1: products(std::integral_constant<int, 2>{}); break;
                case 2: products(std::integral_constant<int, 4>{}); break;
                case 3: products(std::integral_constant<int, 6>{}); break;
                default: products(std::integral_constant<int, 8>{});
            }
            if (r + 1 < nR) load_v(r + 1);
        }
        if constexpr (MODE == ROW_MODE_FWD) {
            if (wave == SUMS) {
                const int before = r0 / GRAN * 2 - 4 * r;   // the round's key blocks before the rows' own granule
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    if (t < before) bsum = fmaf(be[t].x, be[t].y, bsum);
                }
                // the own granule's element by element onto the sum over the keys before it, as a wave of row_kernel does that holds all of them
                if (r == nR - 1) {
#pragma unroll
                    for (int x = 0; x < 16; x++) bsum = fmaf(own[x].x, own[x].y, bsum);
                    if (rt & 1) {
#pragma unroll
                        for (int x = 16; x < 32; x++) bsum = fmaf(own[x].x, own[x].y, bsum);
                    }
                }
            }
        }
    }
    // ---- epilogue: the normaliser, rows that are not finite from their definition (see not_finite), the wave's columns
    float seen = 0.f;
    if (MODE == ROW_MODE_FWD && wave == SUMS) {
        const float b = sum_halves(bsum);
        seen = not_finite(seen, b);
        const float n = fmaxf(fabsf(b), __expf(-m_row)) + 1e-6f;
        if (h == 0) *reinterpret_cast<float2*>(stat + 2 * c32) = make_float2(1.0f / n, b);
    }
#pragma unroll
    for (int x = 0; x < 16; x++) seen = not_finite(seen, acc[x]);
    {
        const unsigned long long halves = __ballot((second || wave == SUMS) && row < S && seen != 0.f);
        if (lane == 0) bads[wave] = (unsigned)halves | (unsigned)(halves >> 32);
    }
    __syncthreads();
    const unsigned bad = bads[0] | bads[1] | bads[2] | bads[3];
    const bool mine = row < S && !((bad >> c32) & 1);
    float onorm = 1.0f;
    if constexpr (MODE == ROW_MODE_FWD) {
        const float2 st = *reinterpret_cast<const float2*>(stat + 2 * c32);
        onorm = st.x;
        if (mine && wave == 0 && h == 0) a.Bsum[hoff + row] = st.y;
    } else {
        if (a.chunk_len > 0 && wave == 0) {
            float rp = 0.f;
            if (chunk > 0) {
#pragma unroll
                for (int d = 0; d < NCB; d++) rp += rix[d * 64 + lane];
                rp = sum_halves(rp);
            }
            if ((mine || (chunk == 0 && row < S)) && h == 0) a.rowinter[hoff + row] = rp;
        }
    }
    if (second && mine) {
        T* out = reinterpret_cast<T*>(a.out) + offO + (size_t)row * rsO;
#pragma unroll
        for (int a4 = 0; a4 < 4; a4++) {
            const int c0 = 32 * wave + 8 * a4 + 4 * h;
            f32x4 v;
#pragma unroll
            for (int c = 0; c < 4; c++) v[c] = acc[4 * a4 + c] * onorm;
            *reinterpret_cast<f32x4*>(out + c0) = v;
            if constexpr (MODE == ROW_MODE_FWD) {
                if (a.O) {
                    const f32x4 o = *reinterpret_cast<const f32x4*>(reinterpret_cast<const T*>(a.O) + offB + (size_t)row * rsB + c0);
                    f32x4 g;
#pragma unroll
                    for (int c = 0; c < 4; c++) g[c] = v[c] * silu(o[c]);
                    *reinterpret_cast<f32x4*>(reinterpret_cast<T*>(a.out_gated) + offB + (size_t)row * rsB + c0) = g;
                }
            }
        }
    }
    for (unsigned rest = bad; rest; rest &= rest - 1) {
        const int b = __builtin_ctz(rest);
        if ((b & 3) != wave) continue;
        row_exact<D, MODE>(a, bh, chunk, r0 + b, S, hoff, poff, goff, X + (size_t)(r0 + b) * rsX, Y1, Y2, rsA, offA, offO, offB, rsO, rsB,
                           __shfl(inv_n, b), __shfl(dbv, b));
    }
#endif
}

template <int D, int MODE>
static int launch_rowf_t(const RowArgs& a, hipStream_t st) {
    if (hipError_t e = lds_limit_once<rowf_kernel<D, MODE>>((int)RowfCfg<D>::LDS_BYTES); e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((rowf_kernel<D, MODE>), dim3(a.BH * a.NG * 2), dim3(256), RowfCfg<D>::LDS_BYTES, st, a);
    return (int)hipGetLastError();
}

int launch_rowf_kernel(int mode, int D, const RowArgs& a, hipStream_t st) {
    if (mode == ROW_MODE_FWD) return D == 64 ? launch_rowf_t<64, ROW_MODE_FWD>(a, st) : launch_rowf_t<128, ROW_MODE_FWD>(a, st);
    return D == 64 ? launch_rowf_t<64, ROW_MODE_DQ>(a, st) : launch_rowf_t<128, ROW_MODE_DQ>(a, st);
}

}  // namespace mlstm
