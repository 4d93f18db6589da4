// Column-parallel backward kernel for the 16-bit types at D = 128 and 256 where few workgroups would run: the same products and,
// element by element, the same order of operations as mlstm_cold.hip, hence the same bits, on half as many keys per workgroup and
// with the work on a query tile spread over eight waves.
//
// What bounds a small call is one workgroup's walk of its query tiles, and a cold_kernel wave takes 1.6 us per 32 queries (2 D / 16
// products, sixteen elements per lane, 2 D / 16 products, one after the other, alone on its SIMD) whatever the number of
// workgroups.  A workgroup here owns 64 keys; its walk is a pipeline of 32-query tiles with one barrier per tile:
//   step v      two producer waves (one per 32 keys) form S = Q K^T and dC = dH V^T of tile v, K and V in their registers;
//   step v + 1  they weigh the elements and leave G and W, the row sums and the column sums in LDS, while the other two producers are
//               at the products of tile v + 1;
//   step v + 2  four consumer waves, one per output and 32 keys, add dK^T += Q^T G or dV^T += dH^T W.
// So every SIMD has one wave of either kind, and the element-wise part runs beside products.  In chunks the chunk's reverse state
// goes first, through two of the tiles' slots.  15 heads x 1001 x 128 (fp16): 56 -> 30 us, 1700 cycles per tile, of which the weighing wave
// needs 1300; 8 x 1500 x 256 in split mode: 66 -> 44.  cold_kernel serves larger launches: it reads Q and dH half as often and pays for a
// prologue (3 us) and an epilogue half as often.
// Replaces, like mlstm_cold.hip, the dK/dV/dI loop of mlstm_matmul_kernel_backward (mlstm_matmul.py:269-316).
#include <type_traits>
#include "mlstm_device.h"
#include "mlstm_kernels.h"

namespace mlstm {

constexpr int CW_QT = 32;                // queries per tile

template <typename T, int D, bool STRICT>
struct ColwCfg {
    static constexpr size_t QT_BYTES = (size_t)CW_QT * D * sizeof(T), SLOT_BYTES = 2 * QT_BYTES;   // a tile of Q, one of dH
    static constexpr int NSLOT = D == 128 ? 8 : 4, AHEAD = NSLOT - 3;   // tiles from memory ahead of the products
    static constexpr size_t POOL_BYTES = NSLOT * SLOT_BYTES;
    static constexpr size_t HALF_BYTES = (STRICT ? 4 : 2) * 64 * 16;   // 16 queries x 32 keys of G and W (then their low-order terms)
    static constexpr int PBUF = STRICT ? 1 : 2;                        // (twice 16 KB and the slots are all of LDS)
    static constexpr size_t P_BYTES = PBUF * 4 * HALF_BYTES;
    static constexpr int E_ROWS = STRICT ? 32 : 64, NE = D / E_ROWS;   // the state in pieces of a slot (split mode: hi, then lo)
    static constexpr size_t MISC_FLOATS = 2 * 2 * 32 + 2 * 64 + D;   // row sums, column sums, the vector state
    static size_t lds_bytes(int granules) { return POOL_BYTES + P_BYTES + (MISC_FLOATS + (size_t)granules * (3 * GRAN + 1)) * sizeof(float); }
};

template <typename T, int D, bool STRICT>
__global__ __launch_bounds__(512) void colw_kernel(ColArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    using R = Tr<T>;
    using Cfg = ColwCfg<T, D, STRICT>;
    using Z = Swz<T, D>;
    typedef typename R::frag frag;
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    static_assert(R::HALF && (D == 128 || D == 256), "16-bit types, D = 128 or 256");
    constexpr int KW = R::KW, NS = D / KW, NXD = D / 32, NSLOT = Cfg::NSLOT, AHEAD = Cfg::AHEAD;
    constexpr bool END_SCALE = std::is_same<T, __bf16>::value;                // (see mlstm_cold.hip)
    extern __shared__ __attribute__((aligned(16))) char smem[];
    char* const pbuf = smem + Cfg::POOL_BYTES;                                // [buffer][key block][half]
    float* const rowtmp = reinterpret_cast<float*>(pbuf + Cfg::P_BYTES);      // [tile parity][key block][32]
    float* const colp = rowtmp + 2 * 2 * 32;                                  // [key block][lane]: the column sums so far
    float* const gvl = colp + 2 * 64;                                         // [D] the chunk's vector state g
    float* const rowvec = gvl + D;                                            // [granule][beta, 1/n, db][64] of the queries

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, c32 = lane & 31;
    const bool producer = wave < 4;
    const int kb = wave & 1, role = (wave >> 1) & 1;   // role: a producer's pair; a consumer's output (0: dK, 1: dV)
    const int S = a.S, NG = a.NG;
    int bh, jt;
    {
        // heaviest first: the first keys of their chunk (or of the sequence); with a multiple of 8 heads a head's tiles run on one XCD
        const int tpc = a.chunk_len > 0 ? a.chunk_len / GRAN : NG, nch = (NG + tpc - 1) / tpc;
        const int ngrp = (a.BH & 7) == 0 ? a.BH >> 3 : a.BH;
        const int rest = (a.BH & 7) == 0 ? (int)blockIdx.x >> 3 : (int)blockIdx.x;
        const int g = rest % ngrp, tile = rest / ngrp;                        // tile: over the chunks' first tiles, then their second ones ...
        bh = (a.BH & 7) == 0 ? 8 * g + (blockIdx.x & 7) : g;
        const int last = NG - (nch - 1) * tpc;                                // tiles of the last chunk: classes below `last` have nch of them
        const int head_n = last * nch;
        if (tile < head_n) jt = (tile % nch) * tpc + tile / nch;
        else jt = ((tile - head_n) % (nch - 1)) * tpc + last + (tile - head_n) / (nch - 1);
    }
    const size_t hoff = (size_t)bh * S, poff = (size_t)bh * NG * GRAN, goff = (size_t)bh * NG;
    const size_t rsA = (size_t)a.la.ss, rsB = (size_t)a.lb.ss, offA = a.la.head(bh), offB = a.lb.head(bh);
    const T* Q = reinterpret_cast<const T*>(a.Q) + offA;
    const T* dH = reinterpret_cast<const T*>(a.dH) + offB;
    const T* K = reinterpret_cast<const T*>(a.K) + offA;
    const T* V = reinterpret_cast<const T*>(a.V) + offA;
    const int key = GRAN * jt + 32 * kb + c32;
    const int chunk = a.chunk_len > 0 ? jt / (a.chunk_len / GRAN) : 0;
    const int jq_end = a.chunk_len > 0 && (chunk + 1) * (a.chunk_len / GRAN) < NG ? (chunk + 1) * (a.chunk_len / GRAN) : NG;
    const int nG = jq_end - jt;                                               // granules of queries, the keys' own first
    const int NQ = (S + CW_QT - 1) / CW_QT;                                   // 32-query tiles of the sequence
    const int it0 = 2 * jt, NT = (2 * jq_end < NQ ? 2 * jq_end : NQ) - it0;   // tiles of the walk: it0 + v, v < NT
    const int full_q = S / CW_QT;
    const bool has_state = a.chunk_len > 0 && chunk < a.n_states;
    float* const sG = rowvec + (size_t)nG * 3 * GRAN;                         // granule bases of the queries minus the first one's

    // Slots: K and V in 0 and 1 until the tiles get there, the state's pieces in turns in 2 and 3, tile v in (2 + v) % NSLOT
    auto slot_at = [&](int n) { return reinterpret_cast<T*>(smem + (size_t)n * Cfg::SLOT_BYTES); };
    auto q_at = [&](int v) { return slot_at((v + 2) & (NSLOT - 1)); };
    auto dh_at = [&](int v) { return reinterpret_cast<T*>(smem + (size_t)((v + 2) & (NSLOT - 1)) * Cfg::SLOT_BYTES + Cfg::QT_BYTES); };
    // a tile's copy by the consumers, in pieces that go between their products
    typedef TileDma<T, D, CW_QT, 256> Tile;
    constexpr int PW = Tile::PER_WAVE;
    const int tidc = tid & 255;
    Tile tdma;
    tdma.init(tidc);
    const auto ra = tdma.rows(tidc, (unsigned)(rsA * sizeof(T))), rb = tdma.rows(tidc, (unsigned)(rsB * sizeof(T)));
    auto copy_piece = [&](int v, int n) {   // piece n < 2 PW of a tile whose rows all exist
        if (n < PW) tdma.issue_range(q_at(v), Q + (size_t)CW_QT * (it0 + v) * rsA, n, n + 1, ra);
        else tdma.issue_range(dh_at(v), dH + (size_t)CW_QT * (it0 + v) * rsB, n - PW, n - PW + 1, rb);
    };
    auto copy_tile = [&](int v) {
        if (it0 + v < full_q) {
            tdma.issue(q_at(v), Q + (size_t)CW_QT * (it0 + v) * rsA, ra);
            tdma.issue(dh_at(v), dH + (size_t)CW_QT * (it0 + v) * rsB, rb);
        } else {
            tile_dma_rolled<T, D, CW_QT, 256>(q_at(v), Q, CW_QT * (it0 + v), S, tidc, rsA);
            tile_dma_rolled<T, D, CW_QT, 256>(dh_at(v), dH, CW_QT * (it0 + v), S, tidc, rsB);
        }
    };

    // ---- prologue: everything that does not depend on anything is requested at once.  K and V come as whole rows (as fragments straight
    // from memory, 16 bytes of a row per lane, the loads of eight waves took 4 us)
    const size_t sbase = has_state ? ((size_t)bh * a.n_states + chunk) * D * D : 0;
    const T* const Eh = reinterpret_cast<const T*>(a.Ev) + sbase;
    const T* const El = STRICT ? reinterpret_cast<const T*>(a.Ev_lo) + sbase : nullptr;
    TileDma<T, D, GRAN, 512> sdma;
    sdma.init(tid);
    TileDma<T, D, Cfg::E_ROWS, 512> edma;
    edma.init(tid);
    auto e_hi = [&](int n) { return slot_at(2 + (n & 1)); };
    auto e_lo = [&](int n) { return slot_at(2 + (n & 1)) + Cfg::E_ROWS * D; };
    auto piece = [&](int n) {   // the state's piece n, or what follows the last one
        if (n < Cfg::NE) {
            edma.issue(e_hi(n), Eh + (size_t)Cfg::E_ROWS * n * D);
            if constexpr (STRICT) edma.issue(e_lo(n), El + (size_t)Cfg::E_ROWS * n * D);
        } else if (n == Cfg::NE && !producer) {
            copy_tile(0);
        }
    };
    static_assert(Cfg::NE % 2 == 0, "tile 0 takes slot 2 behind the last but one piece");
    {
        const auto rk = sdma.rows(tid, (unsigned)(rsA * sizeof(T)));
        if (GRAN * (jt + 1) <= S) {
            sdma.issue(slot_at(0), K + (size_t)GRAN * jt * rsA, rk);
            sdma.issue(slot_at(1), V + (size_t)GRAN * jt * rsA, rk);
        } else {
            tile_dma_rolled<T, D, GRAN, 512>(slot_at(0), K, GRAN * jt, S, tid, rsA);
            tile_dma_rolled<T, D, GRAN, 512>(slot_at(1), V, GRAN * jt, S, tid, rsA);
        }
    }
    if (has_state) { piece(0); piece(1); }
    else if (!producer) copy_tile(0);
    for (int g = wave; g < 3 * nG; g += 8) {   // (padded arrays: always readable)
        const float* src = (g % 3 == 0 ? a.beta2 : (g % 3 == 1 ? a.inv_n : a.db)) + poff + GRAN * (jt + g / 3) + lane;
        dma4(src, __builtin_amdgcn_readfirstlane(lds_offset_of(rowvec + g * GRAN)));
    }
    const int pe = has_state ? (chunk + 1) * a.chunk_len - 1 : 0;   // the chunk's last position
    const double gbase = a.G2[goff + (jt & ~1)], gkey = a.G2[goff + jt];
    const float bend = a.beta2[poff + pe];
    const double Gend = a.G2[goff + pe / GRAN];
    const float al = key < S ? a.alpha2[poff + key] : -INFINITY;    // (a key past the end weighs nothing)
    for (int g = tid; g < nG; g += 512) sG[g] = (float)(a.G2[goff + jt + g] - gbase);
    if (has_state && tid < D) gvl[tid] = a.gvec[((size_t)bh * a.n_states + chunk) * D + tid];
    const float gcorr = (float)(gbase - gkey), log2scale = -0.5f * __log2f((float)D);
    float scale_s = 1.f, log2_s = 0.f, wkg = 0.f, wk = 0.f;   // (see mlstm_cold.hip)
    bool use = true;
    if (has_state) {
        wk = fast_exp2(al - bend + (float)(Gend - gkey));
        use = !END_SCALE || wk > 0x1p-40f;
        if constexpr (END_SCALE) {
            if (use) { scale_s = wk; log2_s = al - bend + (float)(Gend - gkey); }
            wkg = wk;
        }
    }
    dma_wait();
    __syncthreads();
    const int n_steps = NT + 2;
    SwzRowReaderX<T, D> rrd;
    rrd.init(lane);

    if (producer) {
        frag kf[NS], vf[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) { kf[s] = rrd.read(slot_at(0), kb, s); vf[s] = rrd.read(slot_at(1), kb, s); }
#pragma unroll
        for (int s = 0; s < NS; s++) { pin(kf[s]); pin(vf[s]); }
        if (has_state)
            for (int n = 0; n < Cfg::NE; n++) {
                dma_wait();
                __syncthreads();
                piece(n + 2);
            }
        f32x16 wacc, gacc;   // S, then W;  dC, then G
        const int key0 = GRAN * jt + 32 * kb;
        auto active = [&](int v) { return !(v == 0 && kb > 0); };   // (tile 0 lies before the second 32 keys)
        float wt[16];        // the elements' weights E, formed beside the products
        auto products = [&](int v, auto masked_tag) __attribute__((always_inline)) {
            constexpr bool MASKED = decltype(masked_tag)::value;   // a tile on the diagonal, or one that the sequence ends in
            const float argbase = al + (sG[v >> 1] + gcorr + log2scale) - log2_s;
            const float* const srow = rowvec + (v >> 1) * 3 * GRAN + 32 * (v & 1) + 4 * h;
            const unsigned span = (unsigned)(S - key);             // query q takes part iff 0 <= q - key < S - key (unsigned compare)
            const int dq0 = CW_QT * (it0 + v) + 4 * h - key;
            const T* const qt = q_at(v);
            const T* const ht = dh_at(v);
            constexpr int PRE = 3;
            frag qf[NS], hf[NS];
#pragma unroll
            for (int s = 0; s < PRE; s++) { qf[s] = rrd.read(qt, 0, s); hf[s] = rrd.read(ht, 0, s); }
#pragma unroll
            for (int x = 0; x < 16; x++) { wacc[x] = 0.f; gacc[x] = 0.f; }
#pragma unroll
            for (int s = 0; s < NS; s++) {
                if (s + PRE < NS) { qf[s + PRE] = rrd.read(qt, 0, s + PRE); hf[s + PRE] = rrd.read(ht, 0, s + PRE); }
                R::mma(wacc, qf[s], kf[s]);
                R::mma(gacc, hf[s], vf[s]);
                if (s % (NS / 4) == 1) {
                    const int a4 = s / (NS / 4);
                    const f32x4 beta4 = *reinterpret_cast<const f32x4*>(srow + 8 * a4);
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        float arg = argbase - beta4[c];
                        if constexpr (MASKED) arg = (unsigned)(dq0 + 8 * a4 + c) < span ? arg : -INFINITY;
                        wt[4 * a4 + c] = fast_exp2(arg);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto hand_over = [&](int v, const f32x4 (&inv4)[4]) __attribute__((always_inline)) {
            char* const block = pbuf + (size_t)((Cfg::PBUF == 2 ? (v & 1) * 2 : 0) + kb) * 2 * Cfg::HALF_BYTES;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                frag* const out = reinterpret_cast<frag*>(block + t * Cfg::HALF_BYTES) + lane;
                if constexpr (STRICT) {
                    // (the low-order terms take what rounding the products would lose)
                    typename R::vec4 hi[2], lo[2];
                    auto terms = [](const typename R::vec4 (&x)[2]) { return __builtin_shufflevector(x[0], x[1], 0, 1, 2, 3, 4, 5, 6, 7); };
                    auto four = [&](const auto& x, int a4) { return f32x4{x[4 * a4], x[4 * a4 + 1], x[4 * a4 + 2], x[4 * a4 + 3]}; };
#pragma unroll
                    for (int u = 0; u < 2; u++) R::split_products(four(gacc, 2 * t + u), four(wt, 2 * t + u), hi[u], lo[u]);
                    out[0] = terms(hi); out[128] = terms(lo);
#pragma unroll
                    for (int u = 0; u < 2; u++) R::split_products(four(wacc, 2 * t + u), inv4[2 * t + u], hi[u], lo[u]);
                    out[64] = terms(hi); out[192] = terms(lo);
                } else {
                    out[0] = R::from_acc(gacc, t);
                    out[64] = R::from_acc(wacc, t);
                }
            }
        };
        const bool hi1 = lane & 1, hi2 = lane & 2;
        auto weigh = [&](int v) __attribute__((always_inline)) {
            const float* const srow = rowvec + (v >> 1) * 3 * GRAN + 32 * (v & 1) + 4 * h;
            f32x4 inv4[4], db4[4];   // 1/n and db of the tile's queries
#pragma unroll
            for (int a4 = 0; a4 < 4; a4++) {
                inv4[a4] = *reinterpret_cast<const f32x4*>(srow + GRAN + 8 * a4);
                db4[a4] = *reinterpret_cast<const f32x4*>(srow + 2 * GRAN + 8 * a4);
            }
            float dd[16], colsum = colp[kb * 64 + lane];   // (one sum over all queries, as a wave of cold_kernel keeps it: from weighing wave to weighing wave)
#pragma unroll
            for (int a4 = 0; a4 < 4; a4++) {
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const int r = 4 * a4 + c;
                    const float e = wt[r];
                    const float ct = wacc[r] * e;
                    const float dct = fmaf(gacc[r], inv4[a4][c], db4[a4][c]);
                    const float cs = END_SCALE ? ct * scale_s : ct;
                    dd[r] = cs * dct;
                    colsum = fmaf(cs, dct, colsum);
                    gacc[r] = STRICT ? dct : dct * e;   // (split mode: with wt and 1/n, the factors of G and W)
                    wacc[r] = STRICT ? ct : ct * inv4[a4][c];
                }
            }
            colp[kb * 64 + lane] = colsum;
            // (a lane's sum is that of its register: see row_sums8)
            float* const rt = rowtmp + ((v & 1) * 2 + kb) * 32 + (lane & 2) * 4 + 4 * h + (lane & 1) * 2 + ((lane >> 4) & 1);
            rt[0] = row_sums8(dd, hi1, hi2);
            rt[16] = row_sums8(dd + 8, hi1, hi2);
            hand_over(v, inv4);
        };
        if (role == 1) {   // the second pair is one step behind
            if constexpr (Cfg::PBUF == 1) __syncthreads();
            __syncthreads();
        }
        for (int v = role; v < n_steps; v += 2) {
            if constexpr (Cfg::PBUF == 1) __syncthreads();
            if (v < NT && active(v)) {
                const int qi0 = CW_QT * (it0 + v);
                if (qi0 == key0 || qi0 + CW_QT > S) products(v, std::true_type{});
                else products(v, std::false_type{});
            }
            __syncthreads();
            if (v + 1 < n_steps) {
                if constexpr (Cfg::PBUF == 1) __syncthreads();   // (the consumers have read the tile before)
                if (v < NT && active(v)) {
                    weigh(v);
                } else {
                    if (v < NT && lane < 32) rowtmp[((v & 1) * 2 + kb) * 32 + lane] = 0.f;
                }
                __syncthreads();
            }
        }
    } else {
        SwzTransReader<T, D> trd;
        trd.init(lane, 0);
        f32x16 acc[NXD];
#pragma unroll
        for (int x = 0; x < NXD; x++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[x][r] = 0.f;
        // ---- state phase (see mlstm_cold.hip): dK contracts over E's rows (values), dV's columns are rows of E
        float colacc = 0.f;
        if (has_state) {
            const int own_row = (c32 & ~15) | ((c32 & 3) | ((c32 & 4) << 1) | ((c32 & 8) >> 1));   // the stored place of row c32 of a block
            const int own_off = Z::off(own_row, R::EPL * h);
            // the keys' fragments, V for dK, K for dV; a key that drops the state part (END_SCALE) multiplies with zeros
            auto keys = [&](int st) __attribute__((always_inline)) {
                frag f = rrd.read(slot_at(1 - role), kb, st);
                if constexpr (END_SCALE) {
                    i32x4 bits = __builtin_bit_cast(i32x4, f);
#pragma unroll
                    for (int e = 0; e < 4; e++) bits[e] = use ? bits[e] : 0;
                    f = __builtin_bit_cast(frag, bits);
                }
                return f;
            };
            constexpr int PF = D == 128 ? 4 : 3;   // fragments under way: product by product the phase waited for LDS three quarters of its time
#pragma unroll
            for (int n = 0; n < Cfg::NE; n++) {
                const T* const th = e_hi(n);
                const T* const tl = e_lo(n);
                frag ef[PF], el[STRICT ? PF : 1], bf[2];
                if (role == 0) {
                    constexpr int M = Cfg::E_ROWS / KW, N = M * NXD;
                    auto rd = [&](int k) __attribute__((always_inline)) {
                        ef[k % PF] = trd.read(th, KW * (k / NXD), k % NXD);
                        if constexpr (STRICT) el[k % PF] = trd.read(tl, KW * (k / NXD), k % NXD);
                    };
                    bf[0] = keys(M * n);
#pragma unroll
                    for (int k = 0; k < PF - 1; k++) rd(k);
#pragma unroll
                    for (int k = 0; k < N; k++) {
                        const int m = k / NXD, x = k % NXD;
                        if (x == 0 && m + 1 < M) bf[(m + 1) & 1] = keys(M * n + m + 1);
                        if (k + PF - 1 < N) rd(k + PF - 1);
                        R::mma(acc[x], ef[k % PF], bf[m & 1]);
                        if constexpr (STRICT) R::mma(acc[x], el[k % PF], bf[m & 1]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
                    constexpr int I = Cfg::E_ROWS / 32, N = NS * I;
                    auto rd = [&](int k) __attribute__((always_inline)) {
                        const int t = k / I, o = (own_off ^ ((t % 8) << 5)) + (t / 8) * 256 + 32 * (k % I) * Z::ROW_BYTES;
                        ef[k % PF] = *reinterpret_cast<const frag*>(reinterpret_cast<const char*>(th) + o);
                        if constexpr (STRICT) el[k % PF] = *reinterpret_cast<const frag*>(reinterpret_cast<const char*>(tl) + o);
                    };
                    bf[0] = keys(0);
#pragma unroll
                    for (int k = 0; k < PF - 1; k++) rd(k);
#pragma unroll
                    for (int k = 0; k < N; k++) {
                        const int t = k / I, x = I * n + k % I;
                        if (k % I == 0 && t + 1 < NS) bf[(t + 1) & 1] = keys(t + 1);
                        if (k + PF - 1 < N) rd(k + PF - 1);
                        R::mma(acc[x], ef[k % PF], bf[t & 1]);
                        if constexpr (STRICT) R::mma(acc[x], el[k % PF], bf[t & 1]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                dma_wait();
                __syncthreads();
                piece(n + 2);
            }
            // k . (E v + g) w, the column sums of dD over the queries behind the chunk (and, for fp16, the scaling itself)
            // (K out of its slot: tile AHEAD + 1, the first one there, is copied in the second step.  From memory, the
            // rows came behind the copies under way: with them and an epilogue that waited for each of its LDS reads, bf16, chunks of 512: D = 128,
            // 16 x 2048 32.1 us, now 30.2; split mode, D = 256, 8 x 1500: 42.9 -> 41.8)
            static_assert((AHEAD + 1 + 2) % NSLOT == 0, "K outlives the first step");
            if (role == 0) {
                const char* const kt = reinterpret_cast<const char*>(slot_at(0));
                float cp = 0.f;
#pragma unroll
                for (int x = 0; x < NXD; x++) {
#pragma unroll
                    for (int a4 = 0; a4 < 4; a4++) {
                        const f32x4 kv = __builtin_convertvector(*reinterpret_cast<const typename R::vec4*>(kt + Z::off(32 * kb + c32, 32 * x + 8 * a4) + 4 * h * (int)sizeof(T)), f32x4);
                        const f32x4 g4 = *reinterpret_cast<const f32x4*>(gvl + 32 * x + 8 * a4 + 4 * h);
#pragma unroll
                        for (int c = 0; c < 4; c++) {
                            if constexpr (END_SCALE) {
                                cp = fmaf(acc[x][4 * a4 + c] + g4[c], kv[c], cp);
                            } else {
                                const float dkv = (acc[x][4 * a4 + c] + g4[c]) * wk;
                                acc[x][4 * a4 + c] = dkv;
                                cp = fmaf(dkv, kv[c], cp);
                            }
                        }
                    }
                }
                colacc = END_SCALE ? rounded_product(cp, wk) : cp;
            } else if constexpr (!END_SCALE) {
#pragma unroll
                for (int x = 0; x < NXD; x++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[x][r] *= wk;
            }
        }
        if (role == 0) colp[kb * 64 + lane] = colacc;   // (the weighing waves take it on from here)
        // row sums: the slice of these 64 keys
        float* const rowpart_slice = a.rowpart + ((size_t)bh * a.RS + (a.RS == NG ? jt : jt % a.RS)) * S + CW_QT * it0;
        constexpr int PF = 4, N = 2 * NXD;   // fragments under way, products per tile
        frag af[PF];
        auto read_tile = [&](int u, int n) __attribute__((always_inline)) { af[n % PF] = trd.read(role ? dh_at(u) : q_at(u), KW * (n / NXD), n % NXD); };
        auto consumes = [&](int u) { return u >= 0 && u < NT && !(u == 0 && kb > 0); };   // (tile 0 lies before the second 32 keys)
        for (int v = 0; v < n_steps; v++) {
            const int u = v - 2;                       // the tile to consume
            const bool consume = consumes(u);
            // (the store ahead of the copies: behind them, the step's wait would be for it)
            if (u >= 0 && wave == 4 && lane < 32 && CW_QT * (it0 + u) + lane < S)
                rowpart_slice[CW_QT * u + lane] = rowtmp[(u & 1) * 64 + lane] + rowtmp[(u & 1) * 64 + 32 + lane];
            frag b[2], bl[2];
            if (consume) {
#pragma unroll
                for (int n = 0; n < PF - 1; n++) read_tile(u, n);
                const char* const block = pbuf + (size_t)((Cfg::PBUF == 2 ? (u & 1) * 2 : 0) + kb) * 2 * Cfg::HALF_BYTES;
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const frag* const p = reinterpret_cast<const frag*>(block + t * Cfg::HALF_BYTES) + 64 * role + lane;
                    b[t] = p[0];
                    if constexpr (STRICT) bl[t] = p[128];
                }
            }
            if constexpr (Cfg::PBUF == 1) __syncthreads();
            // the copies of the tiles that the products will need next (tile 0 came with the prologue) go between the products
            const int vn = v + AHEAD;
            const bool copy = vn < NT, spread = copy && it0 + vn < full_q;
            if (D == 128 && v == 0) {
#pragma unroll 1
                for (int w = 1; w < AHEAD && w < NT; w++) copy_tile(w);
            }
            if (copy && !(spread && consume)) copy_tile(vn);
            if (consume) {
                constexpr int EVERY = N / (2 * PW);
#pragma unroll
                for (int n = 0; n < N; n++) {
                    const int t = n / NXD, x = n % NXD;
                    if (n + PF - 1 < N) read_tile(u, n + PF - 1);
                    R::mma(acc[x], af[n % PF], b[t]);
                    if constexpr (STRICT) R::mma(acc[x], af[n % PF], bl[t]);
                    if (n % EVERY == 0) {
                        if (spread) copy_piece(vn, n / EVERY);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // the next step's tile has landed: everything but the newest AHEAD - 1 tiles (2 PW loads each; a row sum's store
            // counts as one more and makes the wait a little longer)
            if (vn < NT) dma_wait_but<(AHEAD - 1) * 2 * PW>();
            else dma_wait();
            __syncthreads();
        }
        // ---- epilogue: column sums, dK and dV through LDS in whole rows (16-byte chunk c of row r at chunk c ^ (r & 31))
        if (role == 0) {
            colacc = sum_halves(colp[kb * 64 + lane]);
            if (h == 0 && key < S) a.colsum[hoff + key] = colacc;
        }
        constexpr int ROWB = D * (int)sizeof(T), CPR = ROWB / 16;
        char* const out = smem + (size_t)role * GRAN * ROWB;
        const int row = 32 * kb + c32;
        auto stage_out = [&](auto state_tag) __attribute__((always_inline)) {
            constexpr bool STATE = decltype(state_tag)::value;
            f32x4 gq[2][4];   // (a block ahead, see mlstm_cold.hip)
            auto read_g = [&](int x) __attribute__((always_inline)) {
#pragma unroll
                for (int a4 = 0; a4 < 4; a4++) gq[x & 1][a4] = *reinterpret_cast<const f32x4*>(gvl + 32 * x + 8 * a4 + 4 * h);
            };
            if constexpr (STATE) read_g(0);
#pragma unroll
            for (int x = 0; x < NXD; x++) {
                if constexpr (STATE) { if (x + 1 < NXD) read_g(x + 1); }
#pragma unroll
                for (int a4 = 0; a4 < 4; a4++) {
                    const int d = 32 * x + 8 * a4 + 4 * h;
                    f32x4 w;
#pragma unroll
                    for (int c = 0; c < 4; c++) w[c] = acc[x][4 * a4 + c];
                    if constexpr (END_SCALE) w *= scale_s;
                    if constexpr (STATE) {
#pragma unroll
                        for (int c = 0; c < 4; c++) w[c] = fmaf(gq[x & 1][a4][c], wkg, w[c]);
                    }
                    const int chunk16 = (d * (int)sizeof(T)) >> 4, within = (d * (int)sizeof(T)) & 15;
                    *reinterpret_cast<typename R::vec4*>(out + row * ROWB + (((chunk16 ^ (row & 31)) & (CPR - 1)) << 4) + within) = R::cvt4(w);
                }
            }
        };
        if (END_SCALE && !role && has_state) stage_out(std::integral_constant<bool, END_SCALE>{});
        else stage_out(std::false_type{});
    }
    __syncthreads();
    constexpr int ROWB = D * (int)sizeof(T), CPR = ROWB / 16, NPC = 2 * GRAN * CPR / 512;
    pieces_out<NPC>(
        [&](int i) {
            const int c = tid + 512 * i, row2 = c / CPR, cc = c % CPR;
            return *reinterpret_cast<const uint4*>(smem + row2 * ROWB + (((cc ^ (row2 & 31)) & (CPR - 1)) << 4));
        },
        [&](int i, uint4 v) {
            const int c = tid + 512 * i, row2 = c / CPR, row = row2 % GRAN, which = row2 / GRAN;
            if (GRAN * jt + row < S)
                *reinterpret_cast<uint4*>(reinterpret_cast<char*>(which ? a.dV : a.dK) + (offA + (size_t)(GRAN * jt + row) * rsA) * sizeof(T) + 16 * (c % CPR)) = v;
        });
#endif
}

template <typename T, int D, bool STRICT>
static int launch_colw_t(const ColArgs& a, hipStream_t st) {
    using Cfg = ColwCfg<T, D, STRICT>;
    if (a.chunk_len > 0 && (a.chunk_len % GRAN != 0 || (a.n_states > 0 && (!a.Ev || !a.gvec || (STRICT && !a.Ev_lo))))) return MLSTM_EINVAL;
    const int granules = a.chunk_len > 0 && a.chunk_len / GRAN < a.NG ? a.chunk_len / GRAN : a.NG;   // of queries that a key may meet
    const size_t lds = Cfg::lds_bytes(granules);
    if (granules > CW_MOST_QUERIES / GRAN) return MLSTM_ESHAPE;
    if (hipError_t e = lds_limit_once<colw_kernel<T, D, STRICT>>(160 * 1024); e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((colw_kernel<T, D, STRICT>), dim3(a.BH * a.NG), dim3(512), lds, st, a);
    return (int)hipGetLastError();
}
template <typename T>
static int launch_colw_d(int D, const ColArgs& a, hipStream_t st) {
    if (a.precise) return D == 128 ? launch_colw_t<T, 128, true>(a, st) : launch_colw_t<T, 256, true>(a, st);
    return D == 128 ? launch_colw_t<T, 128, false>(a, st) : launch_colw_t<T, 256, false>(a, st);
}
int launch_colw_kernel(int dtype, int D, const ColArgs& a, hipStream_t st) {
    return dtype == MLSTM_F16 ? launch_colw_d<_Float16>(D, a, st) : launch_colw_d<__bf16>(D, a, st);
}

}  // namespace mlstm
