// Column kernel of the fp32 tensors where few workgroups would run: the math of mlstm_col.hip and its order of operations, hence its
// bits, on 32 keys per workgroup with four waves on them.  (Where something is not finite, keys are formed again in fp32 multiply-adds:
// a workgroup's 32 here, 64 there.  Finite keys beside such a one can then differ in their last places.)
//
// As in mlstm_rowf.hip nothing but the accumulation over the queries is a chain:
//   phase A   wave w = block of 32 queries:  S^T = K Q^T, dC^T = V dH^T, the element-wise part, the terms of G and W to LDS;
//   phase B   wave w = 32 columns of dK and dV (D = 64: waves 0 and 1 of dK, 2 and 3 of dV):  dK^T += Q^T G, dV^T += dH^T W.
// All operands come into LDS by direct copies, the keys' K and V, 128 queries of Q and dH (the length of a chunk: a workgroup of a
// sequence in chunks makes one round), and before Q, in its place, the reverse state.  (Phase B's operands, columns over the queries,
// and the state's straight into registers, a dword per lane and row: 128 such loads per wave took the memory pipeline 3 us.)
#include <type_traits>
#include "mlstm_device.h"
#include "mlstm_kernels.h"
#include "mlstm_col_exact.h"

namespace mlstm {

template <int D>
struct ColfCfg {
    static constexpr size_t BLK_BYTES = (size_t)32 * D * 4;          // 32 rows of Q, dH, K or V
    static constexpr size_t GW_TILE = 32 * 32 * 2;                   // one term of G or W of a query block, [query][key]
    // Q of the four blocks, dH of the four blocks, K, V.  D = 128: the terms of a block's G and W lie over its Q, the column sums of
    // blocks 2 and 3 over their dH and what the epilogue exchanges over K; D = 64: all of these behind V.
    static constexpr bool OVER = D == 128;
    static constexpr size_t K_OFF = 8 * BLK_BYTES, V_OFF = 9 * BLK_BYTES, FREE_OFF = 10 * BLK_BYTES;
    static constexpr size_t GW_OFF = OVER ? 0 : FREE_OFF, GW_STRIDE = OVER ? BLK_BYTES : 6 * GW_TILE;
    static constexpr size_t SUM_BYTES = 16 * 64 * 4, SUM_OFF = OVER ? 6 * BLK_BYTES : GW_OFF + 4 * GW_STRIDE, SUM_STRIDE = OVER ? BLK_BYTES : SUM_BYTES;
    static constexpr size_t TAIL_BYTES = (4 * 32 + 2 * 32 + 4) * sizeof(float), TAIL_OFF = OVER ? K_OFF : SUM_OFF + 2 * SUM_BYTES;
    static constexpr size_t LDS_BYTES = OVER ? FREE_OFF : TAIL_OFF + TAIL_BYTES;
    static_assert(!OVER || (6 * GW_TILE <= BLK_BYTES && SUM_BYTES <= BLK_BYTES), "what lies over the blocks fits them");
};

template <int D>
__global__ __launch_bounds__(256, 1) void colf_kernel(ColArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    using T = float;
    using R = Tr<float>;
    using Cfg = ColfCfg<D>;
    typedef R::frag frag;
    typedef R::terms terms;
    constexpr int KW = R::KW, NS = D / KW;
    constexpr bool BOTH = D == 128;      // a wave has a column block of dK and of dV
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float* const cpart = reinterpret_cast<float*>(smem + Cfg::TAIL_OFF);   // [wave][key] k . dK of the state part
    float* const colx = cpart + 4 * 32;                                    // [parity][key]
    float* const flag = colx + 2 * 32;                                     // [wave]

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, c32 = lane & 31;
    const int S = a.S, NG = a.NG;
    int bh, kbi;
    {
        const int bid = blockIdx.x;   // ascending key blocks: heaviest first
        if ((a.BH & 7) == 0) {
            const int rest = bid >> 3, ngrp = a.BH >> 3;
            bh = (rest % ngrp) * 8 + (bid & 7);
            kbi = rest / ngrp;
        } else {
            bh = bid % a.BH;
            kbi = bid / a.BH;
        }
    }
    const int jt = kbi >> 1, kbA = kbi & 1, key0 = 32 * kbi;
    const size_t hoff = (size_t)bh * S, poff = (size_t)bh * NG * GRAN, goff = (size_t)bh * NG;
    const size_t rsA = (size_t)a.la.ss, rsB = (size_t)a.lb.ss, offA = a.la.head(bh), offB = a.lb.head(bh);
    const T* Q = reinterpret_cast<const T*>(a.Q) + offA;
    const T* dH = reinterpret_cast<const T*>(a.dH) + offB;
    const T* K = reinterpret_cast<const T*>(a.K) + offA;
    const T* V = reinterpret_cast<const T*>(a.V) + offA;
    const int tpc = a.chunk_len > 0 ? a.chunk_len / GRAN : 0;
    const int chunk = a.chunk_len > 0 ? jt / tpc : 0;
    const int NGe = a.chunk_len > 0 ? ((chunk + 1) * tpc < NG ? (chunk + 1) * tpc : NG) : NG;
    const int end = GRAN * NGe < S ? GRAN * NGe : S;                       // one past the last query the keys meet
    const bool has_state = a.chunk_len > 0 && chunk < a.n_states;
    float* const slice = (kbA ? a.rowpart2 : a.rowpart) + ((size_t)bh * a.RS + (a.RS == NG ? jt : jt % a.RS)) * S;
    if (key0 >= S) {   // (uniform over the workgroup) the empty second half of the last granule: its row partials are read all the same
        for (int t = GRAN * jt + tid; t < end; t += 256) slice[t] = 0.f;
        return;
    }
    const int q0 = GRAN * jt;                                              // the first query block is the granule's first
    const int nblocks = (end - q0 + 31) / 32, nR = (nblocks + 3) / 4;

    // ---- requests
    auto block_at = [&](int n) { return reinterpret_cast<T*>(smem + (size_t)n * Cfg::BLK_BYTES); };
    T* const qt = block_at(wave);
    T* const ht = block_at(4 + wave);
    T* const Kt = reinterpret_cast<T*>(smem + Cfg::K_OFF);
    T* const Vt = reinterpret_cast<T*>(smem + Cfg::V_OFF);
    TileDma<T, D, 32, 256> wd;
    wd.init(tid);
    TileDma<T, D, 32, 64> bd;
    bd.init(lane);
    const auto bra = bd.rows(lane, (unsigned)(rsA * sizeof(T))), brb = bd.rows(lane, (unsigned)(rsB * sizeof(T)));
    auto copy_rows = [&](T* dst, const T* src, int row0, size_t rs, const auto& rows) {
        if (row0 + 32 <= S) bd.issue(dst, src + (size_t)row0 * rs, rows);
        else tile_dma_rolled<T, D, 32, 64>(dst, src, row0, S, lane, rs);
    };
    {
        const auto wra = wd.rows(tid, (unsigned)(rsA * sizeof(T)));
        if (key0 + 32 <= S) {
            wd.issue(Kt, K + (size_t)key0 * rsA, wra);
            wd.issue(Vt, V + (size_t)key0 * rsA, wra);
        } else {
            tile_dma_rolled<T, D, 32, 256>(Kt, K, key0, S, tid, rsA);
            tile_dma_rolled<T, D, 32, 256>(Vt, V, key0, S, tid, rsA);
        }
    }
    if (has_state) {   // (the state goes where Q follows it)
        TileDma<T, D, D, 256> ed;
        ed.init(tid);
        ed.issue(block_at(0), reinterpret_cast<const T*>(a.Ev) + ((size_t)bh * a.n_states + chunk) * D * D);
    } else if (wave < nblocks) {
        copy_rows(qt, Q, q0 + 32 * wave, rsA, bra);
    }
    if (wave < nblocks) copy_rows(ht, dH, q0 + 32 * wave, rsB, brb);
    const int cb = BOTH ? wave : wave & 1;                                // the wave's column block
    const bool wants_k = BOTH || wave < 2, wants_v = BOTH || wave >= 2;   // it has one of dK, of dV
    f32x4 gv4[4];   // the reverse vector state of the lane's columns
    if (has_state && wants_k) {
        const float* gv = a.gvec + ((size_t)bh * a.n_states + chunk) * D;
#pragma unroll
        for (int a4 = 0; a4 < 4; a4++) gv4[a4] = *reinterpret_cast<const f32x4*>(gv + 32 * cb + 8 * a4 + 4 * h);
    }
    const double gj = a.G2[goff + jt];
    f32x4 al4[4];
#pragma unroll
    for (int a4 = 0; a4 < 4; a4++) al4[a4] = *reinterpret_cast<const f32x4*>(a.alpha2 + poff + key0 + 8 * a4 + 4 * h);
    const int pe = has_state ? (chunk + 1) * a.chunk_len - 1 : 0;          // the chunk's last position
    const float bend = a.beta2[poff + pe], alk = a.alpha2[poff + key0 + c32];
    const double dG = a.G2[goff + pe / GRAN] - gj;
    float nbeta = 0.f, inv = 0.f, dbv = 0.f;   // of the lane's query
    auto load_scalars = [&](int qstart) {
        const size_t at = poff + qstart + c32;   // (whole granules are there)
        nbeta = -a.beta2[at]; inv = a.inv_n[at]; dbv = a.db[at];
    };
    if (wave < nblocks) load_scalars(q0 + 32 * wave);
    dma_wait();
    __syncthreads();   // K and V (and each wave's own blocks) are there
    SwzRowReader<T, D> rrd;
    rrd.init(lane);
    SwzTransReaderF32<D> trd;   // (block cb & ~1 and the next; which of the two is known at run time only, so its offsets lie in 64 bytes of scratch)
    trd.init(lane, cb & ~1);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 dk, dv;
#pragma unroll
    for (int x = 0; x < 16; x++) { dk[x] = 0.f; dv[x] = 0.f; }
    float cp = 0.f;   // k . dK of the state part, of the lane's key and the wave's columns
    if (has_state) {
        const float wk = fast_exp2(alk - bend + (float)dG);
        if (wants_k) {
            R::template stream<NS>([&](auto n) { return trd.read(block_at(0), KW * n, cb & 1); }, [&](auto n, const auto& f, auto&& between) { R::mma_between(dk, f, R::split(rrd.read(Vt, 0, n)), between); });
#pragma unroll
            for (int a4 = 0; a4 < 4; a4++) {
                const int d = 32 * cb + 8 * a4 + 4 * h;
                const f32x4 g4v = gv4[a4];
                const f32x4 kv = *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(Kt) + Swz<T, D>::off(c32, d));
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const float dkv = (dk[4 * a4 + c] + g4v[c]) * wk;
                    dk[4 * a4 + c] = dkv;
                    cp = fmaf(dkv, kv[c], cp);
                }
            }
            cp = sum_halves(cp);
        }
        if (wants_v) {
            // (the states keep their rows in the contraction order of the transposing reads, see mlstm_chunk.hip)
            const int own = (c32 & ~15) | ((c32 & 3) | ((c32 & 4) << 1) | ((c32 & 8) >> 1));
            const T* const Eo = block_at(0) + (size_t)32 * cb * D;
            R::template stream<NS>([&](auto n) { return swz_frag_rowmajor<T, D>(Eo, own, n, h); }, [&](auto n, const auto& f, auto&& between) { R::mma_between(dv, f, R::split(rrd.read(Kt, 0, n)), between); });
#pragma unroll
            for (int x = 0; x < 16; x++) dv[x] *= wk;
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (has_state) {
        __syncthreads();   // every wave is done with the state
        if (wave < nblocks) copy_rows(qt, Q, q0 + 32 * wave, rsA, bra);
    }
    // factorised weights (see col_kernel)
    float al[16], ekr[16], amaxA;
    {
#pragma unroll
        for (int r = 0; r < 16; r++) al[r] = al4[r >> 2][r & 3];
        float mx = al[0];
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(mx, al[r]);
        amaxA = fmaxf(mx, __shfl_xor(mx, 32));
#pragma unroll
        for (int r = 0; r < 16; r++) ekr[r] = amaxA > -INFINITY ? fast_exp2(al[r] - amaxA) : 0.f;
    }
    const float log2scale = -0.5f * __log2f((float)D);
    float colacc[16];
#pragma unroll
    for (int r = 0; r < 16; r++) colacc[r] = 0.f;
    // terms of G and W of query block n: three tiles each of [query][key], 64 bytes a row, 16-byte piece c of row q at c ^ (q / 4 % 4)
    auto gw_tile = [&](int n, int which, int term) { return smem + Cfg::GW_OFF + n * Cfg::GW_STRIDE + (3 * which + term) * Cfg::GW_TILE; };
    int gwoff[2];
    {
        const int j = lane & 15, sub = (lane >> 4) & 1;
#pragma unroll
        for (int x = 0; x < 2; x++) {
            const int q = 8 * x + 4 * h + (j >> 2), c = 2 * sub + ((j & 3) >> 1);
            gwoff[x] = q * 64 + ((c ^ ((q >> 2) & 3)) << 4) + 8 * (j & 1);
        }
    }
    auto gw_read = [&](int n, int which, int term, int t) __attribute__((always_inline)) {
        const char* tile = gw_tile(n, which, term) + 16 * t * 64;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(tile + gwoff[0]));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(tile + gwoff[1]));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    for (int r = 0; r < nR; r++) {
        const int n = 4 * r + wave, qstart = q0 + 32 * n;
        const bool mine = n < nblocks, first = n < 2;      // (the granule of the keys: weights from their definition, and the causal mask)
        if (r > 0) {
            __syncthreads();   // phase B of the previous round is over
            if (mine) { copy_rows(qt, Q, qstart, rsA, bra); copy_rows(ht, dH, qstart, rsB, brb); load_scalars(qstart); }
        }
        pin(nbeta); pin(inv); pin(dbv);
        __builtin_amdgcn_sched_barrier(0);
        float dd[16];
#pragma unroll
        for (int x = 0; x < 16; x++) dd[x] = 0.f;
        f32x16 g, w;
#pragma unroll
        for (int x = 0; x < 16; x++) { g[x] = 0.f; w[x] = 0.f; }
        float rsum = 0.f;
        const int qrow = qstart + c32;
        if (mine && key0 <= qstart) {
            const double crow = (double)log2scale + (a.G2[goff + qstart / GRAN] - gj);
            f32x16 s = {}, s2 = {}, d = {}, d2 = {};
            if (r > 0) dma_wait();
            R::template stream<NS>([&](auto m) { return rrd.read(ht, 0, m); }, [&](auto m, const auto& f, auto&& between) { R::mma_between(d, d2, R::split(rrd.read(Vt, 0, m)), f, between); });
            dma_wait();   // (the wave's own block of Q, which follows the state)
            R::template stream<NS>([&](auto m) { return rrd.read(qt, 0, m); }, [&](auto m, const auto& f, auto&& between) { R::mma_between(s, s2, R::split(rrd.read(Kt, 0, m)), f, between); });
        __builtin_amdgcn_sched_barrier(0);
            s += s2; d += d2;
            const bool qvalid = qrow < S, diag = key0 == qstart;
            const float er = !qvalid ? 0.f : fast_exp2((float)((double)(amaxA + nbeta) + crow));
            const float inv_er = inv * er, dbv_er = dbv * er;
            // keys above this one, counted from 4 h, are masked.  (As a condition on the weight, each element of the diagonal granule was a branch
            // of its own: 17.4 us, now 16.6, at D = 64, 4 x 2048; D = 128, 32 x 4096: 337 -> 328.)
            const int lastkey = !qvalid ? -1 : diag ? c32 - 4 * h : 32;
            auto element = [&](auto first_tag, int x) __attribute__((always_inline)) {
                if constexpr (decltype(first_tag)::value) {
                    const bool masked = 8 * (x >> 2) + (x & 3) > lastkey;
                    const float e = fast_exp2(masked ? -INFINITY : (al[x] + nbeta) + (float)crow);
                    const float ct = s[x] * e;
                    const float dct = fmaf(d[x], inv, dbv);
                    dd[x] = product_apart(ct, dct);   // (as in col_kernel)
                    rsum = fmaf(ct, dct, rsum);
                    g[x] = dct * e;
                    w[x] = ct * inv;
                } else {
                    const float dct_er = fmaf(d[x], inv_er, dbv_er);
                    const float sk = s[x] * ekr[x];
                    g[x] = dct_er * ekr[x];
                    w[x] = sk * inv_er;
                    dd[x] = product_apart(sk, dct_er);
                    rsum = fmaf(sk, dct_er, rsum);
                }
            };
            if (first) {
#pragma unroll
                for (int x = 0; x < 16; x++) element(std::true_type{}, x);
            } else {
#pragma unroll
                for (int x = 0; x < 16; x++) element(std::false_type{}, x);
            }
        }
        // the wave's columns of the 128 queries, for phase B, before the terms of G and W go where Q is
        frag qc[8], hc[8];
        dma_wait();        // (a wave whose block lies above the diagonal has not waited for its Q)
        __syncthreads();
        if (wants_k) {
#pragma unroll
            for (int n = 0; n < 8; n++) qc[n] = trd.read(block_at(0), KW * n, cb & 1);
        }
        if (wants_v) {
#pragma unroll
            for (int n = 0; n < 8; n++) hc[n] = trd.read(block_at(4), KW * n, cb & 1);
        }
#pragma unroll
        for (int n = 0; n < 8; n++) {
            if (wants_k) pin(qc[n]);
            if (wants_v) pin(hc[n]);
        }
        __syncthreads();
        if (mine) {
#pragma unroll
            for (int a4 = 0; a4 < 4; a4++) {
                f32x4 gv, wv;
#pragma unroll
                for (int c = 0; c < 4; c++) { gv[c] = g[4 * a4 + c]; wv[c] = w[4 * a4 + c]; }
                const terms t = R::split(__builtin_shufflevector(gv, wv, 0, 1, 2, 3, 4, 5, 6, 7));
                const int off = c32 * 64 + ((a4 ^ ((c32 >> 2) & 3)) << 4) + 8 * h;
                auto put = [&](int which, int term, bf16x4 x) { *reinterpret_cast<bf16x4*>(gw_tile(wave, which, term) + off) = x; };
                put(0, 0, __builtin_shufflevector(t.hi, t.hi, 0, 1, 2, 3)); put(1, 0, __builtin_shufflevector(t.hi, t.hi, 4, 5, 6, 7));
                put(0, 1, __builtin_shufflevector(t.mid, t.mid, 0, 1, 2, 3)); put(1, 1, __builtin_shufflevector(t.mid, t.mid, 4, 5, 6, 7));
                put(0, 2, __builtin_shufflevector(t.lo, t.lo, 0, 1, 2, 3)); put(1, 2, __builtin_shufflevector(t.lo, t.lo, 4, 5, 6, 7));
            }
            const float rs = sum_halves(rsum);
            if (h == 0 && qrow < S) slice[qrow] = rs;
        }
        __builtin_amdgcn_sched_barrier(0);
        // column sums: blocks of one parity in order, waves 2 and 3 hand theirs to waves 0 and 1
        float* const handed = reinterpret_cast<float*>(smem + Cfg::SUM_OFF + (wave & 1) * Cfg::SUM_STRIDE) + lane;
        if (wave >= 2) {
#pragma unroll
            for (int x = 0; x < 16; x++) handed[64 * x] = dd[x];
        } else {
#pragma unroll
            for (int x = 0; x < 16; x++) colacc[x] += dd[x];
        }
        __syncthreads();
        if (wave < 2) {
#pragma unroll
            for (int x = 0; x < 16; x++) colacc[x] += handed[64 * x];
        }
        __builtin_amdgcn_sched_barrier(0);
        // ---- phase B
        const int nb = nblocks - 4 * r < 4 ? nblocks - 4 * r : 4;
        // (block by block: as one switch over their number the compiler forms every case's terms ahead of it and spills)
        static_for<4>([&](auto nc) __attribute__((always_inline)) {
            constexpr int n = decltype(nc)::value;
            if (n >= nb) return;
            auto one = [&](f32x16& acc, const frag (&c)[8], int which) __attribute__((always_inline)) {
                R::template stream<2>([&](auto m) { return c[2 * n + m]; }, [&](auto m, const auto& f, auto&& between) {
                    const terms t = {gw_read(n, which, 0, m), gw_read(n, which, 1, m), gw_read(n, which, 2, m)};
                    R::mma_between(acc, f, t, between);
                });
            };
            if constexpr (BOTH) {
                R::template stream<4>([&](auto m) { return m < 2 ? qc[2 * n + m] : hc[2 * n + m - 2]; }, [&](auto m, const auto& f, auto&& between) {
                    constexpr int which = m / 2, t16 = m % 2;
                    const terms t = {gw_read(n, which, 0, t16), gw_read(n, which, 1, t16), gw_read(n, which, 2, t16)};
                    R::mma_between(which ? dv : dk, f, t, between);
                });
            } else if (wants_k) {
                one(dk, qc, 0);
            } else {
                one(dv, hc, 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- epilogue: the column sums over the query lanes, the two parities and the state part
    __syncthreads();   // (what is exchanged lies over K)
    if (wants_k && h == 0) cpart[cb * 32 + c32] = cp;
#pragma unroll
    for (int x = 0; x < 16; x++) {
        float v = colacc[x];
        v = sum_half_wave(v);
        if (wave < 2 && c32 == 0) colx[wave * 32 + 8 * (x >> 2) + 4 * h + (x & 3)] = v;
    }
    float seen = not_finite(0.f, cp);
#pragma unroll
    for (int x = 0; x < 16; x++) seen = not_finite(not_finite(not_finite(seen, colacc[x]), dk[x]), dv[x]);
    const bool any = __any(seen != 0.f);
    if (lane == 0) flag[wave] = any ? 1.f : 0.f;
    dma_wait();        // (the row partials written above: col_exact writes them again)
    __syncthreads();
    if (flag[0] + flag[1] + flag[2] + flag[3] > 0.f) {
        col_exact<D, 32>(a, bh, key0, chunk, NGe, has_state, Q, dH, K, V, rsA, rsB, offA, slice);
        return;
    }
    float far = 0.f;
    if (has_state && tid < 32) far = D == 64 ? cpart[tid] + cpart[32 + tid] : (cpart[tid] + cpart[32 + tid]) + (cpart[64 + tid] + cpart[96 + tid]);
    if (tid < 32 && key0 + tid < S) a.colsum[hoff + key0 + tid] = colx[tid] + colx[32 + tid] + far;
    if (key0 + c32 < S) {
        const size_t at = offA + (size_t)(key0 + c32) * rsA + 32 * cb + 4 * h;
#pragma unroll
        for (int a4 = 0; a4 < 4; a4++) {
            if (wants_k) *reinterpret_cast<f32x4*>(reinterpret_cast<T*>(a.dK) + at + 8 * a4) = f32x4{dk[4 * a4], dk[4 * a4 + 1], dk[4 * a4 + 2], dk[4 * a4 + 3]};
            if (wants_v) *reinterpret_cast<f32x4*>(reinterpret_cast<T*>(a.dV) + at + 8 * a4) = f32x4{dv[4 * a4], dv[4 * a4 + 1], dv[4 * a4 + 2], dv[4 * a4 + 3]};
        }
    }
#endif
}

template <int D>
static int launch_colf_t(const ColArgs& a, hipStream_t st) {
    if (hipError_t e = lds_limit_once<colf_kernel<D>>((int)ColfCfg<D>::LDS_BYTES); e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(colf_kernel<D>, dim3(a.BH * a.NG * 2), dim3(256), ColfCfg<D>::LDS_BYTES, st, a);
    return (int)hipGetLastError();
}

int launch_colf_kernel(int D, const ColArgs& a, hipStream_t st) { return D == 64 ? launch_colf_t<64>(a, st) : launch_colf_t<128>(a, st); }

}  // namespace mlstm
