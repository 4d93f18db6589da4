// Row-parallel tile kernel of split mode (16-bit types, D >= 128) where few workgroups would run: the same math and, element by element,
// the same order of operations as the split mode of mlstm_row.hip, hence the same bits, on half as many rows per workgroup and with
// every key tile's work spread over eight waves.
//
// row_kernel gives a wave 32 rows with all of their work: 3 us per 64 keys at D = 256, with half the chip idle at 96 workgroups.  A
// workgroup here owns one granule of 64 rows; its walk is a pipeline of 64-key tiles with one barrier per tile:
//   step v      four producer waves, (row block of 32, key block of 32):  S^T = K Q^T (dQ pass: dC^T = V dH^T) of tile v, gate weights, the
//               weights' two terms to LDS; the row sums go from wave to wave, one sum per row;
//   step v + 1  four consumer waves, (row block, half of the columns):  H^T += V^T P^T (dQ^T += K^T G^T), both terms.
// The state of the previous chunk goes through the consumers first, while the producers are at tile 0.  A step takes 2300 cycles at D = 256:
// the 64 KB of a tile pair at what a CU gets out of L2 with all of them asking, 26 bytes per cycle.  (The form without terms, measured on
// these lines, was slower than mlstm_roww.hip, which takes two tiles per pair of barriers: 20.9 us against 18.3 at 8 x 1777 x 256.)
// Replaces, like mlstm_row.hip, mlstm_matmul_kernel (mlstm_matmul.py:38-101) and the dQ loop of mlstm_matmul_kernel_backward
// (mlstm_matmul.py:239-267).
#include <type_traits>
#include "mlstm_device.h"
#include "mlstm_kernels.h"

namespace mlstm {

constexpr int RX_FWD = 0, RX_DQ = 1;
constexpr int RX_MOST_KEYS = 1024;   // keys a row may meet: their scalars stay in LDS for the whole kernel

template <typename T, int D>
struct RowxCfg {
    static constexpr size_t TILE_BYTES = (size_t)GRAN * D * sizeof(T);
    static constexpr int NB = D == 256 ? 2 : 4, AHEAD = NB - 1;        // tiles of Y1 and of Y2 in LDS: 128 KB in all
    static constexpr size_t POOL_BYTES = 2 * NB * TILE_BYTES;
    static constexpr size_t BLOCK_BYTES = 2 * 2 * 64 * 16, P_BYTES = 4 * BLOCK_BYTES;   // [key block][row block][16 keys][hi, lo][lane]; one buffer (two and the tiles are all of LDS)
    static constexpr int E_ROWS = 32, NE = D / E_ROWS;                 // the state in pieces of a tile's size, hi, then lo
    static constexpr size_t MISC_FLOATS = 2 * 64 * 2 + 2 * 32 + 2 * 2 * 32 + 2 * 32 * 2 + D + RX_MOST_KEYS / GRAN;   // what producers hand over, row sums, far row sums, 1/n and db, vector state, granule distances
    static size_t lds_bytes(int keys) { return POOL_BYTES + P_BYTES + MISC_FLOATS * 4 + (size_t)keys * 8 + GRAN * 4; }
};

template <typename T, int D, int MODE>
__global__ __launch_bounds__(512) void rowx_kernel(RowArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    using R = Tr<T>;
    using Cfg = RowxCfg<T, D>;
    typedef typename R::frag frag;
    static_assert(R::HALF && (D == 128 || D == 256), "16-bit types, D = 128 or 256");
    constexpr int KW = R::KW, NS = D / KW, NC = D / 64, NB = Cfg::NB, AHEAD = Cfg::AHEAD;   // NC: column blocks of a consumer
    extern __shared__ __attribute__((aligned(16))) char smem[];
    char* const pbuf = smem + Cfg::POOL_BYTES;
    float* const handed = reinterpret_cast<float*>(pbuf + Cfg::P_BYTES);   // [rb][lane] x {sum, row factor} of the second key block; then {row sum so far}
    float* const bex = handed + 2 * 64 * 2;                // [rb][32]
    float* const rpx = bex + 2 * 32;                       // [rb][column half][32]
    float* const stat = rpx + 2 * 2 * 32;                  // [rb][32] x {1/n, db}
    float* const nvl = stat + 2 * 32 * 2;                  // [D]
    float* const sdg = nvl + D;                            // granule of the rows minus granule j
    float* const sek = sdg + RX_MOST_KEYS / GRAN;          // ek of the keys, then alpha, then the block maxima

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, c32 = lane & 31;
    const bool producer = wave < 4;
    const int rb = wave & 1, kb = (wave >> 1) & 1;         // a producer's key block; a consumer's half of the columns
    int S = a.S, NG = a.NG;
    int bh, qt;
    {
        // heaviest row tiles first over all heads; with a multiple of 8 heads a head's tiles run on one XCD
        const int bid = blockIdx.x, nQT = NG;
        if ((a.BH & 7) == 0) {
            const int rest = bid >> 3, ngrp = a.BH >> 3;
            bh = (rest % ngrp) * 8 + (bid & 7);
            qt = nQT - 1 - rest / ngrp;
        } else {
            bh = bid % a.BH;
            qt = nQT - 1 - bid / a.BH;
        }
    }
    size_t hoff = (size_t)bh * S, poff = (size_t)bh * NG * GRAN, goff = (size_t)bh * NG;
    const size_t rsA = (size_t)a.la.ss, rsB = (size_t)a.lb.ss, rsH = (size_t)a.lh.ss;
    size_t offA = a.la.head(bh), offB = a.lb.head(bh), offH = MODE == RX_DQ ? a.lh.head(bh) : 0;
    int chunk = 0;   // in chunks positions count from the chunk's first one (see mlstm_row8.hip)
    if (a.chunk_len > 0) {
        chunk = (qt * GRAN) / a.chunk_len;
        const int p0 = chunk * a.chunk_len;
        hoff += p0; poff += p0; goff += p0 / GRAN;
        offA += (size_t)p0 * rsA; offB += (size_t)p0 * rsB; offH += (size_t)p0 * rsH;
        S -= p0; qt -= p0 / GRAN;
    }
    const int r0 = GRAN * qt;
    const int nJ = qt + 1;                                  // key tiles; the last one is the rows' own
    const int row = r0 + 32 * rb + c32, rowc = row < S ? row : S - 1;
    const size_t rsX = MODE == RX_FWD ? rsA : rsB, offX = MODE == RX_FWD ? offA : offB;
    const size_t rsO = MODE == RX_FWD ? rsB : rsA, offO = MODE == RX_FWD ? offB : offA;
    const T* X = reinterpret_cast<const T*>(a.X) + offX;
    const T* Y1 = reinterpret_cast<const T*>(a.Y1) + offA;
    const T* Y2 = reinterpret_cast<const T*>(a.Y2) + offA;
    const int full_tiles = S / GRAN;
    const int keys = GRAN * nJ;
    float* const sal = sek + keys;
    float* const sam = sal + keys;

    auto y1_at = [&](int j) { return reinterpret_cast<T*>(smem + (size_t)(j & (NB - 1)) * Cfg::TILE_BYTES); };
    auto y2_at = [&](int j) { return reinterpret_cast<T*>(smem + (size_t)(NB + (j & (NB - 1))) * Cfg::TILE_BYTES); };
    // a tile's copy by the consumers, in pieces that go between their products
    typedef TileDma<T, D, GRAN, 256> Tile;
    constexpr int PW = Tile::PER_WAVE;
    const int tidc = tid & 255;
    Tile tdma;
    tdma.init(tidc);
    const auto ra = tdma.rows(tidc, (unsigned)(rsA * sizeof(T)));
    auto copy_tile = [&](T* dst, const T* src, int j) {
        if (j >= nJ) return;
        if (j < full_tiles) tdma.issue(dst, src + (size_t)GRAN * j * rsA, ra);
        else tile_dma_rolled<T, D, GRAN, 256>(dst, src, GRAN * j, S, tidc, rsA);
    };
    auto copy_y1 = [&](int j) { copy_tile(y1_at(j), Y1, j); };
    auto copy_y2 = [&](int j) { copy_tile(y2_at(j), Y2, j); };
    // (plain loads first: what they bring is used behind the copies' issue)
    const double g_rows = a.G2[goff + qt], g_mine = a.G2[goff + (tid < nJ ? tid : 0)], g_end = chunk > 0 ? a.G2[goff - 1] : 0.0;
    const float beta_row = a.beta2[poff + rowc], beta_end = chunk > 0 ? a.beta2[poff - 1] : 0.f;
    const float n_mine = chunk > 0 && tid < D ? a.Nst[((size_t)bh * a.n_states + chunk - 1) * D + tid] : 0.f;
    const bool stats = MODE == RX_DQ && producer && kb == 0;
    const float m_row = MODE == RX_FWD || stats ? a.M[hoff + rowc] : 0.f, b_row = stats ? a.Bin[hoff + rowc] : 0.f;
    // ---- prologue.  The rows' own operand (in Y1's second tile), the first keys and the first pieces of the previous chunk's state are
    // requested at once
    T* const xtile = y1_at(1);
    TileDma<T, D, GRAN, 512> wdma;
    wdma.init(tid);
    {
        const auto rx = wdma.rows(tid, (unsigned)(rsX * sizeof(T)));
        if (r0 + GRAN <= S) wdma.issue(xtile, X + (size_t)r0 * rsX, rx);
        else tile_dma_rolled<T, D, GRAN, 512>(xtile, X, r0, S, tid, rsX);
    }
    const size_t sbase = chunk > 0 ? ((size_t)bh * a.n_states + chunk - 1) * D * D : 0;
    TileDma<T, D, Cfg::E_ROWS, 512> edma;
    edma.init(tid);
    // Piece n of the state lies in ring[n % RING]: Y2's tiles, at D = 256 with Y1's second one (two pieces from memory under way: with one the
    // phase took 24000 cycles for its 256 KB)
    constexpr int RING = D == 256 ? 3 : 4, EW = 2 * TileDma<T, D, Cfg::E_ROWS, 512>::PER_WAVE;   // EW: a wave's loads per piece
    static_assert(D == 256 ? Cfg::NE % 3 == 2 : Cfg::NE == 4, "what follows the last pieces (see the consumers)");
    auto e_hi = [&](int n) { return n % RING == 2 && D == 256 ? y1_at(1) : y2_at(n % RING); };
    auto e_lo = [&](int n) { return e_hi(n) + Cfg::E_ROWS * D; };
    auto piece = [&](int n) {
        if (n >= Cfg::NE) return;
        edma.issue(e_hi(n), reinterpret_cast<const T*>(a.Cst) + sbase + (size_t)Cfg::E_ROWS * n * D);
        edma.issue(e_lo(n), reinterpret_cast<const T*>(a.Cst_lo) + sbase + (size_t)Cfg::E_ROWS * n * D);
    };
    if (!producer) copy_y1(0);
    if (chunk > 0) {
#pragma unroll
        for (int n = 0; n < (D == 256 ? 2 : 4); n++) piece(n);
    }
    else if (!producer) copy_y2(0);
    for (int t = wave; t < nJ; t += 8) {
        dma4(a.ek2 + poff + GRAN * t + lane, __builtin_amdgcn_readfirstlane(lds_offset_of(sek + GRAN * t)));
        dma4(a.alpha2 + poff + GRAN * t + lane, __builtin_amdgcn_readfirstlane(lds_offset_of(sal + GRAN * t)));
    }
    if (tid < GRAN) dma4(a.amax2 + goff * 2 + tid, __builtin_amdgcn_readfirstlane(lds_offset_of(sam)));   // (2 nJ of them count; padded array)
    const float crow_base = -0.5f * __log2f((float)D) - beta_row;
    float dec = 0.f;   // the row's decay since the end of the previous chunk
    if (chunk > 0) dec = fast_exp2(beta_end - beta_row + (float)(g_rows - g_end));
    if (tid < nJ) sdg[tid] = (float)(g_rows - g_mine);
    if (chunk > 0 && tid < D) nvl[tid] = n_mine;
    SwzRowReaderX<T, D> rrd;
    rrd.init(lane);
    float inv_n = 0.f, dbv = 0.f;
    auto p_block = [&](int k) { return pbuf + (size_t)(k * 2 + rb) * Cfg::BLOCK_BYTES; };
    float onorm = 1.0f;
    f32x16 acc[NC];   // the consumers' columns 32 (NC kb + c) ..

    // behind piece n: the next one has landed
    auto state_wait = [&](int n) __attribute__((always_inline)) {
        if (D == 256 && n < Cfg::NE - 2) dma_wait_but<EW>();               // (piece n + 2 is under way)
        else if (D == 256 && n == Cfg::NE - 2 && !producer && nJ > 1) dma_wait_but<PW>();   // (the second tile of Y1 is)
        else if (D == 256 || n == Cfg::NE - 1) dma_wait();                 // (D = 128: all of them came with the prologue)
    };
    auto row_scalars = [&]() __attribute__((always_inline)) {
        if constexpr (MODE == RX_DQ) {
            const float2 st = *reinterpret_cast<const float2*>(stat + (32 * rb + c32) * 2);
            inv_n = st.x; dbv = st.y;
        }
        if (D == 256 && chunk > 0) piece(2);   // (takes the place of X)
    };
    // (either kind of waves keeps X's fragments of its own: as one array in front of both they were spilled, and the reloads waited for the
    // copies under way)
    if (producer) {
        frag hf[NS], hl[NS];
        const bool with_lo = MODE == RX_DQ && a.Hin_lo;
        if (stats) {
            const T* const hrow = reinterpret_cast<const T*>(a.Hin) + offH + (size_t)rowc * rsH;
            const T* const lrow = with_lo ? reinterpret_cast<const T*>(a.Hin_lo) + (hoff + rowc) * D : hrow;
#pragma unroll
            for (int s = 0; s < NS; s++) { hf[s] = frag_rowmajor<T>(hrow, s, h); hl[s] = frag_rowmajor<T>(lrow, s, h); }
        }
        dma_wait();
        __syncthreads();
        frag xf[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) xf[s] = rrd.read(xtile, rb, s);
        if (stats) {   // 1/n and db of the rows (see row_stats), for this kernel and for the column kernel
            float dot = 0.f, dot_lo = 0.f, inv = 0.f, dbr = 0.f;
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int e = 0; e < R::EPL; e++) {
                    dot += (float)xf[s][e] * (float)hf[s][e];
                    dot_lo += (float)xf[s][e] * (float)hl[s][e];
                }
            row_stats_of(sum_halves(with_lo ? dot + dot_lo : dot), b_row, m_row, inv, dbr);
            if (h == 0) {
                *reinterpret_cast<float2*>(stat + (32 * rb + c32) * 2) = make_float2(inv, dbr);
                a.inv_n[poff + row] = row < S ? inv : 0.f;   // (rows behind the sequence: zeros, see mlstm_row.hip)
                a.db[poff + row] = row < S ? dbr : 0.f;
            }
        }
#pragma unroll
        for (int s = 0; s < NS; s++) pin(xf[s]);
        __syncthreads();   // X's tile is free; the rows' scalars are there
        row_scalars();
        // Row sums: one sum per row in the order of the keys, the state part first, as a wave of row_kernel keeps it.  The waves of the first key
        // blocks have it; the others hand their blocks' shares to them, a tile behind, and take it over for the block on the diagonal.
        float bsum = 0.f, blk_was = 0.f, er_was = 0.f;
        float* const mine = handed + (rb * 64 + lane) * 2;
        float s_own[16], e_own[16];   // products and weights of the rows' own granule
        auto add_own = [&] {
#pragma unroll
            for (int x = 0; x < 16; x++) bsum = fmaf(s_own[x], e_own[x], bsum);
        };
        auto weigh_tile = [&](int j) __attribute__((always_inline)) {
            f32x16 s;
            const int k0 = GRAN * j + 32 * kb, rr = r0 + 32 * rb;
            const T* const y1 = y1_at(j);
            const float crow = crow_base + sdg[j];
            if constexpr (MODE == RX_FWD) {
                if (kb == 0 && j > 0) {   // the tile before this one
                    const float2 other = *reinterpret_cast<const float2*>(mine);
                    bsum += fmaf(blk_was, er_was, other.x * other.y);
                }
            }
            constexpr int PRE = 4;
            frag kf[NS];
#pragma unroll
            for (int n = 0; n < PRE; n++) kf[n] = rrd.read(y1, kb, n);
#pragma unroll
            for (int x = 0; x < 16; x++) s[x] = 0.f;
#pragma unroll
            for (int n = 0; n < NS; n++) {
                if (n + PRE < NS) kf[n + PRE] = rrd.read(y1, kb, n + PRE);
                R::mma(s, kf[n], xf[n]);
                __builtin_amdgcn_sched_barrier(0);
                if (n == NS / 2 && j > 0) __syncthreads();   // (the consumers have read the tile before)
            }
            // The weights as factors x y, of which the low-order terms take what rounding the product would lose
            float blk = 0.f, er = 0.f;
            f32x4 wx, wy;
            typename R::vec4 hi[4], lo[4];
            if (k0 > rr) {             // above the diagonal
#pragma unroll
                for (int a4 = 0; a4 < 4; a4++) hi[a4] = lo[a4] = typename R::vec4{};
            } else if (j < nJ - 1) {   // factorised weights, as long as the keys' granule lies before the rows'
                er = fast_exp2(crow + sam[k0 / 32]);
#pragma unroll
                for (int a4 = 0; a4 < 4; a4++) {
                    const f32x4 ek = *reinterpret_cast<const f32x4*>(sek + k0 + 8 * a4 + 4 * h);
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const int x = 4 * a4 + c;
                        if constexpr (MODE == RX_FWD) {
                            blk = fmaf(s[x], ek[c], blk);
                            wx[c] = s[x] * ek[c];
                            wy[c] = er;
                        } else {
                            wx[c] = fmaf(s[x], inv_n, dbv);
                            wy[c] = ek[c] * er;
                        }
                    }
                    R::split_products(wx, wy, hi[a4], lo[a4]);
                }
            } else {                   // the rows' own granule, on the diagonal or below it
#pragma unroll
                for (int a4 = 0; a4 < 4; a4++) {
                    const f32x4 al = *reinterpret_cast<const f32x4*>(sal + k0 + 8 * a4 + 4 * h);
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const int x = 4 * a4 + c;
                        float e = fast_exp2(al[c] + crow);
                        if (k0 == rr && 8 * a4 + 4 * h + c > c32) e = 0.f;
                        if constexpr (MODE == RX_FWD) {
                            wx[c] = s[x];
                            s_own[x] = s[x];
                            e_own[x] = e;
                        } else {
                            wx[c] = fmaf(s[x], inv_n, dbv);
                        }
                        wy[c] = e;
                    }
                    R::split_products(wx, wy, hi[a4], lo[a4]);
                }
            }
            frag* const p = reinterpret_cast<frag*>(p_block(kb)) + lane;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                p[128 * t] = __builtin_shufflevector(hi[2 * t], hi[2 * t + 1], 0, 1, 2, 3, 4, 5, 6, 7);
                p[128 * t + 64] = __builtin_shufflevector(lo[2 * t], lo[2 * t + 1], 0, 1, 2, 3, 4, 5, 6, 7);
            }
            if constexpr (MODE == RX_FWD) {
                blk_was = blk;
                er_was = er;
                if (kb == 1 && j < nJ - 1) *reinterpret_cast<float2*>(mine) = make_float2(blk, er);
            }
        };
        weigh_tile(0);
        if (chunk > 0) {
            float pt = 0.f;   // q . n~ of what lies before the chunk, a piece at a time
#pragma unroll
            for (int n = 0; n < Cfg::NE; n++) {
                state_wait(n);
                __syncthreads();
                if (D == 256) piece(n + 3);
                if constexpr (MODE == RX_FWD) {
                    if (kb == 0) {
#pragma unroll
                        for (int s = NS / Cfg::NE * n; s < NS / Cfg::NE * (n + 1); s++) {
                            const f32x4 n0 = *reinterpret_cast<const f32x4*>(nvl + 8 * h + KW * s), n1 = *reinterpret_cast<const f32x4*>(nvl + 8 * h + KW * s + 4);
                            const f32x8 qv = __builtin_convertvector(xf[s], f32x8);
#pragma unroll
                            for (int e = 0; e < 8; e++) pt = fmaf(qv[e], e < 4 ? n0[e] : n1[e - 4], pt);
                        }
                    }
                }
            }
            bsum = dec * pt;
        } else {
            __syncthreads();
        }
        for (int v = 1; v < nJ; v++) {
            weigh_tile(v);
            __syncthreads();
        }
        if constexpr (MODE == RX_FWD) {
            if (kb == 0) {
                add_own();
                if (rb == 1) mine[0] = bsum;
            }
        }
        __syncthreads();
        if constexpr (MODE == RX_FWD) {
            if (kb == rb) {
                if (kb == 1) {   // the block on the diagonal, onto what the first block's wave has
                    bsum = mine[0];
                    add_own();
                }
                const float b = sum_halves(bsum);
                if (h == 0) bex[rb * 32 + c32] = b;
            }
        }
        __syncthreads();
    } else {
        dma_wait();
        __syncthreads();
        frag xf[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) xf[s] = rrd.read(xtile, rb, s);
#pragma unroll
        for (int s = 0; s < NS; s++) pin(xf[s]);
        __syncthreads();   // X's tile is free; the rows' scalars are there
        row_scalars();
        SwzTransReader<T, D> vrd;
        vrd.init(lane, NC * kb);
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int x = 0; x < 16; x++) acc[c][x] = 0.f;
        if (D == 128 || chunk == 0) {
#pragma unroll
            for (int j = 1; j <= AHEAD; j++) copy_y1(j);
        }
        if (chunk == 0) {
#pragma unroll
            for (int j = 1; j < AHEAD; j++) copy_y2(j);
            dma_wait();
            __syncthreads();
        } else {
#pragma unroll
            for (int n = 0; n < Cfg::NE; n++) {
                const T* const th = e_hi(n);
                const T* const tl = e_lo(n);
                constexpr int N = Cfg::E_ROWS / KW * NC, PF = 3;   // products (of either term), fragments under way
                frag vf[PF], vl[PF];
                auto rd = [&](int k) __attribute__((always_inline)) {
                    vf[k % PF] = vrd.read(th, KW * (k / NC), k % NC);
                    vl[k % PF] = vrd.read(tl, KW * (k / NC), k % NC);
                };
#pragma unroll
                for (int k = 0; k < PF - 1; k++) rd(k);
#pragma unroll
                for (int k = 0; k < N; k++) {
                    if (k + PF - 1 < N) rd(k + PF - 1);
                    R::mma(acc[k % NC], vf[k % PF], xf[Cfg::E_ROWS / KW * n + k / NC]);
                    R::mma(acc[k % NC], vl[k % PF], xf[Cfg::E_ROWS / KW * n + k / NC]);
                    __builtin_amdgcn_sched_barrier(0);
                }
                // (the products stay on this side of the barrier: moved behind it, they kept the fragments of all pieces in registers)
#pragma unroll
                for (int c = 0; c < NC; c++) pin(acc[c]);
                if (D == 128 && n == Cfg::NE - 1) {   // (Y2's second and third tile are under way)
                    if (nJ > 2) dma_wait_but<2 * PW>();
                    else dma_wait();
                } else {
                    state_wait(n);
                }
                __syncthreads();
                if constexpr (D == 256) {
                    piece(n + 3);
                    if (n == Cfg::NE - 3) copy_y1(1);   // (the place of that piece)
                    if (n == Cfg::NE - 2) copy_y2(0);
                } else {
                    if (n < AHEAD) copy_y2(n);
                }
            }
            if constexpr (MODE == RX_FWD) {
#pragma unroll
                for (int c = 0; c < NC; c++)
#pragma unroll
                    for (int x = 0; x < 16; x++) acc[c][x] *= dec;
            } else {
                const float rank1 = dec * dbv, decn = dec * inv_n;
                const T* qrow = reinterpret_cast<const T*>(a.Qrow) + offA + (size_t)rowc * rsA;
                float rph = 0.f;   // q_i . dQ_i of the state part: the row sums of dD over the keys before the chunk
#pragma unroll
                for (int c = 0; c < NC; c++) {
                    float rp = 0.f;
#pragma unroll
                    for (int a4 = 0; a4 < 4; a4++) {
                        const int col = 32 * (NC * kb + c) + 8 * a4 + 4 * h;
                        const f32x4 nv = *reinterpret_cast<const f32x4*>(nvl + col);
                        const f32x4 qv = __builtin_convertvector(*reinterpret_cast<const typename R::vec4*>(qrow + col), f32x4);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            acc[c][4 * a4 + e] = fmaf(rank1, nv[e], acc[c][4 * a4 + e] * decn);
                            rp = fmaf(acc[c][4 * a4 + e], qv[e], rp);
                        }
                    }
                    rph += rp;
                }
                rph = sum_halves(rph);
                if (h == 0) rpx[(rb * 2 + kb) * 32 + c32] = rph;
            }
        }
        for (int v = 1; v <= nJ; v++) {
            const int j = v - 1;
            constexpr int PF = 4;   // fragments under way
            frag vf[PF], p[4], pl[4];
            const T* const y2 = y2_at(j);
            auto rd = [&](int n) __attribute__((always_inline)) { vf[n % PF] = vrd.read(y2, KW * (n / NC), n % NC); };
#pragma unroll
            for (int n = 0; n < PF - 1; n++) rd(n);
#pragma unroll
            for (int g = 0; g < 4; g++) {   // 16 keys each
                const frag* const pp = reinterpret_cast<const frag*>(p_block(g >> 1)) + 128 * (g & 1) + lane;
                p[g] = pp[0];
                pl[g] = pp[64];
            }
            __syncthreads();
            const int n1 = v + AHEAD, n2 = v - 1 + AHEAD;   // the tiles to request
            const bool spread = n1 < nJ && n1 < full_tiles;
            if (!spread) { copy_y1(n1); copy_y2(n2); }
            auto contract = [&](auto groups_tag) __attribute__((always_inline)) {
                constexpr int N = decltype(groups_tag)::value * NC, EVERY = 4 * NC / (2 * PW) > 0 ? 4 * NC / (2 * PW) : 1, EACH = 2 * PW / (4 * NC) > 0 ? 2 * PW / (4 * NC) : 1;
#pragma unroll
                for (int n = 0; n < N; n++) {
                    if (n + PF - 1 < N) rd(n + PF - 1);
                    R::mma(acc[n % NC], vf[n % PF], p[n / NC]);
                    R::mma(acc[n % NC], vf[n % PF], pl[n / NC]);
                    if (n % EVERY == 0 && spread) {
#pragma unroll
                        for (int i = 0; i < EACH; i++) {
                            const int k = (n / EVERY) * EACH + i;
                            if (k < PW) tdma.issue_range(y1_at(n1), Y1 + (size_t)GRAN * n1 * rsA, k, k + 1, ra);
                            else tdma.issue_range(y2_at(n2), Y2 + (size_t)GRAN * n2 * rsA, k - PW, k - PW + 1, ra);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            // (the second keys of the last tile lie above the diagonal of the first rows)
            if (j == nJ - 1 && rb == 0) contract(std::integral_constant<int, 2>{});
            else contract(std::integral_constant<int, 4>{});
            // the next step's tiles have landed: everything but what the newest AHEAD - 1 steps have requested, 2 PW loads each
            if (v >= AHEAD && n1 < nJ) dma_wait_but<(AHEAD - 1) * 2 * PW>();
            else dma_wait();
            __syncthreads();
        }
    }
    // ---- epilogue
    constexpr int CPR = D * (int)sizeof(T) / 16, RB = D * (int)sizeof(T) + 16, NP = 64 * CPR / 512;
    __syncthreads();   // the row sums are there; every wave is done with the pool
    if constexpr (MODE == RX_FWD) {
        const float b = bex[rb * 32 + c32];
        onorm = 1.0f / (fmaxf(fabsf(b), __expf(-m_row)) + 1e-6f);
        if (producer && kb == 0 && h == 0 && row < S) a.Bsum[hoff + row] = b;
    } else {
        if (a.chunk_len > 0 && producer && kb == 0) {
            const float v = chunk > 0 ? rpx[rb * 2 * 32 + c32] + rpx[(rb * 2 + 1) * 32 + c32] : 0.f;
            if (h == 0 && row < S) a.rowinter[hoff + row] = v;
        }
    }
    char* const lo_out = smem + GRAN * RB;   // forward: what rounding h loses
    if (!producer) {
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int a4 = 0; a4 < 4; a4++) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = rounded_product(acc[c][4 * a4 + e], onorm);
            const int at = (32 * rb + c32) * RB + (32 * (NC * kb + c) + 8 * a4 + 4 * h) * (int)sizeof(T);
            if constexpr (MODE == RX_FWD) {
                typename R::vec4 hi, lo;
                R::cvt4_split(v, hi, lo);
                *reinterpret_cast<typename R::vec4*>(smem + at) = hi;
                *reinterpret_cast<typename R::vec4*>(lo_out + at) = lo;
            } else {
                *reinterpret_cast<typename R::vec4*>(smem + at) = R::cvt4(v);
            }
        }
    }
    __syncthreads();
    {
        char* const gout = reinterpret_cast<char*>(a.out) + (offO + (size_t)r0 * rsO) * sizeof(T);
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int c = tid + 512 * i, rr = c / CPR, cc = c % CPR;
            const uint4 v = *reinterpret_cast<const uint4*>(smem + rr * RB + 16 * cc);
            if (r0 + rr < S) {
                *reinterpret_cast<uint4*>(gout + (size_t)rr * rsO * sizeof(T) + 16 * cc) = v;
                if constexpr (MODE == RX_FWD) {
                    if (a.out_lo)
                        *reinterpret_cast<uint4*>(reinterpret_cast<char*>(a.out_lo) + (hoff + r0 + rr) * D * sizeof(T) + 16 * cc) =
                            *reinterpret_cast<const uint4*>(lo_out + rr * RB + 16 * cc);
                }
            }
        }
    }
#endif
}

template <typename T, int D, int MODE>
static int launch_rowx_t(const RowArgs& a, hipStream_t st) {
    using Cfg = RowxCfg<T, D>;
    const int most = a.chunk_len > 0 && a.chunk_len < a.NG * GRAN ? a.chunk_len : a.NG * GRAN;   // keys a row may meet
    if (most > RX_MOST_KEYS) return MLSTM_ESHAPE;
    if (MODE == RX_FWD && a.O) return MLSTM_ESHAPE;   // (the gate takes h as it was before it is rounded)
    if (hipError_t e = lds_limit_once<rowx_kernel<T, D, MODE>>((int)Cfg::lds_bytes(RX_MOST_KEYS)); e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((rowx_kernel<T, D, MODE>), dim3(a.BH * a.NG), dim3(512), Cfg::lds_bytes(most), st, a);
    return (int)hipGetLastError();
}

template <typename T>
static int launch_rowx_m(int mode, int D, const RowArgs& a, hipStream_t st) {
    if (mode == RX_FWD) return D == 128 ? launch_rowx_t<T, 128, RX_FWD>(a, st) : launch_rowx_t<T, 256, RX_FWD>(a, st);
    return D == 128 ? launch_rowx_t<T, 128, RX_DQ>(a, st) : launch_rowx_t<T, 256, RX_DQ>(a, st);
}

int launch_rowx_kernel(int mode, int dtype, int D, const RowArgs& a, hipStream_t st) {
    return dtype == MLSTM_F16 ? launch_rowx_m<_Float16>(mode, D, a, st) : launch_rowx_m<__bf16>(mode, D, a, st);
}

}  // namespace mlstm
