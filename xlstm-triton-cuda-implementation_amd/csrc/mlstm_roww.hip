// Row-parallel tile kernel for the 16-bit types at D >= 128 where few workgroups would run: the same math and, element by
// element, the same order of operations as mlstm_row8.hip, hence the same bits, on half as many rows per workgroup and with every
// key tile's work spread over all waves.
//
// What bounds a small call is one workgroup's walk of its key tiles, and in the eight-wave producer / consumer kernel that walk
// takes 1.2 us per 64 keys (products, weights, hand-over, products, one tile after the other) whatever the number of workgroups.
// There is no online maximum (the row maximum is a prefix maximum of the gates), so the weights of several tiles can be formed
// side by side; only the accumulation over the keys is a chain.  A workgroup here owns 64 rows (RB = 2: eight waves) or 32 (RB = 1: four) and takes
// 128 keys at a time in two phases:
//   phase 1   wave (rb, kb) = (row block of 32, key block of 32):  S^T = K Q^T (dQ pass: dC^T = V dH^T) for its 32 x 32 block, gate
//             weights, the 16-bit weights and the block's share of the row sums to LDS;
//   phase 2   wave (rb, c) = (row block, D / 4 of the output columns):  H^T += V^T P^T (dQ^T += K^T G^T) over the 128 keys.
// Phase 2's chain of products per accumulator is that of the consumers of mlstm_row8.hip, phase 1's blocks are those of its
// producers, and the row sums are added up in its order.  In chunks the state of the previous chunk goes first, as there.
// Replaces, like mlstm_row8.hip, mlstm_matmul_kernel (mlstm_matmul.py:38-101) and the dQ loop of mlstm_matmul_kernel_backward
// (mlstm_matmul.py:239-267).
#include <type_traits>
#include "mlstm_gates.h"

namespace mlstm {

constexpr int RW_FWD = 0, RW_DQ = 1;

template <typename T, int D, int RB>
struct RowwCfg {
    static constexpr size_t TILE_BYTES = (size_t)GRAN * D * sizeof(T);
    static constexpr int NST = D == 256 ? 1 : 2;                       // stages of 128 keys for each of Y1 and Y2: 128 KB in all
    static constexpr size_t POOL_BYTES = 4 * NST * TILE_BYTES;
    static constexpr size_t P_BYTES = 4 * RB * 2 * 64 * 16;            // [key block][row block][16 keys][lane] x 16 B
    static constexpr size_t PART_BYTES = 4 * RB * 64 * 8;              // [key block][row block][lane] x {sum, row factor}; dQ pass: [column block][row block][lane]
    static constexpr size_t MISC_FLOATS = RB * 2 * 32 + RB * 32 * 2 + D + RW_MOST_KEYS / GRAN;   // row sums, 1/n and db, vector state, granule distances
    static size_t lds_bytes(int keys) { return POOL_BYTES + P_BYTES + PART_BYTES + MISC_FLOATS * 4 + (size_t)keys * 8 + GRAN * 4; }
};

// FUSED (forward, uncut sequences): the gates too, see RowArgs::gate_F
template <typename T, int D, int MODE, int RB, bool FUSED>
__global__ __launch_bounds__(256 * RB) void roww_kernel(RowArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    using R = Tr<T>;
    using Cfg = RowwCfg<T, D, RB>;
    constexpr int NT = 256 * RB, ROWS = 32 * RB;
    typedef typename R::frag frag;
    static_assert(R::HALF && (D == 128 || D == 256), "16-bit types, D = 128 or 256");
    constexpr int KW = R::KW, NS = D / KW, NC = D / 128, NST = Cfg::NST;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    frag* const pbuf = reinterpret_cast<frag*>(smem + Cfg::POOL_BYTES);
    float* const part = reinterpret_cast<float*>(smem + Cfg::POOL_BYTES + Cfg::P_BYTES);
    float* const bex = part + Cfg::PART_BYTES / 4;         // [rb][kh][32]
    float* const stat = bex + RB * 2 * 32;                 // [rb][32] x {1/n, db}
    float* const nvl = stat + RB * 32 * 2;                 // [D]
    float* const sdg = nvl + D;                            // granule of the rows minus granule j
    float* const sek = sdg + RW_MOST_KEYS / GRAN;          // ek of the keys, then alpha, then the block maxima

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5, c32 = lane & 31;
    const int rb = wave >> 2, kb = wave & 3;               // phase 1: key block kb; phase 2: column blocks NC * kb ...
    int S = a.S, NG = a.NG;
    int bh, qt;
    {
        // heaviest row tiles first over all heads; with a multiple of 8 heads a head's tiles run on one XCD
        const int bid = blockIdx.x, nQT = NG * (GRAN / ROWS);
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
    size_t offA = a.la.head(bh), offB = a.lb.head(bh), offH = MODE == RW_DQ ? a.lh.head(bh) : 0;
    int chunk = 0;   // in chunks positions count from the chunk's first one (see mlstm_row8.hip)
    if (a.chunk_len > 0) {
        chunk = (qt * ROWS) / a.chunk_len;
        const int p0 = chunk * a.chunk_len;
        hoff += p0; poff += p0; goff += p0 / GRAN;
        offA += (size_t)p0 * rsA; offB += (size_t)p0 * rsB; offH += (size_t)p0 * rsH;
        S -= p0; qt -= p0 / ROWS;
    }
    const int r0 = ROWS * qt, gt = r0 / GRAN;
    const int nJ = gt + 1;                                  // key tiles; the last one is the rows' own
    const int row = r0 + 32 * rb + c32, rowc = row < S ? row : S - 1;
    const size_t rsX = MODE == RW_FWD ? rsA : rsB, offX = MODE == RW_FWD ? offA : offB;
    const size_t rsO = MODE == RW_FWD ? rsB : rsA, offO = MODE == RW_FWD ? offB : offA;
    const T* X = reinterpret_cast<const T*>(a.X) + offX;
    const T* Y1 = reinterpret_cast<const T*>(a.Y1) + offA;
    const T* Y2 = reinterpret_cast<const T*>(a.Y2) + offA;
    const int full_tiles = S / GRAN;
    const int keys = GRAN * nJ;
    float* const sal = sek + keys;
    float* const sam = sal + keys;

    // tiles of 64 rows in the pool: Y1 of stage st at 2 st + t, Y2 behind all of those
    auto tile_at = [&](int n) { return reinterpret_cast<T*>(smem + (size_t)n * Cfg::TILE_BYTES); };
    auto y1_at = [&](int r, int t) { return tile_at(2 * (r & (NST - 1)) + t); };
    auto y2_at = [&](int r, int t) { return tile_at(2 * NST + 2 * (r & (NST - 1)) + t); };
    TileDma<T, D, GRAN, NT> tdma;
    tdma.init(tid);
    const auto ra = tdma.rows(tid, (unsigned)(rsA * sizeof(T)));
    auto copy_tile = [&](T* dst, const T* src, int j) {
        if (j < full_tiles) tdma.issue(dst, src + (size_t)GRAN * j * rsA, ra);
        else tile_dma_rolled<T, D, GRAN, NT>(dst, src, GRAN * j, S, tid, rsA);
    };
    auto copy_y1 = [&](int r) {
        copy_tile(y1_at(r, 0), Y1, 2 * r);
        if (2 * r + 1 < nJ) copy_tile(y1_at(r, 1), Y1, 2 * r + 1);
    };
    auto copy_y2 = [&](int r) {
        copy_tile(y2_at(r, 0), Y2, 2 * r);
        if (2 * r + 1 < nJ) copy_tile(y2_at(r, 1), Y2, 2 * r + 1);
    };
    // The gates of the head's granules up to the rows' own, granule wave + NW k in turn k, are requested first: copies into LDS (the places of
    // their key weights), so that a counted wait can leave the tiles behind them under way while the gates are formed.  (16-bit values one
    // by one: the dword that holds one reaches beyond the tensor at either of its ends.)  Two launches / one, forward, us: 1 x 64 x 128 7.9 / 6.3, 1 x 320 10.9 / 9.7, 1 x 640 13.4 / 13.1 (a granule is 250
    // instructions, 100 of them its logarithms, and a workgroup forms all of its head's: 2 us of a CU for ten), 8 x 1000 17.7 / 17.6, 15 x 1001
    // 22.0 / 19.0, 16 x 256 9.9 / 8.3; D = 256, 1 x 640 15.8 / 15.7, 8 x 1000 22.7 / 22.1, 24 x 1000 29.0 / 26.7, 100 x 128 11.6 / 9.2.
    constexpr int NW = NT / 64, TURNS = FUSED ? RW_MOST_KEYS / GRAN / NW : 1;
    if constexpr (FUSED) {
        const size_t off = a.lg.head(bh), ss = (size_t)a.lg.ss;
        auto request = [&](auto gate, auto&& copy) __attribute__((always_inline)) {
            typedef decltype(gate) G;
#pragma unroll
            for (int k = 0; k < TURNS; k++) {
                const int g = tid / 64 + NW * k;
                if (g < nJ) {
                    const int t = g * GRAN + lane;
                    const size_t at = off + (size_t)(t < S ? t : S - 1) * ss;
                    copy(reinterpret_cast<const G*>(a.gate_F) + at, __builtin_amdgcn_readfirstlane(lds_offset_of(sek + GRAN * g)));
                    copy(reinterpret_cast<const G*>(a.gate_I) + at, __builtin_amdgcn_readfirstlane(lds_offset_of(sal + GRAN * g)));
                }
            }
        };
        if (a.gate_dtype == MLSTM_F32) request(0.f, dma4);
        else request((unsigned short)0, dma2);
    }
    // (plain loads first: what they bring is used behind the copies' issue)
    const double g_rows = FUSED ? 0.0 : a.G2[goff + gt], g_mine = FUSED ? 0.0 : a.G2[goff + (tid < nJ ? tid : 0)], g_end = chunk > 0 ? a.G2[goff - 1] : 0.0;
    float beta_row = FUSED ? 0.f : a.beta2[poff + rowc];
    const float beta_end = chunk > 0 ? a.beta2[poff - 1] : 0.f;
    const float n_mine = chunk > 0 && tid < D ? a.Nst[((size_t)bh * a.n_states + chunk - 1) * D + tid] : 0.f;
    float m_row = !FUSED && (MODE == RW_FWD || kb == 0) ? a.M[hoff + rowc] : 0.f;
    const float b_row = MODE == RW_DQ && kb == 0 ? a.Bin[hoff + rowc] : 0.f;
    // piece i of a pair of complete tiles j, j + 1
    auto copy_piece = [&](const T* src, T* d0, T* d1, int j, int i) {
        constexpr int PW = TileDma<T, D, GRAN, NT>::PER_WAVE;
        const int t = i / PW, n = i % PW;
        tdma.issue_range(t ? d1 : d0, src + (size_t)GRAN * (j + t) * rsA, n, n + 1, ra);
    };
    // the share of slot n of `slots` in the copy of a pair of tiles
    auto pieces = [&](int n, int slots, auto&& f) __attribute__((always_inline)) {
        constexpr int PP = 2 * TileDma<T, D, GRAN, NT>::PER_WAVE;
#pragma unroll
        for (int i = 0; i < PP; i++)
            if (i >= n * PP / slots && i < (n + 1) * PP / slots) f(i);
    };
    // ---- prologue.  The rows' own operand, the state of the previous chunk and the first keys are requested at once, as far as the
    // pool holds them.  D = 256: X in tile 3 (then the last state tile), state tiles in 0, 1, 2; D = 128: X in tile 3 (Y1's second
    // stage), the state in Y2's second stage, the first keys in the first stages.
    const T* const xtile = tile_at(3);
    {
        TileDma<T, D, ROWS, NT> xdma;
        xdma.init(tid);
        const auto rx = xdma.rows(tid, (unsigned)(rsX * sizeof(T)));
        if (r0 + ROWS <= S) xdma.issue(tile_at(3), X + (size_t)r0 * rsX, rx);
        else tile_dma_rolled<T, D, ROWS, NT>(tile_at(3), X, r0, S, tid, rsX);
    }
    const T* const Cst = chunk > 0 ? reinterpret_cast<const T*>(a.Cst) + ((size_t)bh * a.n_states + chunk - 1) * D * D : nullptr;
    if (chunk > 0) {
        if constexpr (NST == 1) {
#pragma unroll
            for (int t = 0; t < 3; t++) tdma.issue(tile_at(t), Cst + (size_t)GRAN * t * D);
        } else {
#pragma unroll
            for (int t = 0; t < 2; t++) tdma.issue(tile_at(6 + t), Cst + (size_t)GRAN * t * D);
        }
    }
    if (NST == 2 || chunk == 0) copy_y1(0);
    if (NST == 2) copy_y2(0);
    GateLocal gown{};     // of the rows' granule, in the wave that forms it
    GateGlobal gbeta{};
    double gbase = 0.0;
    if constexpr (FUSED) {
        // (in the row sums' place until those need it: totals and maxima of the granules, beta and m of the rows' own)
        double* const sT = reinterpret_cast<double*>(part);
        double* const sP = sT + RW_MOST_KEYS / GRAN;
        float* const own = reinterpret_cast<float*>(sP + RW_MOST_KEYS / GRAN);   // [beta, m][64]
        float c = 0.f;
        // all but the copies behind the gates': the rows of X and one or two tiles of Y1 (NST == 2: and of Y2), as many of a wave whatever their rows
        constexpr int PX = TileDma<T, D, ROWS, NT>::PER_WAVE, PT = NST * TileDma<T, D, GRAN, NT>::PER_WAVE;
        if (nJ > 1) dma_wait_but<PX + 2 * PT>();
        else dma_wait_but<PX + PT>();
        // N turns side by side: a granule's 180 instructions are one chain of 1800 cycles
        auto turns = [&](auto n_tag) __attribute__((always_inline)) {
            constexpr int N = decltype(n_tag)::value;
            float lf[N], ig[N], cs[N], al[N];
            GateLocal vs[N];
#pragma unroll
            for (int k = 0; k < N; k++) {
                const int t = (wave + NW * k) * GRAN + lane, tr = (wave + NW * k < nJ ? t : lane);   // (a turn too many: some place that is there)
                unsigned x = __builtin_bit_cast(unsigned, sek[tr]), y = __builtin_bit_cast(unsigned, sal[tr]);
                if (a.gate_dtype == MLSTM_F16) {
                    x = __builtin_bit_cast(unsigned, (float)__builtin_bit_cast(_Float16, (unsigned short)x));
                    y = __builtin_bit_cast(unsigned, (float)__builtin_bit_cast(_Float16, (unsigned short)y));
                } else if (a.gate_dtype == MLSTM_BF16) {
                    x <<= 16;
                    y <<= 16;
                }
                const GateIn in{__builtin_bit_cast(float, x), 0.f, __builtin_bit_cast(float, y)};
                lf[k] = forget_log(in, t, a.gate_form);
                ig[k] = in.i;
            }
#pragma unroll
            for (int k = 0; k < N; k++) cs[k] = wave_scan_inclusive<OpAdd>((wave + NW * k) * GRAN + lane < S ? lf[k] : 0.0f);
#pragma unroll
            for (int k = 0; k < N; k++) {
                const bool ok = (wave + NW * k) * GRAN + lane < S;
                al[k] = ok ? ig[k] - cs[k] : -INFINITY;
                vs[k] = gates_local(al[k], ok, lane);
            }
#pragma unroll
            for (int k = 0; k < N; k++) {
                const int g = wave + NW * k, t = g * GRAN + lane;
                if (g < nJ) {
                    const float tot = last_lane(cs[k]);
                    if (lane == 0) { sT[g] = (double)tot; sP[g] = (double)vs[k].p; }
                    sek[t] = vs[k].ek2;
                    sal[t] = vs[k].alpha2;
                    if ((lane & 31) == 0) sam[2 * g + (lane >> 5)] = vs[k].c0;
                    c = cs[k];
                    gown = vs[k];
                }
            }
        };
        if (nJ <= NW) turns(std::integral_constant<int, 1>{});
        else if (TURNS == 2 || nJ <= 2 * NW) turns(std::integral_constant<int, 2>{});
        else turns(std::integral_constant<int, TURNS>{});
        __syncthreads();
        if (wave == (gt & (NW - 1)) || wave == ((gt + 1) & (NW - 1))) {   // (the wave that holds the rows' granule, and another)
            double incl, excl, mx;
            granule_scan(lane < nJ ? sT[lane] : 0.0, lane < nJ ? sP[lane] : -INFINITY, 0.0, lane, incl, excl, mx);
            const double before = before_lane(mx, lane), Gg = readlane_d(excl, gt);
            if (wave == (gt & (NW - 1))) {
                const int t = gt * GRAN + lane;
                gbeta = gates_global(c, gown.loc, t < S, Gg, readlane_d(before, gt));
                gbase = Gg;
                own[lane] = gbeta.beta2;
                own[GRAN + lane] = gbeta.m;
            } else if (lane < nJ) {
                sdg[lane] = (float)(product_apart(Gg, LOG2E_D) - product_apart(excl, LOG2E_D));
            }
        }
    } else {
        for (int t = tdma.wave_s; t < nJ; t += NT / 64) {
            dma4(a.ek2 + poff + GRAN * t + lane, __builtin_amdgcn_readfirstlane(lds_offset_of(sek + GRAN * t)));
            dma4(a.alpha2 + poff + GRAN * t + lane, __builtin_amdgcn_readfirstlane(lds_offset_of(sal + GRAN * t)));
        }
        if (tid < GRAN) dma4(a.amax2 + goff * 2 + tid, __builtin_amdgcn_readfirstlane(lds_offset_of(sam)));   // (2 nJ of them count; padded array)
    }
    float crow_base = -0.5f * __log2f((float)D) - beta_row;
    float dec = 0.f;   // the row's decay since the end of the previous chunk
    if (chunk > 0) dec = fast_exp2(beta_end - beta_row + (float)(g_rows - g_end));
    if (!FUSED && tid < nJ) sdg[tid] = (float)(g_rows - g_mine);
    if (chunk > 0 && tid < D) nvl[tid] = n_mine;
    frag hfr[NS];
    if constexpr (MODE == RW_DQ) {
        if (kb == 0) {
            const T* hrow = reinterpret_cast<const T*>(a.Hin) + offH + (size_t)rowc * rsH;
#pragma unroll
            for (int s = 0; s < NS; s++) hfr[s] = frag_rowmajor<T>(hrow, s, h);
        }
    }
    SwzRowReaderX<T, D> rrd;
    rrd.init(lane);
    SwzTransReader<T, D> vrd;
    vrd.init(lane, NC * kb);
    f32x16 acc[NC];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int x = 0; x < 16; x++) acc[c][x] = 0.f;
    dma_wait();
    __syncthreads();
    if constexpr (FUSED) {
        const float* const own = part + 4 * (RW_MOST_KEYS / GRAN);
        beta_row = own[rowc - GRAN * gt];
        m_row = own[GRAN + rowc - GRAN * gt];
        crow_base = -0.5f * __log2f((float)D) - beta_row;
        // (of two workgroups with rows of a granule the first one writes its gates)
        if (wave == (gt & (NW - 1)) && (r0 & (GRAN - 1)) == 0) {
            const int t = gt * GRAN + lane;
            store_local(gown, poff + t, goff + gt, lane, const_cast<float*>(a.alpha2), const_cast<float*>(a.ek2), const_cast<float*>(a.amax2));
            store_global(gbeta, t < S, gbase, poff + t, hoff + t, goff + gt, lane, const_cast<float*>(a.beta2), const_cast<double*>(a.G2), const_cast<float*>(a.M));
        }
    }
    frag xf[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) xf[s] = rrd.read(xtile, rb, s);
    if constexpr (MODE == RW_DQ) {   // 1/n and db of the rows (see row_stats), for this kernel and for the column kernel
        if (kb == 0) {
            float dot = 0.f;
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int e = 0; e < R::EPL; e++) dot += (float)xf[s][e] * (float)hfr[s][e];
            float inv = 0.f, dbr = 0.f;
            row_stats_of(sum_halves(dot), b_row, m_row, inv, dbr);
            if (h == 0) {
                *reinterpret_cast<float2*>(stat + (32 * rb + c32) * 2) = make_float2(inv, dbr);
                a.inv_n[poff + row] = row < S ? inv : 0.f;   // (rows behind the sequence: zeros, see mlstm_row.hip)
                a.db[poff + row] = row < S ? dbr : 0.f;
            }
        }
    }
#pragma unroll
    for (int s = 0; s < NS; s++) pin(xf[s]);
    __syncthreads();   // X's tile is free; the rows' scalars are there
    if constexpr (NST == 2) {
        if (nJ > 2) copy_y1(1);
    }

    // G groups of 16 contraction rows out of consecutive tiles, times the fragments operand(g)
    auto chain = [&](auto groups_tag, auto&& tile, auto&& operand, auto&& hook) {
        constexpr int G = decltype(groups_tag)::value;
        frag vf[2][NC], pf[2];
#pragma unroll
        for (int c = 0; c < NC; c++) vf[0][c] = vrd.read(tile(0), 0, c);
        pf[0] = operand(std::integral_constant<int, 0>{});
        static_for<G>([&](auto gc) __attribute__((always_inline)) {
            constexpr int g = decltype(gc)::value;
            if constexpr (g + 1 < G) {
#pragma unroll
                for (int c = 0; c < NC; c++) vf[(g + 1) & 1][c] = vrd.read(tile((g + 1) / 4), KW * ((g + 1) % 4), c);
                pf[(g + 1) & 1] = operand(std::integral_constant<int, g + 1>{});
            }
#pragma unroll
            for (int c = 0; c < NC; c++) R::mma(acc[c], vf[g & 1][c], pf[g & 1]);
            hook(gc);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    typedef std::integral_constant<int, 8> Eight;
    typedef std::integral_constant<int, 4> Four;
    float inv_n = 0.f, dbv = 0.f;
    if constexpr (MODE == RW_DQ) {
        const float2 st = *reinterpret_cast<const float2*>(stat + (32 * rb + c32) * 2);
        inv_n = st.x; dbv = st.y;
    }
    if (chunk > 0) {
        if constexpr (NST == 1) {
            tdma.issue(tile_at(3), Cst + (size_t)GRAN * 3 * D);
            chain(std::integral_constant<int, 12>{}, [&](int t) { return tile_at(t); }, [&](auto g) { return xf[decltype(g)::value]; }, [](auto) {});
            dma_wait();
            __syncthreads();
            copy_y1(0);
            chain(Four{}, [&](int) { return tile_at(3); }, [&](auto g) { return xf[12 + decltype(g)::value]; }, [](auto) {});
        } else {
            chain(Eight{}, [&](int t) { return tile_at(6 + t); }, [&](auto g) { return xf[decltype(g)::value]; }, [](auto) {});
        }
        if constexpr (MODE == RW_FWD) {
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int x = 0; x < 16; x++) acc[c][x] *= dec;
        } else {
            const float rank1 = dec * dbv, decn = dec * inv_n;
            const T* qrow = reinterpret_cast<const T*>(a.Qrow) + offA + (size_t)rowc * rsA;
#pragma unroll
            for (int c = 0; c < NC; c++) {
                float rp = 0.f;   // q_i . dQ_i of the state part: the row sums of dD over the keys before the chunk
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
                part[((NC * kb + c) * RB + rb) * 64 + lane] = rp;
            }
        }
    }

    // ---- the key tiles, two at a time
    const int nR = (nJ + 1) / 2, rr = r0 + 32 * rb;
    float bsum = 0.f;   // waves kb < 2: the row sums over the key blocks of parity kb, in the order of the keys
    const frag* const p = pbuf + rb * 2 * 64 + lane;
    auto weights = [&](auto g) { return p[((decltype(g)::value >> 1) * RB * 2 + (decltype(g)::value & 1)) * 64]; };
    auto none = [](auto) {};
    // weights of a block whose products are in s, by where it lies; blk, er: its share of the row sums
    auto weigh_element = [&](f32x16& s, int x, float ek, float er, float sc, float of, float& blk) __attribute__((always_inline)) {
        if constexpr (MODE == RW_FWD) {
            blk = fmaf(s[x], ek, blk);
            s[x] = (s[x] * ek) * er;
        } else {
            s[x] = (s[x] * sc + of) * ek;
        }
    };
    auto weigh = [&](f32x16& s, int k0, float crow, float& blk, float& er) __attribute__((always_inline)) {
        blk = 0.f; er = 0.f;
        if (k0 > rr) {             // above the diagonal
#pragma unroll
            for (int x = 0; x < 16; x++) s[x] = 0.f;
        } else if (k0 < rr) {      // below it: factorised weights
            er = fast_exp2(crow + sam[k0 / 32]);
            const float sc = inv_n * er, of = dbv * er;
#pragma unroll
            for (int a4 = 0; a4 < 4; a4++) {
                const f32x4 ek = *reinterpret_cast<const f32x4*>(sek + k0 + 8 * a4 + 4 * h);
#pragma unroll
                for (int c = 0; c < 4; c++) weigh_element(s, 4 * a4 + c, ek[c], er, sc, of, blk);
            }
        } else {                   // on it
#pragma unroll
            for (int a4 = 0; a4 < 4; a4++) {
                const f32x4 al = *reinterpret_cast<const f32x4*>(sal + k0 + 8 * a4 + 4 * h);
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const int x = 4 * a4 + c;
                    float e = fast_exp2(al[c] + crow);
                    if (8 * a4 + 4 * h + c > c32) e = 0.f;
                    if constexpr (MODE == RW_FWD) {
                        s[x] *= e;     // (its share of the row sums: behind the loop)
                    } else {
                        s[x] = (s[x] * inv_n + dbv) * e;
                    }
                }
            }
        }
    };
    auto put_weights = [&](const f32x16& s, float blk, float er) __attribute__((always_inline)) {
        frag* const q = pbuf + (kb * RB + rb) * 2 * 64 + lane;
        q[0] = R::from_acc(s, 0);
        q[64] = R::from_acc(s, 1);
        if constexpr (MODE == RW_FWD) *reinterpret_cast<float2*>(part + ((kb * RB + rb) * 64 + lane) * 2) = make_float2(blk, er);
    };
    // S^T of the wave's block of round r, with something between the products
    auto products = [&](f32x16& s, int r, auto&& hook) __attribute__((always_inline)) {
        const T* y1 = y1_at(r, kb >> 1);
        constexpr int AHEAD = 4;
        frag kf[NS];
#pragma unroll
        for (int n = 0; n < AHEAD; n++) kf[n] = rrd.read(y1, kb & 1, n);
        static_for<NS>([&](auto nc) __attribute__((always_inline)) {
            constexpr int n = decltype(nc)::value;
            if constexpr (n + AHEAD < NS) kf[n + AHEAD] = rrd.read(y1, kb & 1, n + AHEAD);
            if constexpr (n == 0) {
#pragma unroll
                for (int x = 0; x < 16; x++) s[x] = 0.f;
            }
            R::mma(s, kf[n], xf[n]);
            hook(nc);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto add_row_sums = [&](bool two) __attribute__((always_inline)) {
        if constexpr (MODE == RW_FWD) {
            if (kb < 2) {   // (a block on the diagonal or above it has left zeros)
#pragma unroll
                for (int t = 0; t < 2; t++)
                    if (t == 0 || two) {
                        const float2 be = *reinterpret_cast<const float2*>(part + (((2 * t + kb) * RB + rb) * 64 + lane) * 2);
                        bsum = fmaf(be.x, be.y, bsum);
                    }
            }
        }
    };
    if constexpr (NST == 1) {
        for (int r = 0; r < nR; r++) {
            const bool two = 2 * r + 1 < nJ;
            dma_wait();
            __syncthreads();   // this round's Y1 has landed; phase 2 of the previous round is over
            // This round's Y2 is copied under phase 1.  A wave that issues its loads back to back waits for the memory pipeline (64 KB: 0.5 us
            // per round, measured), so they go between the products.
            const bool spread1 = two && 2 * r + 1 < full_tiles;
            const int j = 2 * r + (kb >> 1);
            if (!(spread1 && j < nJ)) copy_y2(r);
            auto phase1 = [&](auto spread_tag) __attribute__((always_inline)) {
                constexpr bool SPREAD = decltype(spread_tag)::value;
                f32x16 s;
                products(s, r, [&](auto n) {
                    if constexpr (SPREAD) pieces(decltype(n)::value, NS, [&](int i) { copy_piece(Y2, y2_at(r, 0), y2_at(r, 1), 2 * r, i); });
                });
                float blk, er;
                weigh(s, GRAN * j + 32 * (kb & 1), crow_base + sdg[j], blk, er);
                put_weights(s, blk, er);
            };
            if (j < nJ) {
                if (spread1) phase1(std::true_type{});
                else phase1(std::false_type{});
            }
            dma_wait();
            __syncthreads();
            add_row_sums(two);
            auto y2 = [&](int t) { return y2_at(r, t); };
            const bool spread2 = r + 1 < nR && 2 * r + 3 < nJ && 2 * r + 3 < full_tiles;   // the next round's Y1 under phase 2
            if (r + 1 < nR && !spread2) copy_y1(r + 1);
            if (spread2) chain(Eight{}, y2, weights, [&](auto g) { pieces(decltype(g)::value, 8, [&](int i) { copy_piece(Y1, y1_at(r + 1, 0), y1_at(r + 1, 1), 2 * r + 2, i); }); });
            else if (two) chain(Eight{}, y2, weights, none);
            else chain(Four{}, y2, weights, none);
        }
    } else {
        // D = 128 holds two stages of either operand: phase 1 of a round runs with phase 2 of the one before, its element-wise part between those
        // products, and only the 16-bit weights wait (in 8 registers) until every wave has read the ones before them.  A round is then bound by
        // its LDS traffic (192 KB and 64 KB of copies on 64 rows, 96 and 64 on 32) instead of by the chain products, weights, hand-over, products.
        // Forward, us, before / now: 1 x 640 x 128 on 32 rows 10.6 / 9.9, 8 x 1000 16.1 / 14.9, on 64 rows 15 x 1001 19.1 / 17.9, 4 x 4096 in chunks 13.2 / 12.5.
        f32x16 s;
        float blk = 0.f, er = 0.f;
        auto alone = [&](int r) __attribute__((always_inline)) {   // phase 1 by itself
            const int j = 2 * r + (kb >> 1);
            if (j < nJ) {
                products(s, r, none);
                weigh(s, GRAN * j + 32 * (kb & 1), crow_base + sdg[j], blk, er);
            }
        };
        alone(0);
        if (kb >> 1 < nJ) put_weights(s, blk, er);
        dma_wait();
        __syncthreads();   // the first weights, and Y1 of the second round
        for (int r = 0; r < nR; r++) {
            const bool two = 2 * r + 1 < nJ, next = r + 1 < nR;
            const int j = 2 * r + 2 + (kb >> 1), k0 = GRAN * j + 32 * (kb & 1);
            const bool mine = next && j < nJ;
            auto y2 = [&](int t) { return y2_at(r, t); };
            add_row_sums(two);
            // the copies of this round: Y1 two rounds ahead, Y2 one ahead, into the stages that are free since the last barrier
            auto with_next = [&](auto spread_tag) __attribute__((always_inline)) {
                constexpr bool SPREAD = decltype(spread_tag)::value;
                const float crow = crow_base + sdg[j], cmax = sam[k0 / 32];
                f32x4 ek[4];
#pragma unroll
                for (int a4 = 0; a4 < 4; a4++) ek[a4] = *reinterpret_cast<const f32x4*>(sek + k0 + 8 * a4 + 4 * h);
                products(s, r + 1, [&](auto n) {
                    if constexpr (SPREAD) pieces(decltype(n)::value, NS, [&](int i) { copy_piece(Y1, y1_at(r, 0), y1_at(r, 1), 2 * r + 4, i); });
                });
                er = fast_exp2(crow + cmax);
                blk = 0.f;
                const float sc = inv_n * er, of = dbv * er;
                chain(Eight{}, y2, weights, [&](auto gc) {
                    constexpr int g = decltype(gc)::value;
                    weigh_element(s, 2 * g, ek[g / 2][2 * (g % 2)], er, sc, of, blk);
                    weigh_element(s, 2 * g + 1, ek[g / 2][2 * (g % 2) + 1], er, sc, of, blk);
                    if constexpr (SPREAD) pieces(g, 8, [&](int i) { copy_piece(Y2, y2_at(r + 1, 0), y2_at(r + 1, 1), 2 * r + 2, i); });
                });
            };
            const bool below = mine && k0 < rr, spread = below && r + 2 < nR && 2 * r + 5 < nJ && 2 * r + 5 < full_tiles;
            if (spread) {
                with_next(std::true_type{});
            } else {
                if (r + 2 < nR) copy_y1(r + 2);
                if (next) copy_y2(r + 1);
                if (below) {
                    with_next(std::false_type{});
                } else {
                    if (next) alone(r + 1);
                    if (two) chain(Eight{}, y2, weights, none);
                    else chain(Four{}, y2, weights, none);
                }
            }
            if (!next) break;
            __syncthreads();   // every wave has read this round's weights
            if (mine) put_weights(s, blk, er);
            dma_wait();
            __syncthreads();   // the next ones are there, and the tiles requested above
        }
    }
    if constexpr (MODE == RW_FWD) {
        // The elements of the block on the diagonal go one by one onto the sum over the blocks before it.  They are formed once more here, where
        // that sum is, from tiles that are still in LDS: kept from phase 1 on, products and weights cost 64 moves in every round, and the
        // kernel 1 us of 11 (640 x 128).
        const int own = (r0 / 32 + rb) & 1;   // the block's place in its tile
        if (kb == own) {
            const T* const y1 = y1_at(nR - 1, (nJ - 1) & 1);
            f32x16 s;
#pragma unroll
            for (int x = 0; x < 16; x++) s[x] = 0.f;
#pragma unroll
            for (int n = 0; n < NS; n++) R::mma(s, rrd.read(y1, own, n), xf[n]);
            const float crow = crow_base + sdg[gt];
#pragma unroll
            for (int a4 = 0; a4 < 4; a4++) {
                const f32x4 al = *reinterpret_cast<const f32x4*>(sal + r0 + 32 * rb + 8 * a4 + 4 * h);
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    float e = fast_exp2(al[c] + crow);
                    if (8 * a4 + 4 * h + c > c32) e = 0.f;
                    bsum = fmaf(s[4 * a4 + c], e, bsum);
                }
            }
        }
    }
    // ---- epilogue
    uint4 og[D / 64];   // output gate: this thread's pieces, requested ahead of the barriers
    constexpr int CPR = D * (int)sizeof(T) / 16, ROWB = D * (int)sizeof(T) + 16, NP = ROWS * CPR / NT;
    static_assert(NP == D / 64, "pieces per thread");
    if constexpr (MODE == RW_FWD) {
        if (a.O) {
            const char* go = reinterpret_cast<const char*>(a.O) + (offB + (size_t)r0 * rsB) * sizeof(T);
#pragma unroll
            for (int i = 0; i < NP; i++) {
                const int c = tid + NT * i, rr = c / CPR, cc = c % CPR;
                og[i] = r0 + rr < S ? *reinterpret_cast<const uint4*>(go + (size_t)rr * rsB * sizeof(T) + 16 * cc) : uint4{0, 0, 0, 0};
            }
        }
        if (kb < 2) {
            if (chunk > 0) {   // what lies before the chunk: decay (q . n~), half of the contraction each
                const float* nst = nvl + 8 * h;
                float pt = 0.f;
                auto half_dot = [&](auto first_tag) {
                    constexpr int S0 = decltype(first_tag)::value;
#pragma unroll
                    for (int s = S0; s < S0 + NS / 2; s++) {
                        const f32x4 n0 = *reinterpret_cast<const f32x4*>(nst + KW * s), n1 = *reinterpret_cast<const f32x4*>(nst + KW * s + 4);
                        const f32x8 qv = __builtin_convertvector(xf[s], f32x8);
#pragma unroll
                        for (int e = 0; e < 4; e++) pt += fmaf(qv[e], n0[e], qv[4 + e] * n1[e]);
                    }
                };
                if (kb == 0) half_dot(std::integral_constant<int, 0>{});
                else half_dot(std::integral_constant<int, NS / 2>{});
                bsum = fmaf(pt, dec, bsum);
            }
            const float b = sum_halves(bsum);
            if (h == 0) bex[(rb * 2 + kb) * 32 + c32] = b;
        }
    }
    __syncthreads();   // the row sums are there; every wave is done with the pool
    float onorm = 1.0f;
    if constexpr (MODE == RW_FWD) {
        const float b = bex[(rb * 2 + 0) * 32 + c32] + bex[(rb * 2 + 1) * 32 + c32];
        onorm = 1.0f / (fmaxf(fabsf(b), __expf(-m_row)) + 1e-6f);
        if (kb == 0 && h == 0 && row < S) a.Bsum[hoff + row] = b;
    } else {
        if (a.chunk_len > 0 && kb == 0) {
            float v = 0.f;
            if (chunk > 0) {
#pragma unroll
                for (int half = 0; half < 2; half++) {
                    float rp = 0.f;
#pragma unroll
                    for (int d = 0; d < D / 64; d++) rp += part[((half * (D / 64) + d) * RB + rb) * 64 + lane];
                    rp = sum_halves(rp);
                    v = half ? v + rp : rp;
                }
            }
            if (h == 0 && row < S) a.rowinter[hoff + row] = v;
        }
    }
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int a4 = 0; a4 < 4; a4++) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = acc[c][4 * a4 + e] * onorm;
            *reinterpret_cast<typename R::vec4*>(smem + (32 * rb + c32) * ROWB + (32 * (NC * kb + c) + 8 * a4 + 4 * h) * (int)sizeof(T)) = R::cvt4(v);
        }
    __syncthreads();
    {
        char* const gout = reinterpret_cast<char*>(a.out) + (offO + (size_t)r0 * rsO) * sizeof(T);
        char* const gg = MODE == RW_FWD ? reinterpret_cast<char*>(a.out_gated) + (offB + (size_t)r0 * rsB) * sizeof(T) : nullptr;
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int c = tid + NT * i, rr = c / CPR, cc = c % CPR;
            const uint4 v = *reinterpret_cast<const uint4*>(smem + rr * ROWB + 16 * cc);
            if (r0 + rr < S) {
                *reinterpret_cast<uint4*>(gout + (size_t)rr * rsO * sizeof(T) + 16 * cc) = v;
                if constexpr (MODE == RW_FWD) {
                    if (a.O) {
                        typedef typename R::vec4 V4;
                        struct Pair { V4 lo, hi; };
                        const Pair hv = __builtin_bit_cast(Pair, v), ov = __builtin_bit_cast(Pair, og[i]);
                        Pair res;
                        res.lo = gate4<T>(hv.lo, ov.lo);
                        res.hi = gate4<T>(hv.hi, ov.hi);
                        *reinterpret_cast<Pair*>(gg + (size_t)rr * rsB * sizeof(T) + 16 * cc) = res;
                    }
                }
            }
        }
    }
#endif
}

template <typename T, int D, int MODE, int RB, bool FUSED>
static int launch_roww_f(const RowArgs& a, hipStream_t st) {
    using Cfg = RowwCfg<T, D, RB>;
    const int most = a.chunk_len > 0 && a.chunk_len < a.NG * GRAN ? a.chunk_len : a.NG * GRAN;   // keys a row may meet
    if (most > RW_MOST_KEYS) return MLSTM_ESHAPE;
    if (hipError_t e = lds_limit_once<roww_kernel<T, D, MODE, RB, FUSED>>((int)Cfg::lds_bytes(RW_MOST_KEYS)); e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((roww_kernel<T, D, MODE, RB, FUSED>), dim3(a.BH * a.NG * (2 / RB)), dim3(256 * RB), Cfg::lds_bytes(most), st, a);
    return (int)hipGetLastError();
}

template <typename T, int D, int MODE, int RB>
static int launch_roww_t(const RowArgs& a, hipStream_t st) {
    if constexpr (MODE == RW_FWD) {
        if (a.gate_F) return a.chunk_len > 0 ? MLSTM_EINVAL : launch_roww_f<T, D, MODE, RB, true>(a, st);
    }
    return launch_roww_f<T, D, MODE, RB, false>(a, st);
}

template <typename T, int RB>
static int launch_roww_m(int mode, int D, const RowArgs& a, hipStream_t st) {
    if (mode == RW_FWD) return D == 128 ? launch_roww_t<T, 128, RW_FWD, RB>(a, st) : launch_roww_t<T, 256, RW_FWD, RB>(a, st);
    return D == 128 ? launch_roww_t<T, 128, RW_DQ, RB>(a, st) : launch_roww_t<T, 256, RW_DQ, RB>(a, st);
}

int launch_roww_kernel(int mode, int dtype, int D, const RowArgs& a, hipStream_t st) {
    // 32 rows and four waves per workgroup as long as there is a CU for each: a round's LDS traffic, which bounds it, is half of that of 64 rows but for the
    // tiles' copies.  64 / 32 rows, forward and dQ pass, us, D = 128   1 x 64: 5.1, 6.1 / 5.2, 5.7   1 x 256: 7.1, 8.1 / 6.8, 7.6   1 x 640: 10.9, 12 / 9.9, 10.6
    // 2 x 2048: 11.1, 12.8 / 10.5, 11.8   D = 256   1 x 64: 6.0, 7.8 / 5.9, 7.1   1 x 640: 13.9, 15.6 / 12.6, 13.7   8 x 1000: 22.2, 23.3 / 20.4, 21.4
    // (two workgroups of 32 rows one after the other on a CU: 15 x 1001 x 128 18.0, 19.2 / 21.7, 22.2; 8 x 1777 x 256 18.4, 21.4 / 23.9, 27.0)
    if ((long long)a.BH * a.NG <= 128) return dtype == MLSTM_F16 ? launch_roww_m<_Float16, 1>(mode, D, a, st) : launch_roww_m<__bf16, 1>(mode, D, a, st);
    return dtype == MLSTM_F16 ? launch_roww_m<_Float16, 2>(mode, D, a, st) : launch_roww_m<__bf16, 2>(mode, D, a, st);
}

}  // namespace mlstm
