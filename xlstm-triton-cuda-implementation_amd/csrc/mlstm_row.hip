// Row-parallel tile kernel of the matmul form: one workgroup owns 128 query rows (4 waves x 32 rows) and walks
// the causal key tiles.  Two instantiations share the body:
//
//   MODE_FWD  X=Q, Y1=K, Y2=V:  S^T = K Q^T, P = S * exp2(alpha_j - beta_i + dG) / sqrt(D), b += rowsum P,
//             H^T += V^T P^T, epilogue h = H / (max(|b|, exp(-m)) + 1e-6).
//             Replaces mlstm_matmul_kernel (mlstm_matmul.py:38-101) and the CUDA kernel mlstm_forward
//             (cuda-src/mlstm_forward.cu:14-189).
//   MODE_DQ   X=dH, Y1=V, Y2=K: dC^T = V dH^T, G = (dC / n_i + db_i) * exp2(...) / sqrt(D), dQ^T += K^T G^T.
//             Replaces the dQ loop of mlstm_matmul_kernel_backward (mlstm_matmul.py:239-267).
//
// The products are computed transposed (keys along accumulator rows, queries along lanes) so that the
// accumulator of the first product is already laid out as the B operand of the second one: no lane exchange
// and every per-query scalar (beta, 1/n, db, the running row sum) lives in one register of one lane.
// There is no online max: the row maximum comes from the gate pre-pass as a prefix maximum.
//
// Memory pipeline: the two 64-key tiles of step j+1 are copied global->LDS by direct loads (no registers) into
// the other of two LDS stages while step j is consumed; one barrier per step.  Tiles are XOR-swizzled.
//
// Long sequences in chunks (RowArgs::chunk_len): a row tile walks the key tiles of its own chunk only; what lies before
// the chunk enters through the state at the end of the previous chunk (mlstm_chunk.hip), D/64 tiles of 64 state rows
// that pass through the same LDS stages ahead of the key tiles and are contracted with the rows' own X fragments:
//   forward  H^T += C~^T-tiles x Q^T, then the rows' decay exp(A_e - A_i), and b += decay (q_i . n~);
//   dQ pass  dQ^T += C~-tiles (value-major) x dH^T, then decay / n_i, the rank-one term decay db_i n~, and the row sums
//            q_i . dQ_i of dD over the keys before the chunk.
// In split mode the state comes as two terms, hi + lo (one tile each per stage), and takes two MFMAs per fragment.
//
// Workgroups per CU, by the registers that a lane may have (heads x positions, us per launch).
// 16-bit tensors at D = 128: two (256 registers, 66 KB of LDS), so that one of them multiplies while the other waits for its first tiles or writes out.
// Forward, one / two: 16 x 4096 31.5 / 23.9, 64 x 4096 102 / 70.9, 64 x 16384 406 / 270; the dQ pass keeps to 256 by itself: 29.0, 94.2 and 365.  One eight-wave
// workgroup per CU (mlstm_row8.hip) takes 415 and 489 at 64 x 16384.
// Split mode at D = 128: two; forward and dQ pass, one / two: 12 x 4096 38.4, 43.3 / 30.5, 35.1   16 x 4096 44.0, 49.5 / 34.4, 38.9
// 64 x 4096 146, 173 / 112, 135.
// Split mode at D = 64: two; forward, one / two / three: 18 x 1000 22.0 / 20.2 / 25.3   18 x 3008 21.1 / 16.1 / 16.7   59 x 3008 51.5 / 35.6 / 36.3   64 x 8192
// 143 / 89.0 / 84.9; dQ pass 24.5 / 20.8 / 21.5   18.6 / 18.5 / 18.7   41.2 / 40.4 / 38.6   123 / 120 / 118.
// D = 64: three in the dQ pass (168 registers) and in the forward in chunks, which gain where there are workgroups for them: dQ pass, two / three: 18 x 1000
// 17.1 / 17.2   64 x 1000 20.6 / 21.4   18 x 3008 15.1 / 14.6   59 x 3008 33.3 / 31.7   64 x 8192 93.1 / 86.2; forward in chunks 18 x 3008 11.4 / 12.1
// 59 x 3008 26.1 / 26.4   64 x 8192 67.9 / 61.8.  The forward of a sequence that is not cut stays at two: 18 x 1000 16.9 / 20.2, 64 x 1000 20.0 / 22.5.
// fp32 at D = 64: two; forward and dQ pass, one / two: 16 x 1000 15.5, 17.0 / 15.3, 16.3   64 x 300 23.5, 24.1 / 23.6, 23.6   16 x 4096 32.7, 37.2 / 26.2, 29.5
// 48 x 4096 91.8, 107 / 64.1, 73.7.  At D = 128 the 131 KB of LDS leave room for one.
#include <mutex>
#include <type_traits>
#include "mlstm_device.h"
#include "mlstm_kernels.h"
#include "mlstm_row_exact.h"

namespace mlstm {

constexpr int MODE_FWD = ROW_MODE_FWD, MODE_DQ = ROW_MODE_DQ;
constexpr int ROW_BQ = 128;

template <typename T, int D>
struct RowCfg {
    static constexpr size_t TILE_ELEMS = (size_t)GRAN * D;
    static constexpr size_t STAGE_BYTES = 2 * TILE_ELEMS * sizeof(T) + 3 * GRAN * sizeof(float);  // Y1, Y2, alpha, ek, amax
    static constexpr size_t STAGES_BYTES = 2 * STAGE_BYTES;
    // plus one double per key tile of the head (the granule bases), appended at launch
    // workgroups per CU that the register budget is cut for (the head of this file has the figures)
    static constexpr int per_cu(int mode, bool strict, bool chunks) {
        if (!Tr<T>::HALF) return D == 64 ? 2 : 1;
        if (D > 128) return 1;
        if (D == 64 && !strict) return mode == ROW_MODE_DQ || chunks ? 3 : 1;   // (1: 252 registers, two have room)
        return 2;
    }
};

// STRICT (16-bit types): split mode, see RowArgs::precise.
// PER_CU: workgroups per CU that the register budget is cut for.
template <typename T, int D, int MODE, bool STRICT, int PER_CU>
__global__ __launch_bounds__(256, PER_CU) void row_kernel(RowArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only builtins; the host pass only needs the stub
    using R = Tr<T>;
    using Cfg = RowCfg<T, D>;
    typedef typename R::frag frag;
    constexpr int KW = R::KW, NS = D / KW, NDB = D / 32, NSTEP32 = 32 / KW;
    constexpr bool F32 = !R::HALF;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5, c32 = lane & 31;
    int S = a.S, NG = a.NG;
    const int nQT = (S + ROW_BQ - 1) / ROW_BQ;
    int bh, qt;
    {
        // heaviest query tiles first over ALL heads (a per-head-group order leaves heavy tiles of the last group for the end); all tiles of a head run on one XCD
        // (workgroups are dealt round-robin to the 8 XCDs) so that its K/V stay in that XCD's L2
        const int bid = blockIdx.x;
        if ((a.BH & 7) == 0) {
            int rest = bid >> 3;
            const int ngrp = a.BH >> 3;
            bh = (rest % ngrp) * 8 + (bid & 7);
            qt = nQT - 1 - rest / ngrp;
        } else {
            bh = bid % a.BH;
            qt = nQT - 1 - bid / a.BH;
        }
    }
    size_t hoff = (size_t)bh * S, poff = (size_t)bh * NG * GRAN, goff = (size_t)bh * NG;
    // the caller's tensors: q, k, v, dq in layout la, h, dh, o in lb (element offset of the head, elements per position)
    const size_t rsA = (size_t)a.la.ss, rsB = (size_t)a.lb.ss, rsH = (size_t)a.lh.ss;
    size_t offA = a.la.head(bh), offB = a.lb.head(bh), offH = a.lh.head(bh);
    // In chunks the workgroup's rows lie in chunk `chunk`, and everything below addresses positions relative to the chunk's
    // first one: the sequence "starts" there (offsets move forward; S, NG and the row tile index shrink).
    int chunk = 0;
    if (a.chunk_len > 0) {
        chunk = (qt * ROW_BQ) / a.chunk_len;
        const int p0 = chunk * a.chunk_len;
        hoff += p0; poff += p0; goff += p0 / GRAN;
        offA += (size_t)p0 * rsA; offB += (size_t)p0 * rsB; offH += (size_t)p0 * rsH;
        S -= p0; NG -= p0 / GRAN; qt -= p0 / ROW_BQ;
    }
    const int q0 = qt * ROW_BQ, r0 = q0 + 32 * wave;
    const int row = r0 + c32, rowc = row < S ? row : S - 1;
    const bool wave_active = r0 < S;
    const size_t rsX = MODE == MODE_FWD ? rsA : rsB, offX = MODE == MODE_FWD ? offA : offB;
    const size_t rsO = MODE == MODE_FWD ? rsB : rsA, offO = MODE == MODE_FWD ? offB : offA;
    const T* X = reinterpret_cast<const T*>(a.X) + offX;
    const T* Y1 = reinterpret_cast<const T*>(a.Y1) + offA;
    const T* Y2 = reinterpret_cast<const T*>(a.Y2) + offA;

    // ---- one trip to memory for all that is needed before the first key tile: the rows of X, as two 64-row tiles in whole lines, and with them
    // the state of the previous chunk or, in the first one, key tile 0 (a row per lane straight into registers asks for 32 bytes of 32 lines per
    // instruction, and the state and the first keys came one trip after the other: 64 heads x 16384 x 128,
    // forward 334 -> 297 us, dQ pass 422 -> 400).  Where all state tiles fit one
    // stage, in up to 32 KB (64 KB are no longer one trip: fp32 at D = 128 143 -> 147 us), they lie in stage 1 and X in stage 0; otherwise the first
    // one lies in stage NTL % 2, as below, and X in the other.
    constexpr int NTL = D / GRAN;
    constexpr bool AT_ONCE = !STRICT && NTL <= 2 && NTL * Cfg::TILE_ELEMS * sizeof(T) <= 32 * 1024;
    const bool far = chunk > 0;
#define ST_Y1(st) (reinterpret_cast<T*>(smem + (st) * Cfg::STAGE_BYTES))
#define ST_Y2(st) (ST_Y1(st) + Cfg::TILE_ELEMS)
#define ST_AL(st) (reinterpret_cast<float*>(ST_Y2(st) + Cfg::TILE_ELEMS))
    double* const sG = reinterpret_cast<double*>(smem + Cfg::STAGES_BYTES);   // granule bases of this head
    const int met = a.chunk_len > 0 && a.chunk_len / GRAN < NG ? a.chunk_len / GRAN : NG;   // granules a row may meet
    float* const nvl = reinterpret_cast<float*>(sG + ((met + 1) & ~1));       // in chunks: the vector state of the previous one, [D]
    // (plain loads first: what they bring is used behind the copies' issue)
    const float beta_row = a.beta2[poff + rowc], m_row = a.M[hoff + rowc];
    const float b_row = MODE == MODE_DQ ? a.Bin[hoff + rowc] : 0.f;
    const float beta_end = far ? a.beta2[poff - 1] : 0.f;
    const double g_row = far ? a.G2[goff + rowc / GRAN] : 0.0, g_end = far ? a.G2[goff - 1] : 0.0;
    frag hfr[NS], hlr[STRICT ? NS : 1];
    bool h_low = false;
    if constexpr (MODE == MODE_DQ) {
        const T* hrow = reinterpret_cast<const T*>(a.Hin) + offH + (size_t)rowc * rsH;
#pragma unroll
        for (int s = 0; s < NS; s++) hfr[s] = frag_rowmajor<T>(hrow, s, h);
        if constexpr (STRICT) {
            h_low = a.Hin_lo != nullptr;
            if (h_low) {
                const T* hlo = reinterpret_cast<const T*>(a.Hin_lo) + (hoff + rowc) * D;
#pragma unroll
                for (int s = 0; s < NS; s++) hlr[s] = frag_rowmajor<T>(hlo, s, h);
            }
        }
    }
    TileDma<T, D, GRAN, 256> tdma;
    tdma.init(tid);
    const auto ra = tdma.rows(tid, (unsigned)(rsA * sizeof(T)));
    RowVec3Dma rvdma;   // alpha, ek (64 per tile) and the two block maxima of a tile (padded arrays: always readable)
    rvdma.init(tid, a.alpha2 + poff, a.ek2 + poff, a.amax2 + goff * 2, 64, 64, 2);
    const int full_tiles = S / GRAN;  // key tiles whose 64 rows all exist
#define ROW_DMA(j, st)                                                                   \
    do {                                                                                 \
        if ((j) < full_tiles) {                                                          \
            tdma.issue(ST_Y1(st), Y1 + (size_t)GRAN * (j) * rsA, ra);                     \
            tdma.issue(ST_Y2(st), Y2 + (size_t)GRAN * (j) * rsA, ra);                     \
        } else {                                                                         \
            int t = tid;   /* (formed anew: addresses kept for a tile that rarely comes were spilled) */ \
            if constexpr (R::HALF && D == 128) asm volatile("" : "+v"(t));                 \
            tile_dma<T, D, GRAN, 256>(ST_Y1(st), Y1, GRAN * (j), S, t, rsA);              \
            tile_dma<T, D, GRAN, 256>(ST_Y2(st), Y2, GRAN * (j), S, t, rsA);              \
        }                                                                                \
        rvdma.issue(ST_AL(st), (j));                                                     \
    } while (0)
    const size_t sbase = far ? ((size_t)bh * a.n_states + chunk - 1) * D * D : 0;
    const T* const Cs = reinterpret_cast<const T*>(a.Cst) + sbase;
    const T* const Cl = STRICT ? reinterpret_cast<const T*>(a.Cst_lo) + sbase : nullptr;
    auto issue_state = [&](int tau) {
        if constexpr (AT_ONCE) {
            tdma.issue(tau == 0 ? ST_Y1(1) : ST_Y2(1), Cs + (size_t)GRAN * tau * D);
        } else {
            const int stg = (tau + (NTL & 1)) & 1;
            tdma.issue(ST_Y1(stg), Cs + (size_t)GRAN * tau * D);
            if constexpr (STRICT) tdma.issue(ST_Y2(stg), Cl + (size_t)GRAN * tau * D);
        }
    };
    T* const xtile = ST_Y1(far && (AT_ONCE || (NTL & 1)) ? 0 : 1);
    {
        const auto rx = tdma.rows(tid, (unsigned)(rsX * sizeof(T)));
#pragma unroll
        for (int t = 0; t < 2; t++) {
            if (q0 + GRAN * (t + 1) <= S) tdma.issue(xtile + t * Cfg::TILE_ELEMS, X + (size_t)(q0 + GRAN * t) * rsX, rx);
            else tile_dma_rolled<T, D, GRAN, 256>(xtile + t * Cfg::TILE_ELEMS, X, q0 + GRAN * t, S, tid, rsX);
        }
    }
    if (far) {
        issue_state(0);
        if constexpr (AT_ONCE && NTL == 2) issue_state(1);
        if (tdma.wave_s < D / 64)
            dma4(a.Nst + ((size_t)bh * a.n_states + chunk - 1) * D + 64 * tdma.wave_s + lane, __builtin_amdgcn_readfirstlane(lds_offset_of(nvl + 64 * tdma.wave_s)));
    } else {
        ROW_DMA(0, 0);
    }
    // granule bases of this head in LDS: a global load inside the main loop would have to be waited for with
    // vmcnt(0), which would also wait for the tile copies in flight
    for (int g = tid; g < met; g += 256) sG[g] = a.G2[goff + g];
    // What a weight's exponent has beside alpha of the key.  fp32: its parts stay apart until they are added at the size of the
    // result (alpha less beta of the row; the granules' distance and log2 of 1 / sqrt(D) in fp64): added up per row first they were
    // rounded at the size of the parts, 3 % of the error of h and 6 % of that of dV.
    typedef typename std::conditional<F32, double, float>::type Crow;
    constexpr double LOG2_SCALE = D == 64 ? -3.0 : (D == 128 ? -3.5 : -4.0);
    const float nbeta = -beta_row;
    float crow_base = -0.5f * __log2f((float)D) - beta_row;
    // the rows' decay since the end of the previous chunk
    float dec = far ? fast_exp2(beta_end - beta_row + (float)(g_row - g_end)) : 0.f;
    SwzRowReader<T, D> krd;
    krd.init(lane);
    dma_wait();
    __syncthreads();   // X, what came with it and sG are there
    frag xf[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) xf[s] = krd.read(xtile + (wave >> 1) * Cfg::TILE_ELEMS, wave & 1, s);
    float inv_n = 0.f, dbv = 0.f;
    if constexpr (MODE == MODE_DQ) {
        row_stats_of_frags<T, NS>(xf, hfr, hlr, h_low, b_row, m_row, inv_n, dbv);
        // (the rows behind the sequence, up to the end of its last granule, as zeros: whoever reads whole granules multiplies
        // them by a weight of zero, and what scratch memory holds need not be a number)
        if (row < NG * GRAN && h == 0) { a.inv_n[poff + row] = row < S ? inv_n : 0.f; a.db[poff + row] = row < S ? dbv : 0.f; }
    }
#pragma unroll
    for (int s = 0; s < NS; s++) pin(xf[s]);
    pin(crow_base); pin(inv_n); pin(dbv); pin(dec);
    if (far) __syncthreads();   // X's stage is free
    typename R::terms xt[NS];   // the rows' operand of every first product
#pragma unroll
    for (int s = 0; s < NS; s++) xt[s] = R::split(xf[s]);

    f32x16 oacc[NDB];
#pragma unroll
    for (int d = 0; d < NDB; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[d][r] = 0.f;
    float bsum = 0.f;

    constexpr bool FAST_TR = R::HALF && Swz<T, D>::CPR >= 16;  // precomputed offsets for the transposing reads
    // The 16-bit types at D >= 128 outside split mode share their order of operations with mlstm_row8.hip and mlstm_roww.hip, which spread a
    // row over waves: the row sums over the key blocks of either parity and over either half of the state's rows apart, and the
    // factorised weights wherever a block lies below the diagonal.
    constexpr bool PARITY = FAST_TR && !STRICT;
    float bpar[2] = {0.f, 0.f}, bfar[2] = {0.f, 0.f}, dec_far = 0.f;
    typename std::conditional<F32, SwzTransReaderF32<D>, SwzTransReader<typename std::conditional<FAST_TR, T, __bf16>::type, FAST_TR ? D : 256>>::type vrd;
    if constexpr (FAST_TR || F32) vrd.init(lane);

    const int last_row = (q0 + ROW_BQ - 1 < S - 1) ? q0 + ROW_BQ - 1 : S - 1;
    const int nJ = last_row / GRAN + 1;

    // first product of both 32-key blocks of a tile, S^T (or dC^T) in accumulator layout; the two accumulation
    // chains are interleaved so that consecutive MFMAs never depend on each other
    auto gemm1x2 = [&](const T* y1, f32x16& s0, f32x16& s1, auto&& hook) {
        if constexpr (F32) {
            f32x16 t0 = {}, t1 = {};
            s0 = f32x16{}; s1 = f32x16{};
            R::template stream<2 * NS>([&](auto n) { return krd.read(y1, n & 1, n >> 1); }, [&](auto n, const auto& kf, auto&& between) {
                if (n % 4 == 0) hook(n / 4, NS / 2);
                R::mma_between(n & 1 ? s1 : s0, n & 1 ? t1 : t0, kf, xt[n >> 1], between);
            });
            s0 += t0; s1 += t1;
            return;
        }
        constexpr int BATCH = NS < 4 ? NS : 4;  // fragments fetched ahead of the MFMAs that consume them
#pragma unroll
        for (int b0 = 0; b0 < NS; b0 += BATCH) {
            hook(b0 / BATCH, NS / BATCH);
            frag k0[BATCH], k1[BATCH];
#pragma unroll
            for (int s = 0; s < BATCH; s++) { k0[s] = krd.read(y1, 0, b0 + s); k1[s] = krd.read(y1, 1, b0 + s); }
#pragma unroll
            for (int s = 0; s < BATCH; s++) {
                if (b0 + s == 0) {
                    const f32x16 z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                    s0 = z; s1 = z;
                }
                R::mma(s0, k0[s], xt[b0 + s]);
                R::mma(s1, k1[s], xt[b0 + s]);
            }
        }
    };
    auto gemm1 = [&](const T* y1, int kb, f32x16& sacc) {
#pragma unroll
        for (int r = 0; r < 16; r++) sacc[r] = 0.f;
        if constexpr (F32) {
            f32x16 small = {};
            R::template stream<NS>([&](auto n) { return krd.read(y1, kb, n); },
                                   [&](auto n, const auto& kf, auto&& between) { R::mma_between(sacc, small, kf, xt[n], between); });
            sacc += small;
        } else {
#pragma unroll
            for (int s = 0; s < NS; s++) R::mma(sacc, krd.read(y1, kb, s), xt[s]);
        }
    };
    // Split mode: the weights of a block as they enter the second product, formed four at a time where they are weighed.  They come as factors,
    // x y, of which the low-order term takes what rounding the product would lose; factors kept until the product is due cost 16 registers.
    struct Terms { typename R::vec4 hi[4], lo[4]; };
    auto terms_of = [](const typename R::vec4* x, int t) { return __builtin_shufflevector(x[2 * t], x[2 * t + 1], 0, 1, 2, 3, 4, 5, 6, 7); };
    // gate weights; `diag` masks the keys above the diagonal of a diagonal block
    auto weigh = [&](f32x16& sacc, Terms& w, const float* sal, int kb, Crow crow, bool diag) {
#pragma unroll
        for (int a4 = 0; a4 < 4; a4++) {
            const f32x4 al = *reinterpret_cast<const f32x4*>(sal + 32 * kb + 8 * a4 + 4 * h);
            f32x4 wx, wy;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int r = 4 * a4 + c;
                float e;
                if constexpr (F32) e = fast_exp2((al[c] + nbeta) + (float)crow);
                else e = fast_exp2(al[c] + crow);
                if (diag && (8 * a4 + 4 * h + c > c32)) e = 0.f;
                if constexpr (MODE == MODE_FWD) {
                    float& b = PARITY ? bpar[kb] : bsum;
                    b = fmaf(sacc[r], e, b);
                    wx[c] = sacc[r];
                } else {
                    wx[c] = fmaf(sacc[r], inv_n, dbv);
                }
                wy[c] = e;
                sacc[r] = wx[c] * e;
            }
            if constexpr (STRICT) {
                R::split_products(wx, wy, w.hi[a4], w.lo[a4]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // gate weights of a block entirely below the diagonal, factorised: exp2(alpha_j - c0) comes from the pre-pass
    // (sek), exp2(c0 - beta_i + dG) is one exponential per lane and block
    auto weigh_fact = [&](f32x16& sacc, Terms& w, const float* sek, int kb, Crow crow) {
        float er;
        if constexpr (F32) er = fast_exp2((float)((double)(sek[GRAN + kb] + nbeta) + crow));
        else er = fast_exp2(crow + sek[GRAN + kb]);
        float blk = 0.f;
#pragma unroll
        for (int a4 = 0; a4 < 4; a4++) {
            const f32x4 ek = *reinterpret_cast<const f32x4*>(sek + 32 * kb + 8 * a4 + 4 * h);
            f32x4 wx, wy;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int r = 4 * a4 + c;
                if constexpr (MODE == MODE_FWD) {
                    blk = fmaf(sacc[r], ek[c], blk);
                    wx[c] = sacc[r] * ek[c];
                    wy[c] = er;
                    sacc[r] = wx[c] * er;
                } else if constexpr (PARITY) {
                    sacc[r] = fmaf(sacc[r], inv_n * er, dbv * er) * ek[c];
                } else {
                    wx[c] = fmaf(sacc[r], inv_n, dbv);
                    wy[c] = ek[c] * er;
                    sacc[r] = wx[c] * wy[c];
                }
            }
            if constexpr (STRICT) R::split_products(wx, wy, w.hi[a4], w.lo[a4]);
        }
        if constexpr (MODE == MODE_FWD) {
            float& b = PARITY ? bpar[kb] : bsum;
            b = fmaf(blk, er, b);
        }
    };
    // second product: accumulate this key block into the output
    auto gemm2 = [&](const T* y2, const f32x16& sacc, const Terms& w, int kb, auto&& hook) {
        if constexpr (F32) {
            const typename R::terms p[2] = {R::split(R::from_acc(sacc, 0)), R::split(R::from_acc(sacc, 1))};
            R::template stream<2 * NDB>([&](auto n) { return vrd.read(y2, 32 * kb + KW * (n / NDB), n % NDB); },
                                        [&](auto n, const auto& vf, auto&& between) {
                                            if (n % NDB == 0) hook(2 * kb + n / NDB, 4);
                                            R::mma_between(oacc[n % NDB], vf, p[n / NDB], between);
                                        });
            return;
        }
#pragma unroll
        for (int t = 0; t < NSTEP32; t++) {
            hook(kb * NSTEP32 + t, 2 * NSTEP32);
            frag pf, pl;
            if constexpr (STRICT) { pf = terms_of(w.hi, t); pl = terms_of(w.lo, t); }
            else pf = R::from_acc(sacc, t);
            frag vf[NDB];
#pragma unroll
            for (int d = 0; d < NDB; d++) {
                if constexpr (FAST_TR || F32) vf[d] = vrd.read(y2, 32 * kb + KW * t, d);
                else vf[d] = swz_frag_transposed<T, D>(y2, 32 * kb + KW * t, 32 * d, lane);
            }
#pragma unroll
            for (int d = 0; d < NDB; d++) {
                R::mma(oacc[d], vf[d], pf);
                if constexpr (STRICT) R::mma(oacc[d], vf[d], pl);
            }
        }
    };

    // A whole mask-free tile with the vector work hidden behind the matrix work.  A wave issues in order and an MFMA
    // executes asynchronously, so vector instructions placed between two MFMAs cost nothing while the matrix unit
    // is busy; the tile is therefore walked as
    //     S0 = K0 Q^T | S1 = K1 Q^T with the weighing of S0 between its MFMAs | H += V0^T P0^T with the weighing of S1
    //     between its MFMAs | H += V1^T P1^T
    // and every LDS operand is read a few MFMAs ahead of its use.
    auto tile_overlapped = [&](const T* y1, const T* y2, const float* sek, float crow, auto&& hook1, auto&& hook2) {
      if constexpr (FAST_TR && NSTEP32 == 2) {
        constexpr int AH = NS < 4 ? NS : 4;
        f32x16 s0, s1;
        // one accumulator register of a block below the diagonal: see weigh_fact
        auto weigh_reg = [&](f32x16& sacc, Terms& w, int r, const f32x4 (&ek)[4], float er, float& blk) {
            if constexpr (MODE == MODE_FWD) {
                blk = fmaf(sacc[r], ek[r >> 2][r & 3], blk);
                sacc[r] *= ek[r >> 2][r & 3];
                if constexpr (!STRICT) sacc[r] *= er;
            } else if constexpr (PARITY) {
                sacc[r] = fmaf(sacc[r], inv_n * er, dbv * er) * ek[r >> 2][r & 3];
            } else {
                sacc[r] = fmaf(sacc[r], inv_n, dbv);
                if constexpr (!STRICT) sacc[r] *= ek[r >> 2][r & 3] * er;
            }
            if constexpr (STRICT && MODE == MODE_DQ) {
                if ((r & 3) == 3) R::split_products(f32x4{sacc[r - 3], sacc[r - 2], sacc[r - 1], sacc[r]}, ek[r >> 2] * er, w.hi[r >> 2], w.lo[r >> 2]);
            }
        };
        Terms w0, w1;
        f32x4 ek0[4], ek1[4];
#pragma unroll
        for (int a4 = 0; a4 < 4; a4++) {
            ek0[a4] = *reinterpret_cast<const f32x4*>(sek + 8 * a4 + 4 * h);
            ek1[a4] = *reinterpret_cast<const f32x4*>(sek + 32 + 8 * a4 + 4 * h);
        }
        const float er0 = fast_exp2(crow + sek[GRAN]), er1 = fast_exp2(crow + sek[GRAN + 1]);
        float blk0 = 0.f, blk1 = 0.f;
        frag kq[NS];
        // ---- S0
#pragma unroll
        for (int s = 0; s < AH; s++) kq[s] = krd.read(y1, 0, s);
#pragma unroll
        for (int s = 0; s < NS; s++) {
            if (s % 4 == 0) hook1(s / 4, 2 * (NS / 4));
            if (s + AH < NS) kq[s + AH] = krd.read(y1, 0, s + AH);
            if (s == 0) {
                const f32x16 z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                s0 = z; s1 = z;
            }
            R::mma(s0, kq[s], xt[s]);
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- S1, weighing S0 (16 registers over NS MFMAs)
        frag kr[NS];
#pragma unroll
        for (int s = 0; s < AH; s++) kr[s] = krd.read(y1, 1, s);
#pragma unroll
        for (int s = 0; s < NS; s++) {
            if (s % 4 == 0) hook1(NS / 4 + s / 4, 2 * (NS / 4));
            if (s + AH < NS) kr[s + AH] = krd.read(y1, 1, s + AH);
            R::mma(s1, kr[s], xt[s]);
#pragma unroll
            for (int r = s * 16 / NS; r < (s + 1) * 16 / NS; r++) weigh_reg(s0, w0, r, ek0, er0, blk0);
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- H += V^T P^T: groups g = 2*kb + t of 16 keys; the weighing of S1 rides on the groups of key block 0
        frag vf[2][NDB];
#pragma unroll
        for (int d = 0; d < NDB; d++) vf[0][d] = vrd.read(y2, 0, d);
        frag pf, pl;
        auto take_p = [&](const f32x16& sacc, Terms& w, float er, int t) {
            if constexpr (STRICT) {
                if constexpr (MODE == MODE_FWD) {
#pragma unroll
                    for (int a4 = 2 * t; a4 < 2 * t + 2; a4++)
                        R::split_products(f32x4{sacc[4 * a4], sacc[4 * a4 + 1], sacc[4 * a4 + 2], sacc[4 * a4 + 3]}, f32x4{er, er, er, er}, w.hi[a4], w.lo[a4]);
                }
                pf = terms_of(w.hi, t);
                pl = terms_of(w.lo, t);
            } else {
                pf = R::from_acc(sacc, t);
            }
        };
        take_p(s0, w0, er0, 0);
#pragma unroll
        for (int g = 0; g < 4; g++) {
            hook2(g, 4);
#pragma unroll
            for (int d = 0; d < NDB; d++) {
                if (g + 1 < 4) vf[(g + 1) & 1][d] = vrd.read(y2, KW * (g + 1), d);
                R::mma(oacc[d], vf[g & 1][d], pf);
                if constexpr (STRICT) R::mma(oacc[d], vf[g & 1][d], pl);
                if (g < 2) {
#pragma unroll
                    for (int r = (g * NDB + d) * 16 / (2 * NDB); r < (g * NDB + d + 1) * 16 / (2 * NDB); r++) weigh_reg(s1, w1, r, ek1, er1, blk1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (g == 0) take_p(s0, w0, er0, 1);
            if (g == 1) take_p(s1, w1, er1, 0);
            if (g == 2) take_p(s1, w1, er1, 1);
        }
        if constexpr (MODE == MODE_FWD && PARITY) { bpar[0] = fmaf(blk0, er0, bpar[0]); bpar[1] = fmaf(blk1, er1, bpar[1]); }
        else if constexpr (MODE == MODE_FWD) bsum += fmaf(blk0, er0, blk1 * er1);
      }
    };

    const double GI = sG[(wave_active ? r0 : S - 1) / GRAN];
    if (far) {
        // ---- what lies before the chunk: the state at the end of the previous chunk, as D/64 tiles of 64 rows in the order
        // in which this product contracts them (mlstm_chunk.hip), in split mode each as a hi and a lo tile.  One tile at a time (not
        // AT_ONCE) they go through the stages in turns, hi tile in the Y1 slot and lo tile in the Y2 slot, the last one in stage 1, so that
        // key tile 0 can follow into stage 0 under it.
        constexpr int NGRP = GRAN / KW;
        // dQ pass: the rows of Q for q_i . dQ_i below, requested ahead of the state's products.  A lane holds four columns of every eight, 8 bytes of
        // a 16-byte piece; 16-bit rows are loaded in whole pieces, half of them by either lane of a row, which exchange the halves
        // (64 heads x 16384 x 128 400 -> 394 us).
        constexpr bool QPIECES = MODE == MODE_DQ && R::HALF && D <= 128;
        constexpr int QP = QPIECES ? D / 16 : 1;
        uint4 qpiece[QP];
        if constexpr (QPIECES) {
            const T* qrow = reinterpret_cast<const T*>(a.Qrow) + offA + (size_t)rowc * rsA;
#pragma unroll
            for (int p = 0; p < QP; p++) qpiece[p] = *reinterpret_cast<const uint4*>(qrow + 8 * (QP * h + p));
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (AT_ONCE) ROW_DMA(0, 0);
#pragma unroll
        for (int tau = 0; tau < NTL; tau++) {
            const int stg = AT_ONCE ? 1 : (tau + (NTL & 1)) & 1;
            if constexpr (!AT_ONCE) {
                if (tau > 0) {
                    dma_wait();
                    __syncthreads();   // tile tau has landed; the other stage is free
                }
                if (tau + 1 < NTL) issue_state(tau + 1);
                else ROW_DMA(0, 0);
            }
            const T* th = AT_ONCE && tau == 1 ? ST_Y2(stg) : ST_Y1(stg);
            const T* tl = ST_Y2(stg);
            if constexpr (F32) {
                R::template stream<NGRP * NDB>([&](auto n) { return vrd.read(th, KW * (n / NDB), n % NDB); },
                                               [&](auto n, const auto& cf, auto&& between) {
                                                   R::mma_between(oacc[n % NDB], cf, xt[NGRP * tau + n / NDB], between);
                                               });
                continue;
            }
            auto rd = [&](const T* tile, int g, int d) {
                if constexpr (FAST_TR || F32) return vrd.read(tile, KW * g, d);
                else return swz_frag_transposed<T, D>(tile, KW * g, 32 * d, lane);
            };
            frag vf[2][NDB];
#pragma unroll
            for (int d = 0; d < NDB; d++) vf[0][d] = rd(th, 0, d);
#pragma unroll
            for (int g = 0; g < NGRP; g++) {
                frag vl[STRICT ? NDB : 1];
#pragma unroll
                for (int d = 0; d < NDB; d++) {
                    if constexpr (STRICT) vl[d] = rd(tl, g, d);
                    if (g + 1 < NGRP) vf[(g + 1) & 1][d] = rd(th, g + 1, d);
                    R::mma(oacc[d], vf[g & 1][d], xt[NGRP * tau + g]);
                }
                if constexpr (STRICT) {
#pragma unroll
                    for (int d = 0; d < NDB; d++) R::mma(oacc[d], vl[d], xt[NGRP * tau + g]);
                }
            }
        }
        const float* const nst = nvl;
        if constexpr (MODE == MODE_FWD) {
            // row sums: decay_i (q_i . n~); the lane's half of the row (the halves meet in the epilogue)
            if constexpr (PARITY) {
                dec_far = dec;
#pragma unroll
                for (int s2 = 0; s2 < NS; s2++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float& part = bfar[s2 / (NS / 2)];
                        const float* const n8 = nst + KW * s2 + R::EPL * h;
                        part += fmaf(to_f32(xf[s2][e]), n8[e], to_f32(xf[s2][4 + e]) * n8[4 + e]);
                    }
            } else {
                float part = 0.f;
#pragma unroll
                for (int s2 = 0; s2 < NS; s2++)
#pragma unroll
                    for (int e = 0; e < R::EPL; e++) part = fmaf(to_f32(xf[s2][e]), nst[KW * s2 + R::EPL * h + e], part);
                bsum = fmaf(dec, part, bsum);
            }
#pragma unroll
            for (int d = 0; d < NDB; d++)
#pragma unroll
                for (int r = 0; r < 16; r++) oacc[d][r] *= dec;
        } else {
            const float decn = dec * inv_n, rank1 = dec * dbv;
            // (summed per block of 32 columns, as mlstm_rowf.hip, mlstm_roww.hip and mlstm_rowx.hip, which split a row by columns, have to;
            // 16 bits at D >= 128: and per half of them.  At D = 64 they are one sum.)
            float rp = 0.f, rp_first = 0.f, rpd = 0.f;
            auto block = [&](int d, auto&& n_of, auto&& q_of) {
                if (F32 || FAST_TR) rpd = 0.f;
#pragma unroll
                for (int a4 = 0; a4 < 4; a4++) {
                    const f32x4 n4 = n_of(a4), q4 = __builtin_convertvector(q_of(a4), f32x4);
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const float v = fmaf(rank1, n4[c], oacc[d][4 * a4 + c] * decn);
                        oacc[d][4 * a4 + c] = v;
                        rpd = fmaf(v, q4[c], rpd);
                    }
                }
                if (F32 || FAST_TR || d == NDB - 1) rp += rpd;
                if (FAST_TR && d == NDB / 2 - 1) { rp_first = rp; rp = 0.f; }
            };
            auto n_at = [&](int d, int a4) { return *reinterpret_cast<const f32x4*>(nst + 32 * d + 8 * a4 + 4 * h); };
            if constexpr (QPIECES) {
                // pieces p (lanes h = 0) and QP + p (h = 1) of the row: the low halves to h = 0, the high ones to h = 1
                uint2 qh[2 * QP];
#pragma unroll
                for (int p = 0; p < QP; p++) {
                    const auto x = __builtin_amdgcn_permlane32_swap((int)qpiece[p].x, (int)qpiece[p].z, false, false);
                    const auto y = __builtin_amdgcn_permlane32_swap((int)qpiece[p].y, (int)qpiece[p].w, false, false);
                    qh[p] = make_uint2(x[0], y[0]);
                    qh[QP + p] = make_uint2(x[1], y[1]);
                }
#pragma unroll
                for (int d = 0; d < NDB; d++) block(d, [&](int a4) { return n_at(d, a4); }, [&](int a4) { return __builtin_bit_cast(typename R::vec4, qh[4 * d + a4]); });
            } else {
                const T* qrow = reinterpret_cast<const T*>(a.Qrow) + offA + (size_t)rowc * rsA;
                typename R::vec4 qv[2][4];   // a column block's values, requested a block ahead (left to the compiler: loads one by one, each waited for)
                auto request = [&](int d) {
#pragma unroll
                    for (int a4 = 0; a4 < 4; a4++) qv[d & 1][a4] = *reinterpret_cast<const typename R::vec4*>(qrow + 32 * d + 8 * a4 + 4 * h);
                    __builtin_amdgcn_sched_barrier(0);
                };
                request(0);
#pragma unroll
                for (int d = 0; d < NDB; d++) {
                    if (d + 1 < NDB) request(d + 1);
                    block(d, [&](int a4) { return n_at(d, a4); }, [&](int a4) { return qv[d & 1][a4]; });
                }
            }
            // row sums of dD over the keys before the chunk: q_i . dQ_i of what the accumulators hold now
            rp = sum_halves(rp);
            if constexpr (FAST_TR) rp = sum_halves(rp_first) + rp;
            if (row < S && h == 0) a.rowinter[hoff + row] = rp;
        }
    } else {
        if constexpr (MODE == MODE_DQ) {
            if (a.chunk_len > 0 && row < S && h == 0) a.rowinter[hoff + row] = 0.f;
        }
    }
    // Tiles strictly below this wave's rows take the mask-free path; the last one or two tiles of the workgroup are
    // diagonal, or entirely above the diagonal, for this wave.  Two loops with one code path each keep the output
    // accumulators in place (a two-way branch inside one loop makes the register allocator copy them every step).
    // Every wave executes nJ barriers in total, whichever loop it is in.
    const int jfull = wave_active ? (r0 / GRAN < nJ ? r0 / GRAN : nJ) : 0;   // tiles with 64*j + 63 < r0
    auto no_hook = [](int, int) {};
    constexpr int PW = TileDma<T, D, GRAN, 256>::PER_WAVE;
    // Main loop in two parts, each a single code path.  Part 1: the next tile exists and is complete, and its copy
    // is interleaved with this tile's MFMAs (hooks).  Part 2 (at most a step or two): the next tile is the partial
    // last tile of the sequence, or there is none; the copy is issued in one go through the clamping path.
    const int lim = (nJ < full_tiles ? nJ : full_tiles) - 1;
    const int jspread = jfull < lim ? jfull : (lim > 0 ? lim : 0);
    int j = 0;
    for (; j < jspread; j++) {
        dma_wait();
        __syncthreads();  // tile j has landed for every wave and stage (j+1)&1 is free again
        const int jn = j + 1, stn = jn & 1;
        rvdma.issue(ST_AL(stn), jn);
        const T* gy1 = Y1 + (size_t)GRAN * jn * rsA;
        const T* gy2 = Y2 + (size_t)GRAN * jn * rsA;
        T* const ly1 = ST_Y1(stn);
        T* const ly2 = ST_Y2(stn);
        auto hook1 = [&](int idx, int n) { tdma.issue_range(ly1, gy1, idx * PW / n, (idx + 1) * PW / n, ra); };
        auto hook2 = [&](int idx, int n) { tdma.issue_range(ly2, gy2, idx * PW / n, (idx + 1) * PW / n, ra); };
        const T* y1 = ST_Y1(j & 1);
        const T* y2 = ST_Y2(j & 1);
        const float* sal = ST_AL(j & 1);
        Crow crow;
        if constexpr (F32) crow = LOG2_SCALE + (GI - sG[j]);
        else crow = crow_base + (float)(GI - sG[j]);
        if constexpr (FAST_TR && NSTEP32 == 2) {
            tile_overlapped(y1, y2, sal + GRAN, crow, hook1, hook2);
        } else {
            f32x16 s0, s1;
            gemm1x2(y1, s0, s1, hook1);
            Terms w;
            weigh_fact(s0, w, sal + GRAN, 0, crow);
            gemm2(y2, s0, w, 0, hook2);
            weigh_fact(s1, w, sal + GRAN, 1, crow);
            gemm2(y2, s1, w, 1, hook2);
        }
    }
    for (; j < jfull; j++) {
        dma_wait();
        __syncthreads();
        if (j + 1 < nJ) {
            if (j & 1) ROW_DMA(j + 1, 0); else ROW_DMA(j + 1, 1);
        }
        const T* y1 = ST_Y1(j & 1);
        const T* y2 = ST_Y2(j & 1);
        const float* sal = ST_AL(j & 1);
        Crow crow;
        if constexpr (F32) crow = LOG2_SCALE + (GI - sG[j]);
        else crow = crow_base + (float)(GI - sG[j]);
        if constexpr (FAST_TR && NSTEP32 == 2) {
            tile_overlapped(y1, y2, sal + GRAN, crow, no_hook, no_hook);
        } else {
            f32x16 s0, s1;
            gemm1x2(y1, s0, s1, no_hook);
            Terms w;
            weigh_fact(s0, w, sal + GRAN, 0, crow);
            gemm2(y2, s0, w, 0, no_hook);
            weigh_fact(s1, w, sal + GRAN, 1, crow);
            gemm2(y2, s1, w, 1, no_hook);
        }
    }
    for (; j < nJ; j++) {
        dma_wait();
        __syncthreads();
        if (j + 1 < nJ) {
            if (j & 1) ROW_DMA(j + 1, 0); else ROW_DMA(j + 1, 1);
        }
        if (!wave_active) continue;
        const T* y1 = ST_Y1(j & 1);
        const T* y2 = ST_Y2(j & 1);
        const float* sal = ST_AL(j & 1);
        Crow crow;
        if constexpr (F32) crow = LOG2_SCALE + (GI - sG[j]);
        else crow = crow_base + (float)(GI - sG[j]);
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
            const int kstart = GRAN * j + 32 * kb;
            if (kstart <= r0) {
                f32x16 s0;
                gemm1(y1, kb, s0);
                Terms w;
                if (PARITY && kstart < r0) weigh_fact(s0, w, sal + GRAN, kb, crow);
                else weigh(s0, w, sal, kb, crow, kstart == r0);
                gemm2(y2, s0, w, kb, no_hook);
            }
        }
    }
#undef ROW_DMA
#undef ST_Y1
#undef ST_Y2
#undef ST_AL
    float onorm = 1.0f, brow = 0.f;
    if constexpr (MODE == MODE_FWD) {
        if constexpr (PARITY) {
            if (chunk > 0) { bpar[0] = fmaf(bfar[0], dec_far, bpar[0]); bpar[1] = fmaf(bfar[1], dec_far, bpar[1]); }
            brow = sum_halves(bpar[0]) + sum_halves(bpar[1]);
        } else {
            brow = sum_halves(bsum);
        }
        const float n = fmaxf(fabsf(brow), __expf(-m_row)) + 1e-6f;
        onorm = 1.0f / n;
    }
    const bool mine = row < S;
    unsigned left_out = 0;   // rows that row_exact writes
    if constexpr (F32) {   // rows that are not finite, from their definition (see not_finite)
        float seen = not_finite(0.f, brow);
#pragma unroll
        for (int d = 0; d < NDB; d++)
#pragma unroll
            for (int r = 0; r < 16; r++) seen = not_finite(seen, oacc[d][r]);
        const unsigned long long halves = __ballot(mine && seen != 0.f);
        left_out = (unsigned)halves | (unsigned)(halves >> 32);
        for (unsigned bad = left_out; bad; bad &= bad - 1) {
            const int b = __builtin_ctz(bad);
            row_exact<D, MODE>(a, bh, chunk, r0 + b, S, hoff, poff, goff, X + (size_t)(r0 + b) * rsX, Y1, Y2, rsA, offA, offO, offB, rsO, rsB,
                               __shfl(inv_n, b), __shfl(dbv, b));
        }
    }
    if constexpr (MODE == MODE_FWD) {
        if (mine && h == 0 && !((left_out >> c32) & 1)) a.Bsum[hoff + row] = brow;
    }
    // A lane holds four columns of every eight of its row; stored from there that is 8 or 16 bytes of 32 rows per instruction.  The wave's 32 rows go through
    // LDS (rows padded by 16 bytes; the stages are free behind the barrier) and leave in whole lines: 64 heads x 16384 x 128, forward
    // 297 -> 283 us, dQ pass 394 -> 378; up to two workgroups per CU level (64 x 1000 x 64 20.6 and 22.2 either way, 8 x 1000 x 64, dQ pass, 16.9 -> 17.2).
    constexpr int RB = D * (int)sizeof(T) + 16, CPR = D * (int)sizeof(T) / 16, NPC = 32 * CPR / 64;
    static_assert(4 * 32 * RB <= (int)Cfg::STAGES_BYTES, "the rows fit the stages");
    char* const stage = smem + wave * 32 * RB;
    auto put = [&](int d, int a4, const typename R::vec4& v) {
        *reinterpret_cast<typename R::vec4*>(stage + c32 * RB + (32 * d + 8 * a4 + 4 * h) * (int)sizeof(T)) = v;
    };
    auto pieces = [&](auto&& f) {   // f(row of the wave, piece of the row, piece number) for the rows to write
#pragma unroll
        for (int i = 0; i < NPC; i++) {
            const int c = lane + 64 * i, rr = c / CPR;
            if (r0 + rr < S && !((left_out >> rr) & 1)) f(rr, c % CPR, i);
        }
    };
    auto piece_at = [&](int rr, int cc) { return *reinterpret_cast<const uint4*>(stage + rr * RB + 16 * cc); };
    uint4 og[PARITY && MODE == MODE_FWD ? NPC : 1];   // output gate, ahead of the barrier
    if constexpr (PARITY && MODE == MODE_FWD) {
        if (a.O) {
            const char* go = reinterpret_cast<const char*>(a.O) + (offB + (size_t)r0 * rsB) * sizeof(T);
            pieces([&](int rr, int cc, int i) { og[i] = *reinterpret_cast<const uint4*>(go + (size_t)rr * rsB * sizeof(T) + 16 * cc); });
        }
    }
    __syncthreads();
    typename R::vec4 low[STRICT && MODE == MODE_FWD ? NDB : 1][4];
#pragma unroll
    for (int d = 0; d < NDB; d++)
#pragma unroll
        for (int a4 = 0; a4 < 4; a4++) {
            f32x4 v;
#pragma unroll
            for (int c = 0; c < 4; c++) v[c] = STRICT ? rounded_product(oacc[d][4 * a4 + c], onorm) : oacc[d][4 * a4 + c] * onorm;
            if constexpr (STRICT && MODE == MODE_FWD) {
                typename R::vec4 hi;
                R::cvt4_split(v, hi, low[d][a4]);
                put(d, a4, hi);
            } else {
                put(d, a4, R::cvt4(v));
            }
        }
    {
        char* const gout = reinterpret_cast<char*>(a.out) + (offO + (size_t)r0 * rsO) * sizeof(T);
        pieces([&](int rr, int cc, int) { *reinterpret_cast<uint4*>(gout + (size_t)rr * rsO * sizeof(T) + 16 * cc) = piece_at(rr, cc); });
        if constexpr (PARITY && MODE == MODE_FWD) {
            if (a.O) {   // (from h as it is written, like the other row kernels)
                char* const gg = reinterpret_cast<char*>(a.out_gated) + (offB + (size_t)r0 * rsB) * sizeof(T);
                pieces([&](int rr, int cc, int i) {
                    struct Pair { typename R::vec4 lo, hi; };
                    const Pair hv = __builtin_bit_cast(Pair, piece_at(rr, cc)), ov = __builtin_bit_cast(Pair, og[i]);
                    Pair res;
                    res.lo = gate4<T>(hv.lo, ov.lo);
                    res.hi = gate4<T>(hv.hi, ov.hi);
                    *reinterpret_cast<Pair*>(gg + (size_t)rr * rsB * sizeof(T) + 16 * cc) = res;
                });
            }
        }
    }
    if constexpr (STRICT && MODE == MODE_FWD) {
        if (a.out_lo) {
#pragma unroll
            for (int d = 0; d < NDB; d++)
#pragma unroll
                for (int a4 = 0; a4 < 4; a4++) put(d, a4, low[d][a4]);
            char* const gl = reinterpret_cast<char*>(a.out_lo) + (hoff + r0) * D * sizeof(T);
            pieces([&](int rr, int cc, int) { *reinterpret_cast<uint4*>(gl + (size_t)rr * D * sizeof(T) + 16 * cc) = piece_at(rr, cc); });
        }
    }
    if constexpr (MODE == MODE_FWD && !PARITY) {
        if (a.O && mine && !((left_out >> c32) & 1)) {  // gated copy from the fp32 accumulators
            const T* og = reinterpret_cast<const T*>(a.O) + offB + (size_t)row * rsB;
            T* outg = reinterpret_cast<T*>(a.out_gated) + offB + (size_t)row * rsB;
#pragma unroll
            for (int d = 0; d < NDB; d++)
#pragma unroll
                for (int a4 = 0; a4 < 4; a4++) {
                    const int col = 32 * d + 8 * a4 + 4 * h;
                    const f32x4 of = __builtin_convertvector(*reinterpret_cast<const typename R::vec4*>(og + col), f32x4);
                    f32x4 v;
#pragma unroll
                    for (int c = 0; c < 4; c++) v[c] = oacc[d][4 * a4 + c] * onorm * silu(of[c]);
                    *reinterpret_cast<typename R::vec4*>(outg + col) = R::cvt4(v);
                }
        }
    }
#endif
}

template <typename T, int D, int MODE, bool STRICT, bool CHUNKS>
static int launch_row_ts(const RowArgs& a, hipStream_t st) {
    using Cfg = RowCfg<T, D>;
    auto kern = row_kernel<T, D, MODE, STRICT, Cfg::per_cu(MODE, STRICT, CHUNKS)>;
    static std::once_flag once;
    static hipError_t attr_rc = hipSuccess;
    std::call_once(once, [&] {
        attr_rc = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)(Cfg::STAGES_BYTES + 2048 * sizeof(double) + sizeof(double) + D * sizeof(float)));
    });
    if (attr_rc != hipSuccess) return (int)attr_rc;
    const int nQT = (a.S + ROW_BQ - 1) / ROW_BQ;
    // (the table is as long as what a row may meet: with the whole sequence's, two workgroups shared a CU up to 118784 positions only, 64 more cost
    // 55 -> 74 us in chunks)
    const int met = a.chunk_len > 0 && a.chunk_len / GRAN < a.NG ? a.chunk_len / GRAN : a.NG;
    hipLaunchKernelGGL(kern, dim3(a.BH * nQT), dim3(256), Cfg::STAGES_BYTES + (size_t)met * sizeof(double) + (a.chunk_len > 0 ? sizeof(double) + D * sizeof(float) : 0), st, a);
    return (int)hipGetLastError();
}

template <typename T, int D, int MODE>
static int launch_row_t(const RowArgs& a, hipStream_t st) {
    if constexpr (Tr<T>::HALF) {
        if (a.precise) return launch_row_ts<T, D, MODE, true, false>(a, st);
        if (D == 64 && a.chunk_len > 0) return launch_row_ts<T, D, MODE, false, true>(a, st);
    }
    return launch_row_ts<T, D, MODE, false, false>(a, st);
}

template <typename T, int MODE>
static int launch_row_d(int D, const RowArgs& a, hipStream_t st) {
    switch (D) {
        case 64: return launch_row_t<T, 64, MODE>(a, st);
        case 128: return launch_row_t<T, 128, MODE>(a, st);
        case 256:
            if constexpr (Tr<T>::HALF) return launch_row_t<T, 256, MODE>(a, st);
            else return MLSTM_ESHAPE;
    }
    return MLSTM_ESHAPE;
}

int launch_row_kernel(int mode, int dtype, int D, const RowArgs& a, hipStream_t st) {
    // fp32 up to one (D = 64) or two (D = 128) workgroups of 32 rows per CU: row_kernel / rowf_kernel, forward, us, in chunks of 128 --
    //   D = 64    256: 14.0 / 10.8   384: 14.3 / 17.4     D = 128   256: 27.6 / 16.9   512: 28.8 / 28.8   640 (uncut): 38.6 / 38.0   1024: 33.1 / 49.5
    if (dtype == MLSTM_F32 && D <= 128 && !g_force_generic && 2ll * a.BH * a.NG <= (D == 64 ? 256 : 512)) return launch_rowf_kernel(mode, D, a, st);
    if (mode == MODE_FWD) {
        switch (dtype) {
            case MLSTM_F32: return launch_row_d<float, MODE_FWD>(D, a, st);
            case MLSTM_F16: return launch_row_d<_Float16, MODE_FWD>(D, a, st);
            case MLSTM_BF16: return launch_row_d<__bf16, MODE_FWD>(D, a, st);
        }
    } else {
        switch (dtype) {
            case MLSTM_F32: return launch_row_d<float, MODE_DQ>(D, a, st);
            case MLSTM_F16: return launch_row_d<_Float16, MODE_DQ>(D, a, st);
            case MLSTM_BF16: return launch_row_d<__bf16, MODE_DQ>(D, a, st);
        }
    }
    return MLSTM_EINVAL;
}

}  // namespace mlstm
