// Scan (recurrent, chunked) form of the mLSTM forward with the silu(o) output gate, fp32, D >= 256 (the tile kernels serve
// the smaller head dimensions).
// Replaces stabilize_fi / precompute_mlstm_triton_scan / reduce_mlstm_triton / mlstm_triton_scan
// (mlstm_scan.py:48-278) and their host driver mlstm_scan (mlstm_scan.py:281-327).
//
// State per head (mlstm_scan.py:16-26): C_t = f'_t C_{t-1} + i'_t v_t (k_t/sqrt D)^T, n_t likewise, m_t the running
// stabiliser.  With a_j = i_j - Fc_j and A_t = max_{j<=t} a_j (the gate pre-pass) the stabilised state is
//     C~_t = sum_{j<=t} exp(a_j - A_t) v_j k_j^T / sqrt(D),     h_t = C~_t q_t / (max(|n~_t . q_t|, exp(-m_t)) + 1e-6).
// The sequence is cut into chunks of 64 positions (one gate granule).  Kernels, in launch order:
//   scan_intra_kernel   per (head, chunk): P_c[t][j] = [j <= t] exp(a_j - A_t) (q_t . k_j)/sqrt(D) for the pairs inside
//                       the chunk (the only place a q.k product is formed), its row sums, and the chunk's contribution
//                       dn_c = sum_j exp(a_j - A_end) k_j / sqrt(D) to the vector state n~.
//   scan_ncarry_kernel  n~ at every chunk end: n~_c = gamma_c n~_{c-1} + dn_c, in place, coalesced streaming.
//   scan_state_kernel   one workgroup per (head, value tile, key range) walks the chunks in order and keeps its
//                       slice of C~ in MFMA accumulator registers for the whole sequence (the matrix carry never
//                       leaves the chip): per chunk  num = decay_t (Q_c C~^T) + P_c V_c, then C~ = gamma C~ + (w V_c)^T K_c.
//                       With more than one key range per value tile the partial numerators go to separate buffers.
//   scan_finish_kernel  per row: b_t = decay_t (n~_{c-1} . q_t) + rowsum_t(P_c),
//                       h = (sum of partial numerators) / (max(|b|, exp(-m)) + 1e-6) * silu(o)   (mlstm_scan.py:273-277).
// HBM traffic: the compulsory stream of q, k, v, o, h, one round trip of the numerator per key range, q once more.
// The same four kernels evaluate the causal weighted sums of the backward (mlstm_scan_bwd.hip) with other operands in the
// places of q, k and v: ScanArgs::finish_mode 2 leaves the numerator itself, ScanArgs::rev walks the operands from their
// last row, ScanArgs::Epilogue says what rides along (a vector sum) and what the last kernel does with a row.
#include "mlstm_device.h"
#include "mlstm_kernels.h"
#include <type_traits>

namespace mlstm {

__device__ __forceinline__ f32x16 mma_f32(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }

// ---------------------------------------------------------------------------------------------------------------
// Four workgroups per (head, chunk): three form one 32x32 block of P each (the head dimension split over the four
// waves, summed through LDS), the fourth clears the masked block and forms the chunk's contribution to n~ (mode 2: to the
// vector sum that rides along, over the rows of v, if there is one).
// The products' operands want one row per lane, which from memory would be 32 bytes per row and instruction; so a wave
// fetches its quarter of the head dimension in blocks of FBW columns with whole 128-byte lines per row (four blocks in
// flight), passes them through a piece of LDS of its own (rows padded by four floats: conflict-free both ways) and reads
// the operands from there.
// Shared partial numerators start from zero: two key ranges add to each element, and 0 + a + b is the same number in either
// order, so results do not depend on which comes first.  Workgroups behind those of the chunks write the zeros (SCAN_ZERO_WG floats each),
// beside their loads and not in a pass of its own.  Whole call, us, a pass of its own / beside: forward 4 heads x 2048 x 1024 318 / 312, 16 x 1024 x 512
// 180 / 175, 4 x 64 x 1024 34.0 / 32.5; forward + backward 2 x 2048 x 1024 908 / 888, 40 x 2048 x 256 1989 / 1976.
constexpr int SCAN_ZERO_WG = 16384;
__device__ __forceinline__ void scan_zeros(float* h, float* hpart, size_t n, size_t total, int wg) {
#pragma unroll 4
    for (int i = 0; i < SCAN_ZERO_WG / 1024; i++) {
        const size_t e = (size_t)wg * SCAN_ZERO_WG + 1024 * i + 4 * threadIdx.x;
        if (e < total) *reinterpret_cast<f32x4*>(e < n ? h + e : hpart + (e - n)) = f32x4{0.f, 0.f, 0.f, 0.f};
    }
}
template <int D>
__global__ __launch_bounds__(256) void scan_intra_kernel(ScanArgs a, int parts) {
    constexpr int DW = D / 4, FBW = DW < 32 ? DW : 32, NB = DW / FBW;   // columns per wave, per block; blocks
    constexpr int LPR = FBW / 4, RPI = 64 / LPR, NLD = LPR;             // lanes per row, rows per load instruction, loads per block
    constexpr int LST = FBW + 4, PD = NB < 4 ? NB : 4;                  // LDS row stride (floats); blocks in flight
    __shared__ __align__(16) float stage[4][64 * LST];                  // per wave: 32 rows of q, then 32 rows of k
    static_assert(64 * LST >= 16 * 64, "the partial sums reuse a wave's stage");
    auto red_at = [&](int w, int r, int l) -> float& { return stage[w][r * 64 + l]; };
    const int wgs = a.BH * a.NC * 4;
    if ((int)blockIdx.x >= wgs) {
        const size_t n = (size_t)a.BH * a.S * D;
        scan_zeros(a.h, a.hpart, n, n * parts, blockIdx.x - wgs);
        return;
    }
    // Consecutive workgroups go to the eight XCDs in turn; the four roles of a chunk read the same rows of q and k, so
    // they take workgroups of one XCD (eight apart), which share an L2.
    int role, cidx;
    if ((wgs & 31) == 0) {
        const int xcd = blockIdx.x & 7, r = blockIdx.x >> 3;
        role = r & 3; cidx = (r >> 2) * 8 + xcd;
    } else {
        role = blockIdx.x & 3; cidx = blockIdx.x >> 2;
    }
    const int c = cidx % a.NC, bh = cidx / a.NC;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5, c32 = lane & 31;
    const int S = a.S;
    const size_t hoff = (size_t)bh * S, poff = (size_t)bh * a.NC * GRAN;
    float* P = a.P + ((size_t)bh * a.NC + c) * GRAN * GRAN;
    const float log2scale = -0.5f * __log2f((float)D);
    auto row_of = [&](int t) { return hoff + (a.rev ? S - 1 - t : t); };   // the row of q, k, v that holds walk position t < S
    const bool mode2 = a.finish_mode == 2, vec = mode2 && a.ep.vec;
    if (role == 3) {
        float* sw = &stage[0][0];
        for (int i = tid; i < 32 * 32; i += 256) P[(i >> 5) * GRAN + 32 + (i & 31)] = 0.f;  // queries 0..31, keys 32..63
        if (mode2 && !vec) return;
        if (tid < GRAN) {
            float w = fast_exp2(a.alpha2[poff + GRAN * c + tid] - a.beta2[poff + GRAN * c + GRAN - 1] + log2scale);
            if (vec && a.col_scale) w *= a.col_scale[row_of(GRAN * c + tid < S ? GRAN * c + tid : S - 1)];
            sw[tid] = w;
        }
        __syncthreads();
        const float* const src = mode2 ? a.v : a.k;
        float* dn = a.Nst + ((size_t)bh * a.NC + c) * D;  // dn[k] = sum_j w_j K[j][k]   (w_j = 0 for padded positions)
        for (int k = tid; k < D; k += 256) {   // (the column's 64 loads are issued together: the loop is bound by their latency)
            float kv[GRAN];
#pragma unroll
            for (int j = 0; j < GRAN; j++) {
                int j0 = GRAN * c + j;
                j0 = j0 < S ? j0 : S - 1;
                kv[j] = src[row_of(j0) * D + k];
            }
            float s0 = 0.f, s1 = 0.f;
#pragma unroll
            for (int j = 0; j < GRAN; j += 2) {
                s0 += sw[j] * kv[j];
                s1 += sw[j + 1] * kv[j + 1];
            }
            dn[k] = s0 + s1;
        }
        return;
    }
    const int tb = role > 0, jb = role > 1;  // 32x32 block: queries 32*tb.., keys 32*jb..
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
    {
        float* const stg = stage[wave];
        const int lrow = lane / LPR, lcol = 4 * (lane % LPR);
        const float* src[NLD];   // this lane's rows: load i covers stage rows RPI*i .. RPI*i + RPI-1 (0..31: q, 32..63: k)
#pragma unroll
        for (int i = 0; i < NLD; i++) {
            const int r = RPI * i + lrow;
            int t = GRAN * c + (r < 32 ? 32 * tb + r : 32 * jb + r - 32);
            t = t < S ? t : S - 1;
            src[i] = (r < 32 ? a.q : a.k) + row_of(t) * D + wave * DW + lcol;
        }
        f32x4 rg[PD][NLD];
#pragma unroll
        for (int b = 0; b < PD; b++)
#pragma unroll
            for (int i = 0; i < NLD; i++) rg[b][i] = *reinterpret_cast<const f32x4*>(src[i] + b * FBW);
#pragma unroll
        for (int b = 0; b < NB; b++) {
#pragma unroll
            for (int i = 0; i < NLD; i++) *reinterpret_cast<f32x4*>(stg + (RPI * i + lrow) * LST + lcol) = rg[b % PD][i];
            if (b + PD < NB) {
#pragma unroll
                for (int i = 0; i < NLD; i++) rg[b % PD][i] = *reinterpret_cast<const f32x4*>(src[i] + (b + PD) * FBW);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int s = 0; s < FBW / 8; s++) {
                const f32x4 qv = *reinterpret_cast<const f32x4*>(stg + c32 * LST + 8 * s + 4 * h);
                const f32x4 kv = *reinterpret_cast<const f32x4*>(stg + (32 + c32) * LST + 8 * s + 4 * h);
#pragma unroll
                for (int e = 0; e < 4; e++) acc = mma_f32(qv[e], kv[e], acc);  // rows = queries, columns = keys
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();   // (every wave is done with its stage: the partial sums go there)
#pragma unroll
    for (int r = 0; r < 16; r++) red_at(wave, r, lane) = acc[r];
    __syncthreads();
    // accumulator: column (key) = 32*jb + c32, rows (queries) 32*tb + 8*(r/4) + 4h + r%4; wave w finishes r = 4w..4w+3
    const int jl = 32 * jb + c32;
    const float alj = a.alpha2[poff + GRAN * c + jl];
    const float cs = !vec ? 0.f : (a.col_scale ? a.col_scale[row_of(GRAN * c + jl < S ? GRAN * c + jl : S - 1)] : 1.0f);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int r = 4 * wave + e;
        const int tl = 32 * tb + 8 * (r >> 2) + 4 * h + (r & 3);
        float sum = red_at(0, r, lane) + red_at(1, r, lane) + red_at(2, r, lane) + red_at(3, r, lane);
        if (vec) sum += cs * (a.ep.row_scale ? a.ep.row_scale[hoff + (GRAN * c + tl < S ? GRAN * c + tl : S - 1)] : 1.0f);
        float p = sum * fast_exp2(alj - a.beta2[poff + GRAN * c + tl] + log2scale);
        if (jl > tl) p = 0.f;
        P[tl * GRAN + jl] = p;
    }
}

// n~_c = gamma_c n~_{c-1} + dn_c over the chunks of a head, in place.  One thread per column; the decays of 256 chunks at
// a time are formed side by side, and the column's sums are fetched eight chunks ahead of the serial sum.
__global__ __launch_bounds__(256) void scan_ncarry_kernel(ScanArgs a) {
    __shared__ float sgam[256];
    const int bh = blockIdx.y, tid = threadIdx.x, k = blockIdx.x * 256 + tid, NC = a.NC;
    const bool mine = k < a.D;
    const size_t poff = (size_t)bh * NC * GRAN;
    float* n = a.Nst + (size_t)bh * NC * a.D + (mine ? k : 0);
    float run = mine ? n[0] : 0.f;
    for (int c0 = 1; c0 < NC; c0 += 256) {
        __syncthreads();
        if (const int c = c0 + tid; c < NC)
            sgam[tid] = fast_exp2(a.beta2[poff + GRAN * c - 1] - a.beta2[poff + GRAN * c + GRAN - 1] +
                                  (float)(a.G2[(size_t)bh * NC + c] - a.G2[(size_t)bh * NC + c - 1]));
        __syncthreads();
        const int cn = NC - c0 < 256 ? NC - c0 : 256;
        for (int cb = 0; cb < cn && mine; cb += 8) {
            float x[8];
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] = cb + j < cn ? n[(size_t)(c0 + cb + j) * a.D] : 0.f;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                run = (cb + j < cn ? sgam[cb + j] : 1.0f) * run + x[j];
                if (cb + j < cn) n[(size_t)(c0 + cb + j) * a.D] = run;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// One workgroup: VT = 32 VB value columns, four waves of KPW = 32 NKB key columns each; a wave holds its [KPW x VT] piece of
// C~ in accumulator registers.  The products are those of Tr<float>, three bf16 terms per operand: six 32x32x16 MFMAs per
// block against eight 32x32x2 ones at twice the cycles, and the vector instructions of a split go between them.
//
// What bounds it: one wave per SIMD issues everything, about 1250 split instructions to 200 MFMAs per chunk (VB = NKB = 2),
// so every operand is split as seldom as it can be.  64 value columns per workgroup and not 32 halve the splits (and the L2
// traffic) of Q and K; a wave splits a quarter of the weighted values and the others read its terms from LDS; the state's
// terms serve both query blocks.  Q comes with direct copies into a piece of LDS that belongs to the wave (its fragments want
// one row per lane: 64 lines per load instruction from memory), K and V from memory into registers, 128 bytes per row.
// Measured on 4 heads x 2048 x 1024, forward: 17,200 cycles per chunk (read-out 6400, update 5600) where the 32x32x2 kernel
// took 27,900; whole call 393 -> 308 us.  Eight waves of half the tile each took 18,400: two waves per SIMD overlap splits and
// MFMAs, and lose it again at twice the barriers.
//
// A sequence may also be cut into segments of seg_chunks chunks that run side by side (blockIdx.y), for the cases in
// which heads x value tiles x key ranges alone leave most of the chip idle (one long sequence, small D):
//   STATE_ONLY = true   every segment but the last walks its chunks from a zero state, updates only, and leaves the
//                       state at its end (accumulator registers as they are) in seg_state;
//   scan_segcarry_kernel turns those into the true states at the segment ends (a short serial sum over the segments);
//   STATE_ONLY = false  the walk proper: segment s > 0 starts from the state at the end of segment s - 1.
// REV: q, k and v are walked from their last row (ScanArgs::rev).  A complete chunk's 64 rows then lie in front of the row of
// its first position; the lane parts of the addresses stay non-negative by counting from the chunk's last position.
constexpr int SCAN_NW = 4;   // waves per workgroup: one per SIMD, each wants the full register file
template <int VB, int NKB> constexpr int scan_state_lds() {
    return SCAN_NW * 64 * 32 * NKB * 4      // Q of a chunk, per wave
         + SCAN_NW * 8 * VB * 64 * 16       // partial numerators
         + 4 * VB * 3 * 64 * 16             // terms of the weighted values
         + 3 * 2 * GRAN * 4;                // gate vectors
}
template <int D, int VB, int NKB, bool STATE_ONLY, bool REV, bool SHARED>
__global__ __launch_bounds__(SCAN_NW * 64) void scan_state_kernel(ScanArgs a) {
    constexpr int NW = SCAN_NW, KPW = 32 * NKB, KS = D / KPW / NW, VT = 32 * VB, NVT = D / VT, NS = 2 * NKB;
    static_assert(KS >= 1 && KS * NW * KPW == D && NVT * VT == D, "key ranges and value tiles must divide D");
    typedef Tr<float> X;
    typedef X::frag frag;
    typedef X::terms terms;
    typedef Swz<float, KPW> Z;
    extern __shared__ __align__(16) float lds[];
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, c32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float* const qst = lds + wave * 64 * KPW;                                      // [query][key column], swizzled
    f32x4 (*red)[8 * VB][64] = reinterpret_cast<f32x4 (*)[8 * VB][64]>(lds + NW * 64 * KPW);   // [wave][(tb, vb, r / 4)][lane]
    bf16x8 (*vterm)[VB][3][64] = reinterpret_cast<bf16x8 (*)[VB][3][64]>(lds + NW * 64 * KPW + NW * 8 * VB * 256);   // [16 positions][vb][term][lane]
    float (*sgate)[2][GRAN] = reinterpret_cast<float (*)[2][GRAN]>(lds + NW * 64 * KPW + NW * 8 * VB * 256 + 4 * VB * 3 * 256);   // [chunk mod 3][0: key weights w_j, 1: query decays][position]
    const int bh = blockIdx.x % a.BH;
    const int rest = blockIdx.x / a.BH;
    const int vt = rest % NVT, ks = rest / NVT;
    const int S = a.S, NC = a.NC;
    const int seg = blockIdx.y, c_begin = seg * a.seg_chunks, c_end = c_begin + a.seg_chunks < NC ? c_begin + a.seg_chunks : NC;
    const size_t hoff = (size_t)bh * S, poff = (size_t)bh * NC * GRAN;
    const float* Q = a.q + hoff * D;
    const float* K = a.k + hoff * D;
    const float* V = a.v + hoff * D;
    const double* G2 = a.G2 + (size_t)bh * NC;
    const int part_no = SHARED ? ks / 2 : ks;   // (ScanArgs::shared)
    float* out = (part_no == 0 ? a.h : a.hpart + (size_t)(part_no - 1) * a.BH * S * D) + hoff * D;
    const int kbase = (ks * NW + wave) * KPW, v0 = VT * vt;
    const float log2scale = -0.5f * __log2f((float)D);
    // Position 16 s + 8 h + e of a chunk is contraction element e of lane half h in step s.
    const int hrow = REV ? 8 * (1 - h) : 8 * h;           // the lane half's first row in 16 rows as they lie in memory
    const int v_lofs = hrow * D + v0 + c32;               // lane part of a value address (column v0 + c32)
    const int k_lofs = hrow * D + kbase + c32;            // lane part of a key address
    auto row_of = [&](int t) { return (size_t)(REV ? S - 1 - t : t); };   // the row that holds walk position t < S
    auto row_in = [](int s, int e) { return (size_t)(REV ? 48 - 16 * s + 7 - e : 16 * s + e); };

    // Gate vectors of a chunk: weights of its keys, decays of its queries (from the previous chunk end).  The carried
    // state is kept as st = C~ / Gamma with a running power of two Gamma <= 1, so that the per-chunk decay gamma_c
    // multiplies into Gamma (folded into these vectors) and the registers are rescaled only when Gamma gets small.
    float lg = 0.f;  // log2 Gamma for the read-out of the next chunk to prepare
    struct Gates { float x, bprev, bend; double g, gprev; };
    int vzero = 0;   // (as vector loads: a scalar load in flight would make every wait for LDS a wait for it)
    asm volatile("" : "+v"(vzero));
    const float* const mygate = (tid < GRAN ? a.alpha2 : a.beta2) + poff + (tid & (GRAN - 1));
    auto gates_fetch = [&](int c) {
        Gates g;
        const int cp = c > 0 ? c - 1 : 0;
        g.bprev = a.beta2[poff + GRAN * cp + GRAN - 1 + vzero];
        g.bend = a.beta2[poff + GRAN * c + GRAN - 1 + vzero];
        g.g = G2[c + vzero];
        g.gprev = G2[cp + vzero];
        g.x = tid < 2 * GRAN ? mygate[(size_t)GRAN * c] : 0.f;
        return g;
    };
    auto gates_store = [&](int c, const Gates& g) {   // returns the rescale before this chunk's update (0: none)
        const float dG = (float)(g.g - g.gprev);
        const float dec_add = g.bprev + dG + lg;
        float lnew = lg + (c > 0 ? g.bprev - g.bend + dG : 0.f), rescale = 0.f;
        if (lnew < -24.f) { rescale = lnew; lnew = 0.f; }
        const float w_add = log2scale - g.bend - lnew;
        lg = lnew;
        const int pos = tid & (GRAN - 1);
        if (tid < GRAN) sgate[c % 3][0][pos] = fast_exp2(g.x + w_add);
        else if (tid < 2 * GRAN) sgate[c % 3][1][pos] = c > 0 ? fast_exp2(dec_add - g.x) : 1.0f;
        return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, rescale)));
    };
    // Q of a chunk into the wave's LDS (rows clamped: the chunk may be the partial one).  The 16-byte copies want rows on 16-byte
    // boundaries; every other access of these kernels takes any boundary of four bytes.
    const unsigned qst_off = __builtin_amdgcn_readfirstlane(lds_offset_of(qst));
    constexpr int RPI = 64 / Z::CPR, QI = 64 / RPI, QP = 16 / RPI;   // rows per copy instruction, instructions, period of the swizzle key
    unsigned q_lofs[QP];               // lane part of the source, in bytes
#pragma unroll
    for (int i = 0; i < QP; i++)
        q_lofs[i] = (unsigned)(((REV ? RPI - 1 - lane / Z::CPR : lane / Z::CPR) * D + 4 * ((lane % Z::CPR) ^ Z::key(RPI * i + lane / Z::CPR))) * 4);
    auto fetch_q_part = [&](int c, int part) {   // a quarter of a complete chunk
        const float* base = Q + (REV ? (size_t)(S - GRAN - GRAN * c) : (size_t)(GRAN * c)) * D + kbase;
#pragma unroll
        for (int j = 0; j < QI / 4; j++) {
            const int i = part * (QI / 4) + j;
            dma16_s(base + (size_t)(REV ? GRAN - RPI - RPI * i : RPI * i) * D, q_lofs[i % QP], qst_off, 1024 * i);
        }
    };
    const bool q16 = (reinterpret_cast<size_t>(a.q) & 15) == 0;   // (uniform; D is a multiple of four: one answer for all rows)
    auto fetch_q_clamped = [&](int c) {
        if (!q16) {   // rows of a view that starts inside a tensor: the same places, four bytes at a time
#pragma unroll 1
            for (int i = 0; i < KPW; i++) {
                const int w = 64 * i + lane, r = w / KPW, p = w % KPW;
                const int t = GRAN * c + r < S ? GRAN * c + r : S - 1;
                dma4(Q + row_of(t) * D + kbase + 4 * ((p / 4) ^ Z::key(r)) + p % 4, __builtin_amdgcn_readfirstlane(qst_off + 256 * i));
            }
            return;
        }
#pragma unroll 1
        for (int i = 0; i < QI; i++) {
            const int r = RPI * i + lane / Z::CPR;
            const int t = GRAN * c + r < S ? GRAN * c + r : S - 1;
            dma16(Q + row_of(t) * D + kbase + 4 * ((lane % Z::CPR) ^ Z::key(r)), __builtin_amdgcn_readfirstlane(qst_off + 1024 * i));
        }
    };
    auto read_q = [&](int s, int tb) {   // key columns 16 s + 8 x + 4 h + e' of row 32 tb + c32, the order of from_acc
        const char* base = reinterpret_cast<const char*>(qst);
        const f32x4 x0 = *reinterpret_cast<const f32x4*>(base + Z::off(32 * tb + c32, 16 * s + 4 * h));
        const f32x4 x1 = *reinterpret_cast<const f32x4*>(base + Z::off(32 * tb + c32, 16 * s + 8 + 4 * h));
        return __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7);
    };

    f32x16 st[NKB][VB];  // st[kb][vb][r] = C~[v = v0 + 32 vb + c32][k = kbase + 32 kb + 8*(r/4) + 4h + r%4]
    // a workgroup's state in seg_state: [segment][workgroup][wave][kb][vb][r][lane]
    const size_t seg_stride = (size_t)gridDim.x * NW * NKB * VB * 16 * 64;
    float* const seg_mine = a.seg_state + ((size_t)blockIdx.x * NW + wave) * NKB * VB * 16 * 64 + lane;
#pragma unroll
    for (int b = 0; b < NKB * VB; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) st[b / VB][b % VB][r] = 0.f;
    if (!STATE_ONLY && seg > 0) {
#pragma unroll
        for (int b = 0; b < NKB * VB; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) st[b / VB][b % VB][r] = seg_mine[(size_t)(seg - 1) * seg_stride + (b * 16 + r) * 64];
    }
    if constexpr (!STATE_ONLY) fetch_q_clamped(c_begin);
    float lg_done = 0.f;   // log2 Gamma of the last chunk whose update is in st
    float rescale_cur = gates_store(c_begin, gates_fetch(c_begin));
    __syncthreads();

    // One chunk.  LAST: the final chunk of a walk (possibly partial: rows clamped; no state update follows).
    auto chunk = [&](const int c, auto last_tag) {
        constexpr bool LAST = decltype(last_tag)::value;
        const int t0 = GRAN * c;
        const float* sw = sgate[c % 3][0];
        const float* sdec = sgate[c % 3][1];
        // uniform: the first of the chunk's 64 rows in memory (REV: the row of its last position; only complete chunks use it)
        const size_t r0 = LAST ? 0 : (REV ? (size_t)(S - GRAN - t0) : (size_t)t0);
        const float* vrow = V + r0 * D;
        const float* krow = K + r0 * D;
        frag vraw[VB];          // this wave's 16 positions of the values (step `wave`)
        frag kraw[4][NKB];
        auto load_v = [&]() {
#pragma unroll
            for (int vb = 0; vb < VB; vb++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    if constexpr (LAST) {
                        int j = t0 + 16 * wave + 8 * h + e;
                        j = j < S ? j : S - 1;
                        vraw[vb][e] = V[row_of(j) * D + v0 + 32 * vb + c32];
                    } else {
                        vraw[vb][e] = (vrow + row_in(wave, e) * D + 32 * vb)[v_lofs];
                    }
                }
        };
        auto load_k = [&](int s) {
#pragma unroll
            for (int kb = 0; kb < NKB; kb++)
#pragma unroll
                for (int e = 0; e < 8; e++) kraw[s][kb][e] = (krow + row_in(s, e) * D + 32 * kb)[k_lofs];
        };
        // The pairs inside the chunk: 2 VB blocks of P V with four steps each, step `wave` of block (tb, vb) in key range
        // (tb + 2 vb) mod KS.
        auto pair_mine = [&](int tb, int vb) { return KS == 1 || (tb + 2 * vb) % KS == ks; };
        frag praw[2];
        if constexpr (!STATE_ONLY) {
            dma_wait();   // Q of this chunk
            const float* Pc = a.P + ((size_t)bh * NC + c) * GRAN * GRAN + 16 * wave + 8 * h;
#pragma unroll
            for (int tb = 0; tb < 2; tb++) praw[tb] = *reinterpret_cast<const frag*>(Pc + (32 * tb + c32) * GRAN);
        }
        load_v();
        Gates gn;
        lg_done = lg;
        if constexpr (!LAST) gn = gates_fetch(c + 1);

        // N splits, step by step in the gaps of PN products: 5 PN gaps of 5 N steps
        X::Splitting sp;
        auto gap = [&](auto n_tag, auto pn_tag, auto g_tag, auto&& src, auto&& dst) __attribute__((always_inline)) {
            constexpr int N = decltype(n_tag)::value, PN = decltype(pn_tag)::value, g = decltype(g_tag)::value;
            constexpr int i0 = g * N / PN, i1 = (g + 1) * N / PN;
            static_for<i1 - i0>([&](auto d) __attribute__((always_inline)) {
                constexpr int job = (i0 + d) / 5, step = (i0 + d) % 5;
                if constexpr (step == 0) sp.start(src(std::integral_constant<int, job>{}));
                sp.template step<step>(dst(std::integral_constant<int, job>{}));
            });
            __builtin_amdgcn_sched_barrier(0);
        };
        terms kt[2][NKB];
        if constexpr (STATE_ONLY) {
#pragma unroll
            for (int s = 0; s < 4; s++) load_k(s);
#pragma unroll
            for (int kb = 0; kb < NKB; kb++) kt[0][kb] = X::split(kraw[0][kb]);
        }
        terms vt_mine[VB];   // this wave's share of the weighted values
        auto weighted = [&](int vb) {
            const f32x4 w0 = *reinterpret_cast<const f32x4*>(sw + 16 * wave + 8 * h), w1 = *reinterpret_cast<const f32x4*>(sw + 16 * wave + 8 * h + 4);
            return vraw[vb] * __builtin_shufflevector(w0, w1, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        if constexpr (STATE_ONLY) {
#pragma unroll
            for (int vb = 0; vb < VB; vb++) vt_mine[vb] = X::split(weighted(vb));
        }
        const bool next_full = q16 && t0 + 2 * GRAN <= S;
        // ---- read-out of the carried state: acc[tb][vb] = decay_t * Q_c[32 tb.., k-range of this wave] . C~^T
        f32x16 acc[2][VB];
        if constexpr (!STATE_ONLY) {
#pragma unroll
            for (int b = 0; b < 2 * VB; b++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[b / VB][b % VB][r] = 0.f;
            terms qt[2][2], ct[2][VB];
            frag qraw[2];
#pragma unroll
            for (int tb = 0; tb < 2; tb++) qraw[tb] = read_q(0, tb);
#pragma unroll
            for (int vb = 0; vb < VB; vb++) ct[0][vb] = X::split(X::from_acc(st[0][vb], 0));
#pragma unroll
            for (int tb = 0; tb < 2; tb++) qt[0][tb] = X::split(qraw[tb]);
            static_for<NS>([&](auto s_tag) __attribute__((always_inline)) {
                constexpr int s = decltype(s_tag)::value, PN = 2 * VB;
                constexpr bool more = s + 1 < NS;
                if constexpr (more) {
#pragma unroll
                    for (int tb = 0; tb < 2; tb++) qraw[tb] = read_q(s + 1, tb);
                }
                if constexpr (!LAST) {
#pragma unroll
                    for (int i = 0; i < 4 / NS; i++) load_k(s * (4 / NS) + i);
                }
                __builtin_amdgcn_sched_barrier(0);
                static_for<PN>([&](auto p_tag) __attribute__((always_inline)) {
                    constexpr int p = decltype(p_tag)::value, tb = p / VB, vb = p % VB;
                    if constexpr (!more && !LAST) {   // (this wave's reads of its piece are over: queries of the next chunk)
                        if (next_full) {
#pragma unroll
                            for (int j = 0; j < 4 / PN; j++) fetch_q_part(c + 1, p * (4 / PN) + j);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    X::mma_between(acc[tb][vb], qt[s & 1][tb], ct[s & 1][vb], [&](auto i_tag) __attribute__((always_inline)) {
                        typedef std::integral_constant<int, 5 * p + decltype(i_tag)::value> G;
                        typedef std::integral_constant<int, PN> P;
                        if constexpr (more)   // the next step's state and queries
                            gap(std::integral_constant<int, VB + 2>{}, P{}, G{},
                                [&](auto j) __attribute__((always_inline)) {
                                    if constexpr (j < VB) return X::from_acc(st[(s + 1) / 2][j < VB ? (int)j : 0], (s + 1) % 2);
                                    else return qraw[j - VB];
                                },
                                [&](auto j) __attribute__((always_inline)) -> terms& {
                                    if constexpr (j < VB) return ct[(s + 1) & 1][j < VB ? (int)j : 0];
                                    else return qt[(s + 1) & 1][j - VB];
                                });
                        else if constexpr (!LAST)   // the first keys of the update and the weighted values
                            gap(std::integral_constant<int, NKB + VB>{}, P{}, G{},
                                [&](auto j) __attribute__((always_inline)) {
                                    if constexpr (j < NKB) return kraw[0][j < NKB ? (int)j : 0];
                                    else return weighted(j - NKB);
                                },
                                [&](auto j) __attribute__((always_inline)) -> terms& {
                                    if constexpr (j < NKB) return kt[0][j < NKB ? (int)j : 0];
                                    else return vt_mine[j - NKB];
                                });
                    });
                });
            });
            if constexpr (!LAST) {
                if (!next_full) fetch_q_clamped(c + 1);
            }
#pragma unroll
            for (int tb = 0; tb < 2; tb++)
#pragma unroll
                for (int x = 0; x < 4; x++) {
                    const f32x4 dec = *reinterpret_cast<const f32x4*>(sdec + 32 * tb + 8 * x + 4 * h);
#pragma unroll
                    for (int vb = 0; vb < VB; vb++)
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[tb][vb][4 * x + e] *= dec[e];
                }
            // ---- pairs inside the chunk: acc += P_c[:, 16 wave ..] . V_c
#pragma unroll
            for (int vb = 0; vb < VB; vb++)
#pragma unroll
                for (int tb = 0; tb < 2; tb++)
                    if (pair_mine(tb, vb)) X::mma(acc[tb][vb], praw[tb], vraw[vb]);
        }
        // ---- terms of the weighted values, partial numerators of the waves and the next gates, for all waves.  The first
        // barrier: everybody is done with those of the chunk before.
        float rescale_next = 0.f;
        __syncthreads();
        if constexpr (!LAST) {
#pragma unroll
            for (int vb = 0; vb < VB; vb++) {
                vterm[wave][vb][0][lane] = vt_mine[vb].hi;
                vterm[wave][vb][1][lane] = vt_mine[vb].mid;
                vterm[wave][vb][2][lane] = vt_mine[vb].lo;
            }
            rescale_next = gates_store(c + 1, gn);
        }
        if constexpr (!STATE_ONLY) {
#pragma unroll
            for (int g = 0; g < 8 * VB; g++) {
                const f32x16& x = acc[g / (4 * VB)][g / 4 % VB];
                const int r = 4 * (g % 4);
                red[wave][g][lane] = f32x4{x[r], x[r + 1], x[r + 2], x[r + 3]};
            }
        }
        __syncthreads();
        f32x4 part[NW];
        auto sum_read = [&](int g) {   // four rows of the numerator: the waves' parts ...
#pragma unroll
            for (int w = 0; w < NW; w++) part[w] = red[w][g][lane];
        };
        auto sum_store = [&](int g) {  // ... their sum
            f32x4 sum = part[0];
#pragma unroll
            for (int w = 1; w < NW; w++) sum += part[w];
            const int t = t0 + 32 * (g / (4 * VB)) + 8 * (g % 4) + 4 * h;
            float* o = out + (size_t)t * D + v0 + 32 * (g / 4 % VB) + c32;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (!LAST || t + e < S) {
                    if constexpr (SHARED) unsafeAtomicAdd(o + e * D, sum[e]);   // (one hardware add, nothing returned)
                    else o[e * D] = sum[e];
                }
        };
        if constexpr (LAST) {
            for (int g = wave; g < 8 * VB; g += NW) { sum_read(g); sum_store(g); }
        } else {
            // ---- state update: st += (w V_c)^T K_c (the weights carry 1/Gamma), rescaled first when Gamma got small
            if (rescale_cur != 0.f) {
                const float f = fast_exp2(rescale_cur);
#pragma unroll
                for (int b = 0; b < NKB * VB; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++) st[b / VB][b % VB][r] *= f;
            }
            rescale_cur = rescale_next;
            terms vt_s[2][VB];
            auto read_v = [&](int s, terms (&t)[VB]) {
#pragma unroll
                for (int vb = 0; vb < VB; vb++) t[vb] = terms{vterm[s][vb][0][lane], vterm[s][vb][1][lane], vterm[s][vb][2][lane]};
            };
            read_v(0, vt_s[0]);
            static_for<4>([&](auto s_tag) __attribute__((always_inline)) {
                constexpr int s = decltype(s_tag)::value, PN = NKB * VB;
                if constexpr (s < 3) read_v(s + 1, vt_s[(s + 1) & 1]);
                if constexpr (!STATE_ONLY && s < 2 * VB) sum_read(wave + NW * s);
                __builtin_amdgcn_sched_barrier(0);
                static_for<PN>([&](auto p_tag) __attribute__((always_inline)) {
                    constexpr int p = decltype(p_tag)::value, kb = p / VB, vb = p % VB;
                    X::mma_between(st[kb][vb], kt[s & 1][kb], vt_s[s & 1][vb], [&](auto i_tag) __attribute__((always_inline)) {
                        if constexpr (s < 3)
                            gap(std::integral_constant<int, NKB>{}, std::integral_constant<int, PN>{}, std::integral_constant<int, 5 * p + decltype(i_tag)::value>{},
                                [&](auto j) __attribute__((always_inline)) { return kraw[s + 1][j]; },
                                [&](auto j) __attribute__((always_inline)) -> terms& { return kt[(s + 1) & 1][j]; });
                    });
                    if constexpr (!STATE_ONLY && s < 2 * VB && p == PN / 2) {
                        sum_store(wave + NW * s);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                });
            });
        }
    };
    if constexpr (STATE_ONLY) {
        // (never the last segment: every chunk is complete and has a successor whose gates the walk fetches ahead)
        for (int c = c_begin; c < c_end; c++) chunk(c, std::false_type{});
        const float f = fast_exp2(lg_done);   // st = C~ / Gamma
#pragma unroll
        for (int b = 0; b < NKB * VB; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) seg_mine[(size_t)seg * seg_stride + (b * 16 + r) * 64] = st[b / VB][b % VB][r] * f;
    } else {
        for (int c = c_begin; c + 1 < c_end; c++) chunk(c, std::false_type{});
        chunk(c_end - 1, std::true_type{});
    }
}

// States at the segment ends from the segments' own sums, in place: x_s = exp(A_{e(s-1)} - A_{e(s)}) x_{s-1} + x_s with
// e(s) the last position of segment s.  One thread per state element; elems = floats per segment, wg_elems = floats per
// workgroup of the state kernel (whose index modulo BH is the head).
__global__ __launch_bounds__(256) void scan_segcarry_kernel(ScanArgs a, size_t elems, int wg_elems) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= elems) return;
    const int bh = (int)((e / wg_elems) % a.BH);
    const size_t poff = (size_t)bh * a.NC * GRAN;
    float run = a.seg_state[e];
    for (int s = 1; s + 1 < a.nseg; s++) {
        const int c1 = (s + 1) * a.seg_chunks - 1, c0 = s * a.seg_chunks - 1;   // last chunks of segments s and s - 1
        const double A1 = (double)a.beta2[poff + GRAN * c1 + GRAN - 1] - a.G2[(size_t)bh * a.NC + c1];
        const double A0 = (double)a.beta2[poff + GRAN * c0 + GRAN - 1] - a.G2[(size_t)bh * a.NC + c0];
        run = fast_exp2((float)(A0 - A1)) * run + a.seg_state[(size_t)s * elems + e];
        a.seg_state[(size_t)s * elems + e] = run;
    }
}

// ---------------------------------------------------------------------------------------------------------------
// The numerator of a row from its definition (see not_finite in mlstm_device.h): columns 4 lane + 256 n .. of
//   sum_{j<=t} exp(a_j - A_t) / sqrt(D) (q_t . k_j) v_j,
// the vector sum that may ride along (ScanArgs::Epilogue::vec) for the pairs inside the row's chunk only, as in P.
template <int D>
__device__ __forceinline__ void scan_numerator_exact(const ScanArgs& a, int bh, int t, f32x4 (&x)[D / 256]) {
    constexpr int NB = D / 256;
    const int lane = threadIdx.x & 63, S = a.S, c = t / GRAN;
    const size_t hoff = (size_t)bh * S, poff = (size_t)bh * a.NC * GRAN;
    auto row_of = [&](int j) { return (hoff + (a.rev ? S - 1 - j : j)) * D; };
    const float log2scale = -0.5f * __log2f((float)D);
    const bool vec = a.finish_mode == 2 && a.ep.vec;
    const float rs = vec && a.ep.row_scale ? a.ep.row_scale[hoff + t] : 1.0f;
    const double G = a.G2[(size_t)bh * a.NC + c];
    const float beta = a.beta2[poff + t];
    const float* q = a.q + row_of(t) + 4 * lane;
#pragma unroll
    for (int n = 0; n < NB; n++) x[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int j = 0; j <= t; j++) {
        const size_t r = row_of(j);
        float s = 0.f;
#pragma unroll 1   // (as few registers as it takes: the kernel around this wants its waves)
        for (int k = 0; k < D; k += 256) {
            const f32x4 qv = *reinterpret_cast<const f32x4*>(q + k), kv = *reinterpret_cast<const f32x4*>(a.k + r + 4 * lane + k);
            s += qv[0] * kv[0] + qv[1] * kv[1] + qv[2] * kv[2] + qv[3] * kv[3];
        }
        s = wave_reduce<OpAdd>(s);
        if (vec && j / GRAN == c) s += rs * (a.col_scale ? a.col_scale[hoff + (a.rev ? S - 1 - j : j)] : 1.0f);
        s *= fast_exp2(a.alpha2[poff + j] - beta + (float)(G - a.G2[(size_t)bh * a.NC + j / GRAN]) + log2scale);
#pragma unroll
        for (int n = 0; n < NB; n++) {
            const int k = 4 * lane + 256 * n;
            x[n] += s * *reinterpret_cast<const f32x4*>(a.v + r + k);
        }
        if ((j & 15) == 15) {   // (a row of nothing but NaN stays that)
            bool number = false;
#pragma unroll
            for (int n = 0; n < NB; n++)
#pragma unroll
                for (int e = 0; e < 4; e++) number = number || x[n][e] == x[n][e];
            if (!__any(number)) break;
        }
    }
}

// one wave per row: normaliser sum, then the row of h
template <int D>
__global__ __launch_bounds__(256) void scan_finish_kernel(ScanArgs a, int KS) {
    constexpr int NB = D / 256;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t rows = (size_t)a.BH * a.S;
    for (size_t row = (size_t)blockIdx.x * 4 + wave; row < rows; row += (size_t)gridDim.x * 4) {
        const int bh = (int)(row / a.S), t = (int)(row % a.S), c = t / GRAN;
        const size_t poff = (size_t)bh * a.NC * GRAN;
        f32x4 num[NB];   // the row's numerator, columns 4 lane + 256 n ..
        float seen = 0.f;
#pragma unroll
        for (int n = 0; n < NB; n++) {
            const int k = 4 * lane + 256 * n;
            num[n] = *reinterpret_cast<const f32x4*>(a.h + row * D + k);
            for (int p = 1; p < KS; p++) num[n] += *reinterpret_cast<const f32x4*>(a.hpart + ((size_t)(p - 1) * rows + row) * D + k);
#pragma unroll
            for (int e = 0; e < 4; e++) seen = not_finite(seen, num[n][e]);
        }
        if (__any(seen != 0.f)) scan_numerator_exact<D>(a, bh, t, num);
        if (a.finish_mode == 2) {
            const ScanArgs::Epilogue& ep = a.ep;
            const size_t orow = ep.out_rev ? (size_t)bh * a.S + (a.S - 1 - t) : row;
            const bool carried = ep.vec && c > 0;
            // rs_t decay_t, the factor of the vector sum at the end of the chunk before
            const float cf = !carried ? 0.f : (ep.row_scale ? ep.row_scale[row] : 1.0f) *
                                                  fast_exp2(a.beta2[poff + GRAN * c - 1] - a.beta2[poff + t] +
                                                            (float)(a.G2[(size_t)bh * a.NC + c] - a.G2[(size_t)bh * a.NC + c - 1]));
            const float* cr = carried ? a.Nst + ((size_t)bh * a.NC + c - 1) * D : nullptr;
            const float wd = ep.wd_alpha2 ? fast_exp2(ep.wd_alpha2[poff + (orow - (size_t)bh * a.S)] - ep.wd_beta2[poff + (orow - (size_t)bh * a.S)]) : 1.0f;
            float* const dst = (ep.out ? ep.out : a.h) + orow * D;
            float acc = 0.f;
#pragma unroll
            for (int n = 0; n < NB; n++) {
                const int k = 4 * lane + 256 * n;
                f32x4 x = num[n];
                if (carried) {
                    const f32x4 cv = *reinterpret_cast<const f32x4*>(cr + k);
#pragma unroll
                    for (int e = 0; e < 4; e++) x[e] += cf * cv[e];
                }
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] *= wd;
                if (ep.dot_with) {
                    const f32x4 dv = *reinterpret_cast<const f32x4*>(ep.dot_with + orow * D + k);
                    acc += dv[0] * x[0] + dv[1] * x[1] + dv[2] * x[2] + dv[3] * x[3];
                }
                *reinterpret_cast<f32x4*>(dst + k) = x;
            }
            if (ep.dot_with) {
                acc = wave_reduce<OpAdd>(acc);
                if (lane == 0) {
                    ep.dot_out[orow] = acc;
                    if (ep.x_out) ep.x_out[orow] = acc - ep.dot_minus[orow];
                }
            }
            continue;
        }
        float dot = 0.f;
        if (c > 0) {
            const float* n = a.Nst + ((size_t)bh * a.NC + c - 1) * D;
            const float* q = a.q + row * D;
            for (int k = 4 * lane; k < D; k += 256) {
                const f32x4 nv = *reinterpret_cast<const f32x4*>(n + k);
                const f32x4 qv = *reinterpret_cast<const f32x4*>(q + k);
                dot += nv[0] * qv[0] + nv[1] * qv[1] + nv[2] * qv[2] + nv[3] * qv[3];
            }
            dot = wave_reduce<OpAdd>(dot);
            dot *= fast_exp2(a.beta2[poff + GRAN * c - 1] - a.beta2[poff + t] +
                             (float)(a.G2[(size_t)bh * a.NC + c] - a.G2[(size_t)bh * a.NC + c - 1]));
        }
        const float prow = a.P[((size_t)bh * a.NC + c) * GRAN * GRAN + (size_t)(t - GRAN * c) * GRAN + lane];
        const float b = dot + wave_reduce<OpAdd>(prow);
        const float inv = 1.0f / (fmaxf(fabsf(b), __expf(-a.M[row])) + 1e-6f);
        if (a.Bout && lane == 0) a.Bout[row] = b;
#pragma unroll
        for (int n = 0; n < NB; n++) {
            const int k = 4 * lane + 256 * n;
            f32x4 x = num[n];
            if (a.finish_mode == 0) {
                const f32x4 ov = *reinterpret_cast<const f32x4*>(a.o + row * D + k);
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] *= inv;
                if (a.Hun) *reinterpret_cast<f32x4*>(a.Hun + row * D + k) = x;
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] = x[e] * (ov[e] / (1.0f + __expf(-ov[e])));
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] *= inv;
            }
            *reinterpret_cast<f32x4*>(a.h + row * D + k) = x;
        }
    }
}

template <int D, int VB, int NKB, bool REV, bool SHARED>
static void launch_state(const ScanArgs& a, hipStream_t st) {
    constexpr int lds_bytes = scan_state_lds<VB, NKB>(), wg_elems = SCAN_NW * NKB * VB * 16 * 64;
    // (a failure here shows up as a launch error, which the caller reads with hipGetLastError)
    (void)lds_limit_once<scan_state_kernel<D, VB, NKB, false, REV, SHARED>>(lds_bytes);
    const int wgs = a.BH * (D / (32 * VB)) * (D / (32 * NKB * SCAN_NW));
    if (a.nseg > 1) {
        (void)lds_limit_once<scan_state_kernel<D, VB, NKB, true, REV, false>>(lds_bytes);
        hipLaunchKernelGGL((scan_state_kernel<D, VB, NKB, true, REV, false>), dim3(wgs, a.nseg - 1), dim3(SCAN_NW * 64), lds_bytes, st, a);
        const size_t elems = (size_t)wgs * wg_elems;   // = BH * D * D
        hipLaunchKernelGGL(scan_segcarry_kernel, dim3((unsigned)((elems + 255) / 256)), dim3(256), 0, st, a, elems, wg_elems);
    }
    hipLaunchKernelGGL((scan_state_kernel<D, VB, NKB, false, REV, SHARED>), dim3(wgs, a.nseg), dim3(SCAN_NW * 64), lds_bytes, st, a);
}

template <int D, int VB, int NKB>
static void launch_state_r(const ScanArgs& a, hipStream_t st) {
    if constexpr (D / (32 * NKB * SCAN_NW) >= 2 && VB == 2) {
        if (a.shared) {
            if (a.rev) launch_state<D, VB, NKB, true, true>(a, st);
            else launch_state<D, VB, NKB, false, true>(a, st);
            return;
        }
    }
    if (a.rev) launch_state<D, VB, NKB, true, false>(a, st);
    else launch_state<D, VB, NKB, false, false>(a, st);
}

// Tile of a wave in blocks of 32: 64 value x 64 key columns while that gives every CU a workgroup, otherwise half of the key
// columns, otherwise half of the value columns too.
struct ScanTile { int vb, nkb; };
static ScanTile scan_tile(int BH, int D) {
    const int wgs = BH * (D / 64) * (D / 256);
    if (wgs >= 256) return {2, 2};
    if (2 * wgs >= 256) return {2, 1};
    return {1, 1};
}

template <int D>
static int launch_scan_d(const ScanArgs& a, int parts, hipStream_t st, void (*mark)(int, hipStream_t, bool)) {
    mark(MLSTM_K_SCAN_CARRY, st, true);
    const size_t zeros = a.shared ? (size_t)a.BH * a.S * D * parts : 0;
    hipLaunchKernelGGL(scan_intra_kernel<D>, dim3(a.BH * a.NC * 4 + (unsigned)((zeros + SCAN_ZERO_WG - 1) / SCAN_ZERO_WG)), dim3(256), 0, st, a, parts);
    if (a.finish_mode != 2 || a.ep.vec) hipLaunchKernelGGL(scan_ncarry_kernel, dim3((D + 255) / 256, a.BH), dim3(256), 0, st, a);
    mark(MLSTM_K_SCAN_CARRY, st, false);
    mark(MLSTM_K_SCAN_STATE, st, true);
    const ScanTile tile = scan_tile(a.BH, D);
    if (tile.nkb == 2) launch_state_r<D, 2, 2>(a, st);
    else if (tile.vb == 2) launch_state_r<D, 2, 1>(a, st);
    else launch_state_r<D, 1, 1>(a, st);
    mark(MLSTM_K_SCAN_STATE, st, false);
    mark(MLSTM_K_SCAN_OUT, st, true);
    const size_t rows = (size_t)a.BH * a.S;
    const int blocks = (int)((rows + 3) / 4 < 16384 ? (rows + 3) / 4 : 16384);
    hipLaunchKernelGGL(scan_finish_kernel<D>, dim3(blocks), dim3(256), 0, st, a, parts);
    mark(MLSTM_K_SCAN_OUT, st, false);
    return (int)hipGetLastError();
}

void launch_scan_ncarry(const ScanArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(scan_ncarry_kernel, dim3((a.D + 255) / 256, a.BH), dim3(256), 0, st, a);
}

// Key ranges per value tile.  A walk with 64 value columns per workgroup has twice the key ranges that one with 32 would have; pairs
// of them share a partial numerator, so that the workspace does not grow with them (in tensors beside the output: D = 1024 from 4
// heads on one instead of three, D = 512 from 16 heads on none instead of one).  It costs zeros and adds in place of stores, in us apart / shared
// with the zeros in a pass of their own (now 1 to 3 % less, see scan_zeros): forward 4 heads x 2048 x 1024 306 / 311, 2 x 2048 x 1024 210 / 224, 16 x 1024 x 512 172 / 178,
// 8 x 1024 x 512 118 / 129, 40 x 2048 x 256 456 / 474; forward + backward 2 x 2048 x 1024 868 / 905, 8 x 1024 x 512 482 / 521,
// 40 x 2048 x 256 1902 / 2001.
bool scan_can_share(int BH, int D) { return scan_tile(BH, D).vb == 2 && scan_key_splits(BH, D) >= 2; }
int scan_key_parts(int BH, int D, bool shared) { return shared ? scan_key_splits(BH, D) / 2 : scan_key_splits(BH, D); }
int scan_key_splits(int BH, int D) { return D / (32 * SCAN_NW * scan_tile(BH, D).nkb); }

// Segments of a sequence that run side by side: none while heads x value tiles x key ranges fill the chip; otherwise
// enough for about two workgroups per CU, of at least eight chunks each.
void scan_segments(int BH, int S, int D, int* nseg, int* seg_chunks) {
    const int NC = (S + GRAN - 1) / GRAN, wgs = BH * (D / (32 * scan_tile(BH, D).vb)) * scan_key_splits(BH, D);
    int n = 1;
    if (wgs < 256) {
        n = (512 + wgs - 1) / wgs;
        if (n > NC / 8) n = NC / 8;
        if (n < 1) n = 1;
    }
    const int len = (NC + n - 1) / n;
    *seg_chunks = len;
    *nseg = (NC + len - 1) / len;
}
size_t scan_segment_state_bytes(int BH, int S, int D) {
    int n, len; scan_segments(BH, S, D, &n, &len);
    return n > 1 ? (size_t)(n - 1) * BH * D * D * sizeof(float) : 0;
}

int launch_scan(const ScanArgs& a_in, int KS, hipStream_t st, void (*mark)(int, hipStream_t, bool)) {
    ScanArgs a = a_in;
    scan_segments(a.BH, a.S, a.D, &a.nseg, &a.seg_chunks);
    if (a.nseg > 1 && !a.seg_state) return MLSTM_EWORKSPACE;
    if (a.finish_mode != 2 && (a.rev || a.col_scale)) return MLSTM_EINVAL;
    if (a.finish_mode == 2 && ((a.ep.out_rev && (!a.ep.out || a.ep.out == a.h)) ||
                               (a.ep.dot_with && !a.ep.dot_out) || (a.ep.x_out && !(a.ep.dot_with && a.ep.dot_minus)) ||
                               (!a.ep.wd_alpha2 != !a.ep.wd_beta2)))
        return MLSTM_EINVAL;
    if ((a.D != 256 && a.D != 512 && a.D != 1024) || KS != scan_key_splits(a.BH, a.D)) return MLSTM_ESHAPE;
    if (a.shared && !scan_can_share(a.BH, a.D)) return MLSTM_EINVAL;
    const int parts = scan_key_parts(a.BH, a.D, a.shared != 0);
    switch (a.D) {
        case 256: return launch_scan_d<256>(a, parts, st, mark);
        case 512: return launch_scan_d<512>(a, parts, st, mark);
        case 1024: return launch_scan_d<1024>(a, parts, st, mark);
    }
    return MLSTM_ESHAPE;
}

}  // namespace mlstm
