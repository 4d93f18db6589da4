// Chunk states for the matmul form of long sequences.
//
// The forward of a row i only needs the keys of its own chunk of L positions one by one; everything before the chunk
// enters through the state the scan form carries (mlstm_scan.py:16-26; the two forms are the same function):
//     C~_c = sum_{j <= e_c} exp(a_j - A_{e_c}) k_j v_j^T / sqrt(D),     n~_c likewise with k_j alone,
// with e_c the last position of chunk c, a_j = i_j - Fc_j and A the running maximum of a (the gate pre-pass), so that
//     sum_{j <= e_c} C~_ij v_j = exp(A_{e_c} - A_i) q_i^T C~_c     for every row i behind the chunk (A_i >= A_{e_c}).
// The row kernel then walks the key tiles of the row's own chunk and D/64 "tiles" of the state instead of all the key
// tiles back to position 0: 2 L/64 + D/64 tiles at most, whatever the sequence length.
//
//   chunk_sum_kernel    per (head, chunk, 128 value columns): dC_c = sum_{j in chunk} w_j k_j v_j^T with
//                       w_j = exp(a_j - A_{e_c}) / sqrt(D), as a bf16 / fp16 MFMA product over the chunk's positions (both
//                       operands are contracted over positions: transposing LDS reads; V is scaled by w on its way
//                       into LDS), fp32 result; and dn_c = sum_j w_j k_j.  Eight waves: four multiply, four bring the tiles.
//   chunk_sum_narrow_kernel  the same sums, bit for bit, on 64 x 64 blocks, for few heads.
//   chunk_carry_kernel  C~_c = gamma_c C~_{c-1} + dC_c over the chunks of a head (gamma_c = exp(A_{e_{c-1}} - A_{e_c})),
//                       element-wise, written in the element type; n~_c likewise, in place, fp32.
//   chunk_seq_kernel    both in one pass, bit for bit, for launches that fill the chip.
//   chunk_sum_small_kernel, chunk_carry_small_kernel  the same two steps for fp32 and for 16-bit types at D = 64 (fp32 MFMA).
//   chunk_sum_terms_kernel  the chunk sums of bf16 at D = 64, outside split mode, with the weighted values as three bf16 terms.
// State rows are stored in the order in which the row kernel's second product contracts them (see PERM16 below).
#include "mlstm_device.h"
#include "mlstm_kernels.h"
#include <type_traits>
#include <utility>

namespace mlstm {

// The row kernel feeds the state tiles to its second product with the lanes' own row-major Q fragments as the other
// operand: the lane of half h holds columns 16 s + 8 h + e (e = 0..7) of step s, while the transposing read of the
// tile hands it rows 16 s + 4 h + e (e < 4) and 16 s + 8 + 4 h + e - 4 (e >= 4).  Tile row u (mod 16) therefore holds
// state row PERM16(u): the two middle groups of four swap places.
__device__ __forceinline__ int perm16(int u) { return (u & ~12) | ((u & 4) << 1) | ((u & 8) >> 1); }
__device__ __forceinline__ int state_row(int u) { return (u & ~15) | perm16(u & 15); }

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// What the chunk sums read for a position past the sequence's end: a piece of zeros.  (The sequence's last row in its place, with a weight of 0, would make
// every sum that an infinity or NaN of that row enters NaN; and how many such rows a kernel reads depends on its tiles.)
__device__ const u32x4 zero_piece = {0, 0, 0, 0};
// A piece of a row, if the row is there.  (Both addresses as global ones: constants have an address space of their own, and a choice between the two is a flat
// load, whose waits cost the sums 3 to 7 %; a variable that is no constant has its address fetched from memory.)
typedef const __attribute__((address_space(1))) u32x4* GlobalPiece;
__device__ __forceinline__ u32x4 piece_or_zeros(bool there, const void* piece) { return *(there ? (GlobalPiece)(size_t)piece : (GlobalPiece)(size_t)&zero_piece); }
template <typename T>
__device__ __forceinline__ T element_or_zero(bool there, const T* element) {
    typedef const __attribute__((address_space(1))) T* Global;
    return *(there ? (Global)(size_t)element : (Global)(size_t)&zero_piece);
}

// STRICT: split mode, the weighted V rows go to LDS as two tiles, hi and lo (ChunkArgs::precise)
template <typename T, int D, bool STRICT = false>
struct ChunkCfg {
    static constexpr int VW = 128;                                  // value columns per workgroup
    static constexpr int STAGES = 2;                                // LDS stages: the tile worked on and the next one
    static constexpr int RSETS = 3;                                 // register sets: tiles in flight from memory
    static constexpr size_t K_BYTES = (size_t)GRAN * D * sizeof(T), V_TILE = (size_t)GRAN * VW * sizeof(T);
    static constexpr size_t V_BYTES = (STRICT ? 2 : 1) * V_TILE;    // per stage: the hi tile, then the lo tile
    static constexpr size_t TILE_BYTES = STAGES * (K_BYTES + V_BYTES);   // plus one float per position of the chunk
    static constexpr int MAX_L = (int)((160 * 1024 - TILE_BYTES) / (2 * sizeof(float))) / 128 * 128;
};

// Eight 16-bit elements (four dwords) as floats.  bf16 by hand: one shift or mask per element (the generic vector
// conversion costs several instructions per element, in a kernel that is bound by instruction issue).
template <typename T>
__device__ __forceinline__ void unpack8(const u32x4& d, float (&x)[8]) {
    if constexpr (std::is_same<T, __bf16>::value) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            x[2 * i] = __builtin_bit_cast(float, d[i] << 16);
            x[2 * i + 1] = __builtin_bit_cast(float, d[i] & 0xffff0000u);
        }
    } else {
        typedef _Float16 h8 __attribute__((ext_vector_type(8)));
        const h8 v = __builtin_bit_cast(h8, d);
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = (float)v[e];
    }
}

// NTT: tiles per chunk as a compile-time constant (the tile loop is then straight-line code), or 0 for any chunk length
template <typename T, int D, int NTT, bool STRICT>
__global__ __launch_bounds__(512) void chunk_sum_kernel(ChunkArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    using R = Tr<T>;
    using Cfg = ChunkCfg<T, D, STRICT>;
    typedef typename R::frag frag;
    static_assert(R::HALF && (D == 128 || D == 256), "16-bit types, D = 128 or 256");
    constexpr int VW = Cfg::VW, VH = D / VW, MB = D / 128, NB = VW / 32, KW = R::KW, ST = Cfg::STAGES;
    using ZK = Swz<T, D>;
    using ZV = Swz<T, VW>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    char* const ks = smem;
    char* const vs = smem + ST * Cfg::K_BYTES;
    float* const sw = reinterpret_cast<float*>(smem + Cfg::TILE_BYTES);   // [L] position weights of the matrix sum
    float* const sw2 = sw + a.L;                                           // [L] ... of the vector sum

    // Eight waves, two on every SIMD.  Waves 0..3 multiply: operand reads and MFMAs, nothing else.  Waves 4..7 feed them: they
    // load the tiles, scale V, write the LDS stages and add up the vector state from the K pieces they hold anyway.  With
    // four waves doing both in turn the kernel was bound by instruction issue (about 430 other instructions per tile next to
    // 1024 cycles of MFMAs, on a SIMD with nothing else to run); the two kinds of work now overlap.
    const bool feeder = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) != 0;
    const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6, h = lane >> 5, c32 = lane & 31;
    // Workgroups go round-robin to the 8 XCDs, each with an L2 of its own: the VH workgroups of a (head, chunk), which read
    // the same K, sit 8 apart in the launch order, on one XCD
    int vh, pair;
    if (VH == 2 && (gridDim.x & 15) == 0) { vh = (blockIdx.x >> 3) & 1; pair = (blockIdx.x & 7) | ((blockIdx.x >> 4) << 3); }
    else { vh = blockIdx.x % VH; pair = blockIdx.x / VH; }
    const int cc = pair % a.NCS, bh = pair / a.NCS;
    const int S = a.S, L = a.L, NT = NTT ? NTT : L / GRAN;
    const size_t hoff = (size_t)bh * S, poff = (size_t)bh * a.NG * GRAN, goff = (size_t)bh * a.NG;
    // forward states: sum cc is over chunk cc, relative to its own last position; reverse states (K = Q, V = dH): sum cc
    // is over chunk cc + 1 (the last chunk may be short), relative to the last position of chunk cc
    const int p0 = (a.reverse ? cc + 1 : cc) * L, pe = a.reverse ? p0 - 1 : p0 + L - 1;
    // K and V are the caller's tensors, each in its layout (elements per position rsK / rsV)
    const size_t rsK = (size_t)a.lk.ss, rsV = (size_t)a.lv.ss;
    const T* Kh = reinterpret_cast<const T*>(a.K) + a.lk.head(bh) + (size_t)p0 * rsK;
    const T* Vh = reinterpret_cast<const T*>(a.V) + a.lv.head(bh) + (size_t)p0 * rsV + VW * vh;

    // vector state: a feeder thread's K pieces of a tile are rows pg + NPG it (it < KP) of the eight keys 8 kc .. 8 kc + 7
    const int kc = tid & (D / 8 - 1), pg = tid / (D / 8);
    constexpr int NPG = 256 / (D / 8);

    // The two kinds of waves run code of their own from here on (every value of one kind is dead in the other: the registers
    // of a wave hold either the accumulators or the tiles in flight); both pass the same barriers.
    auto feed = [&]() __attribute__((always_inline)) {
    f32x8 nacc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // Tiles travel memory -> registers -> LDS.  A thread's pieces of a tile: KP 16-byte pieces of K (piece tid + 256 it of
    // the tile's rows of CPR pieces) and four of V (rows tid/16 + 16 it, piece tid%16); tile j uses register set j % 3 and
    // LDS stage j % 2.  Rows past the end of the sequence are zeros.
    constexpr int KP = GRAN * ZK::CPR / 256, LPT = KP + 4;   // loads per thread and tile
    const int vrow = tid >> 4, vch = tid & 15;
    u32x4 kset[Cfg::RSETS][KP], vset[Cfg::RSETS][4];
    // A thread's pieces lie a fixed number of rows apart (K: 256 / CPR, V: 16): one per-lane element offset each, everything
    // else of an address is the same for all lanes.  Only the tiles of a short last chunk need a look at each row.
    constexpr int KROWS = 256 / ZK::CPR;
    const unsigned koff = (unsigned)((tid / ZK::CPR) * rsK + 8 * (tid % ZK::CPR)), voff = (unsigned)(vrow * rsV + 8 * vch);
    auto issue = [&](auto set_tag, int j) __attribute__((always_inline)) {
        constexpr int P = decltype(set_tag)::value;
        if (__builtin_expect(p0 + GRAN * (j + 1) <= S, 1)) {
            const T* kt = Kh + (size_t)GRAN * j * rsK;
            const T* vt = Vh + (size_t)GRAN * j * rsV;
#pragma unroll
            for (int it = 0; it < KP; it++) kset[P][it] = *reinterpret_cast<const u32x4*>(kt + (size_t)(KROWS * it) * rsK + koff);
#pragma unroll
            for (int it = 0; it < 4; it++) vset[P][it] = *reinterpret_cast<const u32x4*>(vt + (size_t)(16 * it) * rsV + voff);
        } else {
#pragma unroll
            for (int it = 0; it < KP; it++) {
                const int pc = tid + 256 * it, pos = GRAN * j + pc / ZK::CPR;
                kset[P][it] = piece_or_zeros(p0 + pos < S, Kh + (size_t)pos * rsK + 8 * (pc % ZK::CPR));
            }
#pragma unroll
            for (int it = 0; it < 4; it++) {
                const int pos = GRAN * j + vrow + 16 * it;
                vset[P][it] = piece_or_zeros(p0 + pos < S, Vh + (size_t)pos * rsV + 8 * vch);
            }
        }
        __builtin_amdgcn_sched_barrier(0);   // the loads go out here, not where the scheduler would like them
    };
    // K of tile j as it is, V times the positions' weights, into stage j % 2
    auto commit = [&](auto set_tag, int j) __attribute__((always_inline)) {
        constexpr int P = decltype(set_tag)::value;
        typedef typename R::vec4 V4;
        struct Pair { V4 lo, hi; };
#pragma unroll
        for (int it = 0; it < KP; it++) {
            const int pc = tid + 256 * it;
            *reinterpret_cast<u32x4*>(ks + (j % ST) * Cfg::K_BYTES + ZK::off(pc / ZK::CPR, 8 * (pc % ZK::CPR))) = kset[P][it];
            if (vh == 0) {   // the vector state's share of this piece
                float x[8];
                unpack8<T>(kset[P][it], x);
                const float w2 = sw2[GRAN * j + pc / ZK::CPR];
#pragma unroll
                for (int e = 0; e < 8; e++) nacc[e] = fmaf(x[e], w2, nacc[e]);
            }
        }
#pragma unroll
        for (int it = 0; it < 4; it++) {
            const int row = vrow + 16 * it;
            const float w = sw[GRAN * j + row];
            float x[8];
            unpack8<T>(vset[P][it], x);
            Pair out;
            if constexpr (STRICT) {   // the weighted row as two terms: what rounding to the element type loses goes to the lo tile
                Pair rest;
                R::cvt4_split(f32x4{x[0] * w, x[1] * w, x[2] * w, x[3] * w}, out.lo, rest.lo);
                R::cvt4_split(f32x4{x[4] * w, x[5] * w, x[6] * w, x[7] * w}, out.hi, rest.hi);
                *reinterpret_cast<Pair*>(vs + (j % ST) * Cfg::V_BYTES + Cfg::V_TILE + ZV::off(row, 8 * vch)) = rest;
            } else {
                out.lo = R::cvt4(f32x4{x[0] * w, x[1] * w, x[2] * w, x[3] * w});
                out.hi = R::cvt4(f32x4{x[4] * w, x[5] * w, x[6] * w, x[7] * w});
            }
            *reinterpret_cast<Pair*>(vs + (j % ST) * Cfg::V_BYTES + ZV::off(row, 8 * vch)) = out;
        }
    };
    // Iteration t, feeders (register set P = t % 3): the loads of tile t + 3 go out into the registers tile t left in the previous
    // iteration; tile t + 1 moves to the LDS stage that tile t - 1 left behind the last barrier.  The others multiply tile t.
    // Two to three tiles are in flight while a tile is worked on.  The loads are ordinary ones, so that the compiler places the counted
    // waits itself; it counts exactly in straight-line code (hence NTT: the default chunk's eight iterations are unrolled)
    // and falls back to waiting for everything across a loop's back edge.  Loads issued by hand -- direct-to-LDS copies of
    // K, or register loads from inline assembly -- gave wrong states now and then at full size as soon as a wait was a
    // counted one: the compiler moves or stashes a register it believes written while the load is still in flight.  With
    // one tile in flight and a wait for everything the kernel waited for memory latency in every iteration.
    auto iteration = [&](auto set_tag, int t) __attribute__((always_inline)) {
        constexpr int P = decltype(set_tag)::value, P1 = (P + 1) % 3;
        if (t + 3 < NT) issue(std::integral_constant<int, P>{}, t + 3);
        if (t + 1 < NT) commit(std::integral_constant<int, P1>{}, t + 1);
        __syncthreads();
    };

    // The positions' weights.  Forward: w_j = exp(a_j - A_e) / sqrt(D) for both sums, e the chunk's last position.
    // Reverse: rho_i = exp(A_e - A_i) / sqrt(D), e the last position BEFORE the chunk, times 1/n_i (matrix sum) or db_i
    // (vector sum), the per-row scalars of the dQ pass.
    const float log2scale = -0.5f * __log2f((float)D);
    if constexpr (NTT > 0) {
        // Their inputs are requested first and used behind the first tile's loads: the waits the compiler places for them
        // then count the tile loads as "behind" and do not wait for those (requested after the tiles, the weights waited
        // for all three tiles: 13 k cycles before the first iteration, measured).  The other two tiles' loads follow one
        // by one, so that the first tile's data is not queued behind theirs.
        {
            constexpr int WPT = NTT * GRAN / 256;   // positions per thread
            float x0[WPT], x1[WPT], x2[WPT];
            double xg[WPT];
            const float bend = a.beta2[poff + pe];
            const double Gend = a.G2[goff + pe / GRAN];
#pragma unroll
            for (int n = 0; n < WPT; n++) {
                int pos = p0 + tid + 256 * n;
                pos = pos < S ? pos : S - 1;
                xg[n] = a.G2[goff + pos / GRAN];
                if (a.reverse) { x0[n] = a.beta2[poff + pos]; x1[n] = a.inv_n[poff + pos]; x2[n] = a.db[poff + pos]; }
                else { x0[n] = a.alpha2[poff + pos]; x1[n] = 0.f; x2[n] = 0.f; }
            }
            __builtin_amdgcn_sched_barrier(0);
            issue(std::integral_constant<int, 0>{}, 0);
#pragma unroll
            for (int n = 0; n < WPT; n++) {
                const int p = tid + 256 * n;
                float w = 0.f, w2 = 0.f;
                if (p0 + p < S) {
                    if (a.reverse) {
                        const float rho = fast_exp2(bend - x0[n] + (float)(xg[n] - Gend) + log2scale);
                        w = rho * x1[n];
                        w2 = rho * x2[n];
                    } else {
                        w = w2 = fast_exp2(x0[n] - bend + (float)(Gend - xg[n]) + log2scale);
                    }
                }
                sw[p] = w;
                sw2[p] = w2;
            }
            __builtin_amdgcn_sched_barrier(0);
            issue(std::integral_constant<int, 1>{}, 1);   // (NT >= 2: a chunk is a multiple of 128 positions)
        }
        __syncthreads();   // the weights are in LDS
        commit(std::integral_constant<int, 0>{}, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (2 < NT) issue(std::integral_constant<int, 2>{}, 2);
        __syncthreads();
    } else {
        {
            issue(std::integral_constant<int, 0>{}, 0);
            issue(std::integral_constant<int, 1>{}, 1);
            if (2 < NT) issue(std::integral_constant<int, 2>{}, 2);
            const float bend = a.beta2[poff + pe];
            const double Gend = a.G2[goff + pe / GRAN];
            for (int p = tid; p < L; p += 256) {
                const int pos = p0 + p;
                float w = 0.f, w2 = 0.f;
                if (pos < S) {
                    if (a.reverse) {
                        const float rho = fast_exp2(bend - a.beta2[poff + pos] + (float)(a.G2[goff + pos / GRAN] - Gend) + log2scale);
                        w = rho * a.inv_n[poff + pos];
                        w2 = rho * a.db[poff + pos];
                    } else {
                        w = w2 = fast_exp2(a.alpha2[poff + pos] - bend + (float)(Gend - a.G2[goff + pos / GRAN]) + log2scale);
                    }
                }
                sw[p] = w;
                sw2[p] = w2;
            }
        }
        __syncthreads();   // the weights are in LDS
        commit(std::integral_constant<int, 0>{}, 0);
        __syncthreads();
    }
    if constexpr (NTT > 0) {
        static_for<NTT>([&](auto tt) __attribute__((always_inline)) { iteration(std::integral_constant<int, decltype(tt)::value % 3>{}, decltype(tt)::value); });
    } else {
        for (int t = 0; t < NT; t += 3) {
            iteration(std::integral_constant<int, 0>{}, t);
            if (t + 1 < NT) iteration(std::integral_constant<int, 1>{}, t + 1);
            if (t + 2 < NT) iteration(std::integral_constant<int, 2>{}, t + 2);
        }
    }
    if (vh == 0) {   // the partial sums (one per group of rows) meet in LDS (the tiles are done with: the last barrier)
        float* red = reinterpret_cast<float*>(smem);   // [NPG][D]
        *reinterpret_cast<f32x8*>(red + pg * D + 8 * kc) = nacc;
        __syncthreads();
        if (tid < D) {
            float sum = 0.f;
#pragma unroll
            for (int g = 0; g < NPG; g++) sum += red[g * D + tid];
            a.Nst[((size_t)bh * a.NCS + cc) * D + tid] = sum;
        }
    }
    };

    auto multiply = [&]() __attribute__((always_inline)) {
    SwzTransReader<T, D> krd;        // per-lane offsets of the transposing reads, computed once
    krd.init(lane, (D / 128) * wave);
    SwzTransReader<T, VW> vrd;
    vrd.init(lane, 0);
    f32x16 acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
            for (int x = 0; x < 16; x++) acc[mb][nb][x] = 0.f;
    auto compute = [&](int t) __attribute__((always_inline)) {
        const T* kt = reinterpret_cast<const T*>(ks + (t % ST) * Cfg::K_BYTES);
        const T* vt = reinterpret_cast<const T*>(vs + (t % ST) * Cfg::V_BYTES);
        // the operand reads of a contraction step run one step ahead of its MFMAs (read, wait, multiply in turns left the
        // matrix unit idle for an LDS round trip per step: 3000 cycles per tile for 1024 of MFMAs, measured)
        constexpr int NSTEP = GRAN / KW;
        frag af[2][MB], bf[2][NB], bl[STRICT ? NB : 1];
        const T* vl = reinterpret_cast<const T*>(vs + (t % ST) * Cfg::V_BYTES + Cfg::V_TILE);   // (split mode: the lo tile)
        auto rd = [&](int s) __attribute__((always_inline)) {
#pragma unroll
            for (int mb = 0; mb < MB; mb++) af[s & 1][mb] = krd.read(kt, KW * s, mb);
#pragma unroll
            for (int nb = 0; nb < NB; nb++) bf[s & 1][nb] = vrd.read(vt, KW * s, nb);
        };
        rd(0);
#pragma unroll
        for (int s = 0; s < NSTEP; s++) {
            // (split mode: the lo fragments of this step are single-buffered -- a second set does not fit the registers at
            // D = 256 -- and requested here, behind the MFMAs on the hi fragments)
            if constexpr (STRICT) {
#pragma unroll
                for (int nb = 0; nb < NB; nb++) bl[nb] = vrd.read(vl, KW * s, nb);
            }
            if (s + 1 < NSTEP) rd(s + 1);
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int nb = 0; nb < NB; nb++) R::mma(acc[mb][nb], af[s & 1][mb], bf[s & 1][nb]);
            if constexpr (STRICT) {
#pragma unroll
                for (int mb = 0; mb < MB; mb++)
#pragma unroll
                    for (int nb = 0; nb < NB; nb++) R::mma(acc[mb][nb], af[s & 1][mb], bl[nb]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    __syncthreads();   // (the weights are in LDS)
    __syncthreads();   // (the first tile is)
    if constexpr (NTT > 0) {
        static_for<NTT>([&](auto tt) __attribute__((always_inline)) { compute(decltype(tt)::value); __syncthreads(); });
    } else {
        for (int t = 0; t < NT; t++) { compute(t); __syncthreads(); }
    }
    // accumulator block (mb, nb): column (value) 32 nb + c32, rows (keys) 8 (r / 4) + 4 h + r % 4
    float* out = a.dC + ((size_t)bh * a.NCS + cc) * D * D + VW * vh;
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int k = (D / 4) * wave + 32 * mb + 8 * (r >> 2) + 4 * h + (r & 3);
                out[(size_t)k * D + 32 * nb + c32] = acc[mb][nb][r];
            }
    if (vh == 0) __syncthreads();   // (the feeders' sum of the vector state)
    };

    if (feeder) feed();
    else multiply();
#endif
}

// The chunk sums of chunk_sum_kernel -- the same products in the same order, hence the same bits -- where few workgroups would run:
// one workgroup per (head, chunk, 64 keys, 64 values), a wave per 32 x 32 block.  With 48 workgroups that kernel takes as long as its
// eight tiles one after the other (D = 256 17 us, split mode 24, D = 128 12, whatever the number of heads); here a workgroup's
// 64 columns of K and V are 64 KB each, V's requested at once, K's in two parts, and two trips to memory, 32 products and the
// write-out remain: 8 to 10 us.  K and V are read D / 64 times over, which is what the larger workgroups save where there are enough of them.
template <typename T, bool STRICT>
struct ChunkNarrowCfg {
    static constexpr int L = 512, W = 64, PART = 256;               // positions per chunk, columns per workgroup, positions per part
    static constexpr size_t PART_BYTES = (size_t)PART * W * sizeof(T);
    // One part of K and V at a time, so that two workgroups fit a CU (both at once: level up to 256 workgroups, 15.4 us instead of
    // 11.9 at 384).  Split mode: V's part as hi and lo, next to all of K.  And the positions' weights of the two sums.
    static constexpr int KPARTS = STRICT ? 2 : 1, VPARTS = STRICT ? 2 : 1;
    static constexpr size_t LDS_BYTES = (KPARTS + VPARTS) * PART_BYTES + 2 * L * sizeof(float);
};
template <typename T, int D, bool STRICT>
__global__ __launch_bounds__(256) void chunk_sum_narrow_kernel(ChunkArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    using R = Tr<T>;
    using Cfg = ChunkNarrowCfg<T, STRICT>;
    using Z = Swz<T, Cfg::W>;
    typedef typename R::frag frag;
    constexpr int L = Cfg::L, W = Cfg::W, PART = Cfg::PART, KW = R::KW, NBK = (D / W) * (D / W);
    extern __shared__ __attribute__((aligned(16))) char smem[];
    auto kpart = [&](int p) { return smem + (STRICT ? p : 0) * Cfg::PART_BYTES; };
    char* const vt = smem + Cfg::KPARTS * Cfg::PART_BYTES;   // (split mode: the lo tile behind it)
    float* const sw = reinterpret_cast<float*>(smem + (Cfg::KPARTS + Cfg::VPARTS) * Cfg::PART_BYTES);
    float* const sw2 = sw + L;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, c32 = lane & 31;
    int pair, blk;   // (head, chunk) and block of its sum: with a multiple of 8 pairs a pair's workgroups run on one XCD
    if (((a.BH * a.NCS) & 7) == 0) { pair = (blockIdx.x & 7) | ((blockIdx.x >> 3) / NBK << 3); blk = (blockIdx.x >> 3) % NBK; }
    else { pair = blockIdx.x / NBK; blk = blockIdx.x % NBK; }
    const int cc = pair % a.NCS, bh = pair / a.NCS, kcol = W * (blk / (D / W)), vcol = W * (blk % (D / W));
    const int S = a.S;
    const size_t poff = (size_t)bh * a.NG * GRAN, goff = (size_t)bh * a.NG;
    const int p0 = (a.reverse ? cc + 1 : cc) * L, pe = a.reverse ? p0 - 1 : p0 + L - 1;   // (see chunk_sum_kernel)
    const size_t rsK = (size_t)a.lk.ss, rsV = (size_t)a.lv.ss;
    const T* Kh = reinterpret_cast<const T*>(a.K) + a.lk.head(bh) + (size_t)p0 * rsK + kcol;
    const T* Vh = reinterpret_cast<const T*>(a.V) + a.lv.head(bh) + (size_t)p0 * rsV + vcol;

    // what the weights need, then K straight into LDS and V into registers, all positions at once
    float x0[2], x1[2] = {0.f, 0.f}, x2[2] = {0.f, 0.f};
    double xg[2];
    const float bend = a.beta2[poff + pe];
    const double Gend = a.G2[goff + pe / GRAN];
#pragma unroll
    for (int n = 0; n < 2; n++) {
        const int pos = p0 + tid + 256 * n < S ? p0 + tid + 256 * n : S - 1;
        xg[n] = a.G2[goff + pos / GRAN];
        x0[n] = a.reverse ? a.beta2[poff + pos] : a.alpha2[poff + pos];
        if (a.reverse) { x1[n] = a.inv_n[poff + pos]; x2[n] = a.db[poff + pos]; }
    }
    constexpr int NP = 2 * PART * Z::CPR / 256;   // a thread's 16-byte pieces of V: row vrow + 32 i, piece vch
    const int vrow = tid / Z::CPR, vch = tid % Z::CPR;
    u32x4 vset[NP];
    const bool whole = p0 + L <= S;
    auto request_v = [&](auto whole_tag) __attribute__((always_inline)) {   // (rows past the end are zeros)
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int r = vrow + 32 * i;
            vset[i] = piece_or_zeros(decltype(whole_tag)::value || p0 + r < S, Vh + (size_t)r * rsV + Z::EPC * vch);
        }
    };
    if (whole) request_v(std::true_type{});
    else request_v(std::false_type{});
    // K: 1 KB (eight rows) per load of a wave; piece c of row r at piece c ^ key(r) of the row
    auto copy_k = [&](int p) __attribute__((always_inline)) {
        const unsigned kbase = lds_offset_of(kpart(p));
        const int kr = lane / Z::CPR, kc = lane % Z::CPR;
        auto rows = [&](auto whole_tag) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < PART / 32; i++) {
                const int r = 32 * i + 8 * wave;
                const T* piece = Kh + (size_t)(PART * p + r + kr) * rsK + Z::EPC * (kc ^ Z::key(r + kr));
                if (!decltype(whole_tag)::value && p0 + PART * p + r + kr >= S) piece = reinterpret_cast<const T*>(&zero_piece);
                dma16(piece, __builtin_amdgcn_readfirstlane(kbase + r * Z::ROW_BYTES));
            }
        };
        if (whole) rows(std::true_type{});
        else rows(std::false_type{});
    };
    copy_k(0);
    if constexpr (STRICT) copy_k(1);
    const float log2scale = -0.5f * __log2f((float)D);
#pragma unroll
    for (int n = 0; n < 2; n++) {
        float w = 0.f, w2 = 0.f;
        if (p0 + tid + 256 * n < S) {
            if (a.reverse) {
                const float rho = fast_exp2(bend - x0[n] + (float)(xg[n] - Gend) + log2scale);
                w = rho * x1[n];
                w2 = rho * x2[n];
            } else {
                w = w2 = fast_exp2(x0[n] - bend + (float)(Gend - xg[n]) + log2scale);
            }
        }
        sw[tid + 256 * n] = w;
        sw2[tid + 256 * n] = w2;
    }
    __syncthreads();   // the weights are there
    auto commit = [&](auto part_tag) __attribute__((always_inline)) {   // V times the weights, rounded
        constexpr int P = decltype(part_tag)::value;
        typedef typename R::vec4 V4;
        struct Pair { V4 lo, hi; };
#pragma unroll
        for (int i = 0; i < NP / 2; i++) {
            const int row = vrow + 32 * i;
            const float w = sw[PART * P + row];
            float x[8];
            unpack8<T>(vset[P * (NP / 2) + i], x);
            Pair out;
            if constexpr (STRICT) {
                Pair rest;
                R::cvt4_split(f32x4{x[0] * w, x[1] * w, x[2] * w, x[3] * w}, out.lo, rest.lo);
                R::cvt4_split(f32x4{x[4] * w, x[5] * w, x[6] * w, x[7] * w}, out.hi, rest.hi);
                *reinterpret_cast<Pair*>(vt + Cfg::PART_BYTES + Z::off(row, Z::EPC * vch)) = rest;
            } else {
                out.lo = R::cvt4(f32x4{x[0] * w, x[1] * w, x[2] * w, x[3] * w});
                out.hi = R::cvt4(f32x4{x[4] * w, x[5] * w, x[6] * w, x[7] * w});
            }
            *reinterpret_cast<Pair*>(vt + Z::off(row, Z::EPC * vch)) = out;
        }
    };
    // per-lane offsets of the transposing reads (see frag_transposed): rows 16 apart meet the same swizzle
    const int kb = wave & 1, vb = wave >> 1;
    const int j16 = lane & 15, sub = (lane >> 4) & 1, trow = 4 * h + (j16 >> 2), tcol = 16 * sub + 4 * (j16 & 3);
    const int ko0 = Z::off(trow, 32 * kb + tcol), ko1 = Z::off(trow + 8, 32 * kb + tcol);
    const int vo0 = Z::off(trow, 32 * vb + tcol), vo1 = Z::off(trow + 8, 32 * vb + tcol);
    auto read = [&](const char* tile, int o0, int o1) __attribute__((always_inline)) {
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(tile + o0));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(tile + o1));
        return __builtin_bit_cast(frag, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    f32x16 acc;
#pragma unroll
    for (int x = 0; x < 16; x++) acc[x] = 0.f;
    auto compute = [&](int p) __attribute__((always_inline)) {
        constexpr int NSTEP = PART / KW, AHEAD = 4;
        const char* kt = kpart(p);
        frag af[NSTEP], bf[NSTEP], bl[STRICT ? NSTEP : 1];
        auto rd = [&](int n) __attribute__((always_inline)) {
            const int at = KW * n * Z::ROW_BYTES;
            af[n] = read(kt + at, ko0, ko1);
            bf[n] = read(vt + at, vo0, vo1);
            if constexpr (STRICT) bl[n] = read(vt + Cfg::PART_BYTES + at, vo0, vo1);
        };
#pragma unroll
        for (int n = 0; n < AHEAD; n++) rd(n);
#pragma unroll
        for (int n = 0; n < NSTEP; n++) {
            if (n + AHEAD < NSTEP) rd(n + AHEAD);
            R::mma(acc, af[n], bf[n]);
            if constexpr (STRICT) R::mma(acc, af[n], bl[n]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // the vector state of the workgroup's keys (the workgroups of the first values), added up as the feeders of chunk_sum_kernel do:
    // position modulo NPG, then over those sums; a thread takes two keys of a row
    constexpr int NPG = 256 / (D / 8), NH = NPG / 8;
    float n0[NH], n1[NH];
    const int k2 = tid & 31, pg = tid >> 5;
#pragma unroll
    for (int u = 0; u < NH; u++) { n0[u] = 0.f; n1[u] = 0.f; }
    auto vector_part = [&](int p) __attribute__((always_inline)) {
        if (vcol != 0) return;
#pragma unroll
        for (int u = 0; u < NH; u++)
#pragma unroll 8
            for (int r = pg + 8 * u; r < PART; r += NPG) {
                typedef T T2 __attribute__((ext_vector_type(2)));
                const T2 kv = *reinterpret_cast<const T2*>(kpart(p) + Z::off(r, 2 * k2));
                const float w2 = sw2[PART * p + r];
                n0[u] = fmaf((float)kv[0], w2, n0[u]);
                n1[u] = fmaf((float)kv[1], w2, n1[u]);
            }
    };
    commit(std::integral_constant<int, 0>{});
    dma_wait();
    __syncthreads();
    compute(0);
    vector_part(0);
    __syncthreads();
    if constexpr (!STRICT) copy_k(1);
    commit(std::integral_constant<int, 1>{});
    dma_wait();
    __syncthreads();
    compute(1);
    vector_part(1);
    float* out = a.dC + ((size_t)bh * a.NCS + cc) * D * D + (size_t)(kcol + 32 * kb) * D + vcol + 32 * vb + c32;
#pragma unroll
    for (int r = 0; r < 16; r++) out[(size_t)(8 * (r >> 2) + 4 * h + (r & 3)) * D] = acc[r];
    if (vcol == 0) {
        float* const red = reinterpret_cast<float*>(vt);   // [NPG][W]
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NH; u++) *reinterpret_cast<float2*>(red + (pg + 8 * u) * W + 2 * k2) = make_float2(n0[u], n1[u]);
        __syncthreads();
        if (tid < W) {
            float sum = 0.f;
#pragma unroll
            for (int g = 0; g < NPG; g++) sum += red[g * W + tid];
            a.Nst[((size_t)bh * a.NCS + cc) * D + kcol + tid] = sum;
        }
    }
#endif
}

// The chunk sums of bf16 at D = 64: chunk_sum_small_kernel forms them in fp32 products; here each weighted value, w_j v_j in fp32, is three bf16 terms (24
// bits, as in Tr<float>) and a key is one, so that three bf16 products do at 96 cycles per 32 x 32 x 16 block what the fp32 ones do at 512.  One
// workgroup per (head, chunk) forms the whole 64 x 64 block, a 32 x 32 one per wave: all of a chunk of 256 positions is requested at once in whole lines, 16 bytes
// a lane (that kernel: two bytes, and every row twice), and passes through LDS in parts of 64 (of 128, two workgroups per CU and not three: 38.6 us for 35.6).
// A block that is not finite is formed again in fp32 multiply-adds (see not_finite).  Split mode and fp16, whose keys would be two terms and
// whose sums are relied upon bit by bit, stay on fp32 products.
// us, fp32 products / here, forward and reverse sums together: 64 heads x 8192 160 / 75 (K and V take 26 each way at the rate of a copy), 8 x 4096 18.2 / 17.5, 1 x 1100
// 17.0 / 16.0; training step of 64 x 8192 642 / 565.  Errors against 64 bits (h and all gradients, 1100 and 1500 positions) 0.998 to
// 1.001 of those before.
struct ChunkTermsCfg {
    static constexpr int L = 256, W = 64, PART = 64;
    static constexpr size_t TILE_BYTES = (size_t)PART * W * 2, LDS_BYTES = 4 * TILE_BYTES + 2 * L * sizeof(float);
};
__global__ __launch_bounds__(256) void chunk_sum_terms_kernel(ChunkArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __bf16 T;
    using R = Tr<T>;
    using Cfg = ChunkTermsCfg;
    using Z = Swz<T, Cfg::W>;
    typedef typename R::frag frag;
    typedef typename R::vec4 V4;
    struct Pair { V4 lo, hi; };
    constexpr int L = Cfg::L, W = Cfg::W, PART = Cfg::PART, KW = R::KW, D = 64, NP = PART * Z::CPR / 256, ROWS = 256 / Z::CPR;   // pieces per thread and part, rows of 256 threads
    extern __shared__ __attribute__((aligned(16))) char smem[];
    char* const kt = smem;
    auto vt = [&](int term) { return smem + (1 + term) * Cfg::TILE_BYTES; };
    float* const sw = reinterpret_cast<float*>(smem + 4 * Cfg::TILE_BYTES);
    float* const sw2 = sw + L;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, c32 = lane & 31;
    const int cc = blockIdx.x % a.NCS, bh = blockIdx.x / a.NCS, S = a.S;
    const size_t poff = (size_t)bh * a.NG * GRAN, goff = (size_t)bh * a.NG;
    const int p0 = (a.reverse ? cc + 1 : cc) * L, pe = a.reverse ? p0 - 1 : p0 + L - 1;   // (see chunk_sum_kernel)
    const size_t rsK = (size_t)a.lk.ss, rsV = (size_t)a.lv.ss;
    const T* const Kh = reinterpret_cast<const T*>(a.K) + a.lk.head(bh) + (size_t)p0 * rsK;
    const T* const Vh = reinterpret_cast<const T*>(a.V) + a.lv.head(bh) + (size_t)p0 * rsV;

    // what the weight of position tid needs, then all of the chunk
    const int pos = p0 + tid < S ? p0 + tid : S - 1;
    const float bend = a.beta2[poff + pe];
    const double Gend = a.G2[goff + pe / GRAN], xg = a.G2[goff + pos / GRAN];
    const float x0 = a.reverse ? a.beta2[poff + pos] : a.alpha2[poff + pos];
    const float x1 = a.reverse ? a.inv_n[poff + pos] : 0.f, x2 = a.reverse ? a.db[poff + pos] : 0.f;
    const int vrow = tid / Z::CPR, vch = tid % Z::CPR;   // a thread's 16-byte pieces: row vrow + ROWS i, piece vch
    const bool whole = p0 + L <= S;
    u32x4 kset[L / PART][NP], vset[L / PART][NP];
#pragma unroll
    for (int p = 0; p < L / PART; p++)
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int r = PART * p + vrow + ROWS * i, rr = whole || p0 + r < S ? r : S - 1 - p0;   // (past the end: the last row, whose place takes zeros below)
            kset[p][i] = *reinterpret_cast<const u32x4*>(Kh + (size_t)rr * rsK + Z::EPC * vch);
            vset[p][i] = *reinterpret_cast<const u32x4*>(Vh + (size_t)rr * rsV + Z::EPC * vch);
        }
    {
        const float log2scale = -0.5f * __log2f((float)D);
        float w = 0.f, w2 = 0.f;
        if (p0 + tid < S) {
            if (a.reverse) {
                const float rho = fast_exp2(bend - x0 + (float)(xg - Gend) + log2scale);
                w = rho * x1;
                w2 = rho * x2;
            } else {
                w = w2 = fast_exp2(x0 - bend + (float)(Gend - xg) + log2scale);
            }
        }
        sw[tid] = w;
        sw2[tid] = w2;
    }
    // per-lane offsets of the transposing reads (see frag_transposed): rows 16 apart meet the same swizzle
    const int kb = wave & 1, vb = wave >> 1;
    const int j16 = lane & 15, sub = (lane >> 4) & 1, trow = 4 * h + (j16 >> 2), tcol = 16 * sub + 4 * (j16 & 3);
    const int ko0 = Z::off(trow, 32 * kb + tcol), ko1 = Z::off(trow + 8, 32 * kb + tcol);
    const int vo0 = Z::off(trow, 32 * vb + tcol), vo1 = Z::off(trow + 8, 32 * vb + tcol);
    auto read = [&](const char* tile, int o0, int o1) __attribute__((always_inline)) {
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(tile + o0));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(tile + o1));
        return __builtin_bit_cast(frag, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    f32x16 acc, small;   // (the products of the smaller terms apart: the large ones' sum then has one rounding per 16 positions)
#pragma unroll
    for (int x = 0; x < 16; x++) acc[x] = small[x] = 0.f;
    float n0 = 0.f, n1 = 0.f;   // the vector state of keys 2 k2, 2 k2 + 1 over every eighth position
    const int k2 = tid & 31, pg = tid >> 5;
#pragma unroll
    for (int p = 0; p < L / PART; p++) {
        __syncthreads();   // the weights are there; the part before has been read
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int row = vrow + ROWS * i, to = Z::off(row, Z::EPC * vch);
            u32x4 k8 = kset[p][i], v8 = vset[p][i];
            if (!whole && p0 + PART * p + row >= S) k8 = v8 = u32x4{0, 0, 0, 0};   // (a weight of 0 would not do: the last row may be infinite)
            *reinterpret_cast<u32x4*>(kt + to) = k8;
            const float w = sw[PART * p + row];
            float x[8];
            unpack8<T>(v8, x);
            f32x4 lo4{x[0] * w, x[1] * w, x[2] * w, x[3] * w}, hi4{x[4] * w, x[5] * w, x[6] * w, x[7] * w};
#pragma unroll
            for (int term = 0; term < 3; term++) {
                const Pair t{R::cvt4(lo4), R::cvt4(hi4)};
                *reinterpret_cast<Pair*>(vt(term) + to) = t;
                lo4 -= __builtin_convertvector(t.lo, f32x4);
                hi4 -= __builtin_convertvector(t.hi, f32x4);
            }
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < PART / KW; n++) {
            const int at = KW * n * Z::ROW_BYTES;
            const frag af = read(kt + at, ko0, ko1);
            R::mma(small, af, read(vt(2) + at, vo0, vo1));
            R::mma(small, af, read(vt(1) + at, vo0, vo1));
            R::mma(acc, af, read(vt(0) + at, vo0, vo1));
        }
#pragma unroll 8
        for (int r = pg; r < PART; r += 8) {
            typedef T T2 __attribute__((ext_vector_type(2)));
            const T2 kv = *reinterpret_cast<const T2*>(kt + Z::off(r, 2 * k2));
            const float w2 = sw2[PART * p + r];
            n0 = fmaf((float)kv[0], w2, n0);
            n1 = fmaf((float)kv[1], w2, n1);
        }
    }
    acc += small;
    float seen = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) seen = not_finite(seen, acc[r]);
    float* const out = a.dC + ((size_t)bh * a.NCS + cc) * D * D + (size_t)(32 * kb) * D + 32 * vb + c32;
    if (__any(seen != 0.f)) {
#pragma unroll 1
        for (int r = 0; r < 16; r++) {
            const int k = 8 * (r >> 2) + 4 * h + (r & 3);
            float sum = 0.f;
#pragma unroll 1
            for (int j = 0; j < L && p0 + j < S; j++) sum = fmaf((float)Kh[(size_t)j * rsK + 32 * kb + k], (float)Vh[(size_t)j * rsV + 32 * vb + c32] * sw[j], sum);
            out[(size_t)k * D] = sum;
        }
    } else {
#pragma unroll
        for (int r = 0; r < 16; r++) out[(size_t)(8 * (r >> 2) + 4 * h + (r & 3)) * D] = acc[r];
    }
    __syncthreads();
    float* const red = reinterpret_cast<float*>(smem);   // [eighth][key]
    *reinterpret_cast<float2*>(red + pg * W + 2 * k2) = make_float2(n0, n1);
    __syncthreads();
    if (tid < W) {
        float sum = 0.f;
#pragma unroll
        for (int g = 0; g < 8; g++) sum += red[g * W + tid];
        a.Nst[((size_t)bh * a.NCS + cc) * D + tid] = sum;
    }
#endif
}

// The chunk sums for the shapes the kernel above does not serve (fp32 at D = 64 and 128, 16-bit types at D = 64), as fp32
// MFMA products with both operands straight from global memory: the positions are the inner dimension, so a lane's share of
// an operand is one element of a row and a wave's load is a piece of two rows.  No tile passes through LDS and no wave waits
// for another until the end.  One workgroup per (head, chunk, 32 value columns); a wave forms one 32 x 32 block (D = 128: four
// key blocks; D = 64: two, each by two waves that take the chunk's tiles of 32 positions in turns and add up at the end).
// What bounds it is one trip to memory and the products of a wave, 64 MFMAs of 64 cycles per 128 positions: the loads of two
// tiles leave before the first product.
// (Before: plain multiply-adds out of LDS tiles, 11.5 us at B1 H4 S2048 D64 fp32, 20.7 us at B2 H4 S4096 D64 bf16.)
template <typename T, int D>
__global__ __launch_bounds__(256, 2) void chunk_sum_small_kernel(ChunkArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int VB = D / 32, KB = D / 32, PG = 4 / KB;   // PG: waves that share a key block
    constexpr int TP = 32, NS = TP / 2;                     // positions per tile, MFMAs of two positions
    __shared__ float sw[4][2][TP];                          // [wave][matrix, vector][position: even ones, then odd]
    __shared__ float red[PG > 1 ? KB : 1][16][64];
    __shared__ float redn[D];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, c32 = lane & 31;
    const int kb = wave % KB, pg = wave / KB;
    const int vb = blockIdx.x % VB, pair = blockIdx.x / VB;
    const int cc = pair % a.NCS, bh = pair / a.NCS;
    const int S = a.S, L = a.L;
    const size_t poff = (size_t)bh * a.NG * GRAN, goff = (size_t)bh * a.NG;
    // (the positions and the reference point of a sum: see chunk_sum_kernel)
    const int p0 = (a.reverse ? cc + 1 : cc) * L, pe = a.reverse ? p0 - 1 : p0 + L - 1;
    const size_t rsK = (size_t)a.lk.ss, rsV = (size_t)a.lv.ss;
    const T* Kh = reinterpret_cast<const T*>(a.K) + a.lk.head(bh) + 32 * kb;
    const T* Vh = reinterpret_cast<const T*>(a.V) + a.lv.head(bh) + 32 * vb;
    const float log2scale = -0.5f * __log2f((float)D);
    const float bend = a.beta2[poff + pe];
    const double Gend = a.G2[goff + pe / GRAN];
    const int n_pos = p0 + L <= S ? L : S - p0, n_tiles = (n_pos + TP - 1) / TP;

    struct Tile { T k[NS], v[NS]; float x, x1, x2; double g; };
    auto load = [&](Tile& t, int j) __attribute__((always_inline)) {   // step s: position 2 s + h of tile j
        const int t0 = p0 + TP * j;
        {   // what the weight of position t0 + c32 needs
            const int pos = t0 + c32 < S ? t0 + c32 : S - 1;
            t.g = a.G2[goff + pos / GRAN];
            t.x = a.reverse ? a.beta2[poff + pos] : a.alpha2[poff + pos];
            t.x1 = a.reverse ? a.inv_n[poff + pos] : 0.f;
            t.x2 = a.reverse ? a.db[poff + pos] : 0.f;
        }
        const T* kt = Kh + (size_t)t0 * rsK;   // (the same for all lanes)
        const T* vt = Vh + (size_t)t0 * rsV;
        const unsigned ko = (unsigned)(h * rsK) + c32, vo = (unsigned)(h * rsV) + c32;
        if (__builtin_expect(t0 + TP <= S, 1)) {
#pragma unroll
            for (int s = 0; s < NS; s++) { t.k[s] = (kt + (size_t)(2 * s) * rsK)[ko]; t.v[s] = (vt + (size_t)(2 * s) * rsV)[vo]; }
        } else {   // (rows past the end are zeros)
#pragma unroll
            for (int s = 0; s < NS; s++) {
                t.k[s] = element_or_zero(t0 + 2 * s + h < S, kt + (size_t)(2 * s) * rsK + ko);
                t.v[s] = element_or_zero(t0 + 2 * s + h < S, vt + (size_t)(2 * s) * rsV + vo);
            }
        }
    };
    f32x16 acc;
#pragma unroll
    for (int x = 0; x < 16; x++) acc[x] = 0.f;
    float nacc = 0.f;
    auto work = [&](const Tile& t, int j) __attribute__((always_inline)) {
        float w = 0.f, w2 = 0.f;
        if (p0 + TP * j + c32 < S) {
            if (a.reverse) {
                const float rho = fast_exp2(bend - t.x + (float)(t.g - Gend) + log2scale);
                w = rho * t.x1;
                w2 = rho * t.x2;
            } else {
                w = w2 = fast_exp2(t.x - bend + (float)(Gend - t.g) + log2scale);
            }
        }
        // (the wave's own part of LDS: no barrier)
        if (h == 0) {
            sw[wave][0][(c32 & 1) * NS + (c32 >> 1)] = w;
            sw[wave][1][(c32 & 1) * NS + (c32 >> 1)] = w2;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s4 = 0; s4 < NS; s4 += 4) {
            const f32x4 wv = *reinterpret_cast<const f32x4*>(&sw[wave][0][h * NS + s4]), wn = *reinterpret_cast<const f32x4*>(&sw[wave][1][h * NS + s4]);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float kv = (float)t.k[s4 + e];
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv, (float)t.v[s4 + e] * wv[e], acc, 0, 0, 0);
                nacc += kv * wn[e];
            }
        }
        __builtin_amdgcn_wave_barrier();
    };
    Tile ta, tb;
    int j = pg;
    if (j < n_tiles) load(ta, j);
    for (; j < n_tiles; j += 2 * PG) {
        if (j + PG < n_tiles) load(tb, j + PG);
        work(ta, j);
        if (j + PG < n_tiles) {
            if (j + 2 * PG < n_tiles) load(ta, j + 2 * PG);
            work(tb, j + PG);
        }
    }
    nacc = sum_halves(nacc);
    if constexpr (PG > 1) {
        if (pg == 1) {
#pragma unroll
            for (int x = 0; x < 16; x++) red[kb][x][lane] = acc[x];
            if (h == 0) redn[32 * kb + c32] = nacc;
        }
        __syncthreads();
        if (pg == 1) return;
#pragma unroll
        for (int x = 0; x < 16; x++) acc[x] += red[kb][x][lane];
        nacc += redn[32 * kb + c32];
    }
    float* out = a.dC + ((size_t)bh * a.NCS + cc) * D * D + (size_t)(32 * kb) * D + 32 * vb + c32;
#pragma unroll
    for (int r = 0; r < 16; r++) out[(size_t)(8 * (r >> 2) + 4 * h + (r & 3)) * D] = acc[r];
    if (vb == 0 && h == 0) a.Nst[((size_t)bh * a.NCS + cc) * D + 32 * kb + c32] = nacc;
#endif
}

// gamma_c = exp(A_{e_{c-1}} - A_{e_c}), e_c the last position of chunk c (c >= 1, both chunks complete): what the state
// at the end of chunk c - 1 decays by until the end of chunk c, and what the reverse state behind chunk c decays by
// until it is seen from the end of chunk c - 1
__device__ __forceinline__ float carry_gamma(const ChunkArgs& a, size_t poff, size_t goff, int c) {
    const int e0 = c * a.L - 1, e1 = e0 + a.L;
    return fast_exp2(a.beta2[poff + e0] - a.beta2[poff + e1] + (float)(a.G2[goff + e1 / GRAN] - a.G2[goff + e0 / GRAN]));
}

template <typename T, int D>
__global__ __launch_bounds__(256) void chunk_carry_kernel(ChunkArgs a) {
    const int bh = blockIdx.y, tid = threadIdx.x;
    const int idx = blockIdx.x * 256 + tid;
    const int k = idx / (D / 8), v8 = (idx % (D / 8)) * 8;
    const size_t poff = (size_t)bh * a.NG * GRAN, goff = (size_t)bh * a.NG;
    const int L = a.L;
    const size_t hbase = (size_t)bh * a.NCS * D * D;
    const float* src = a.dC + hbase + (size_t)k * D + v8;
    const size_t koff = hbase + (size_t)state_row(k) * D + v8;   // key-major: eight values of key k
    float* nst = a.Nst + (size_t)bh * a.NCS * D + tid;
    const bool vec = blockIdx.x == 0 && tid < D;
    f32x4 run0 = {0.f, 0.f, 0.f, 0.f}, run1 = {0.f, 0.f, 0.f, 0.f};
    float nrun = 0.f;
    typedef typename Tr<T>::vec4 V4;
    struct Pair { V4 lo, hi; };
    // The steps depend on each other through the running state only: the chunk sums, the decay factors and the vector
    // sums of four steps are requested together (one memory round trip per four steps; with few heads this kernel is a
    // handful of workgroups waiting for memory, step by step)
    constexpr int AHEAD = 4;
    for (int step0 = 0; step0 < a.NCS; step0 += AHEAD) {
      f32x4 d0s[AHEAD], d1s[AHEAD];
      float gams[AHEAD], nin[AHEAD];
#pragma unroll
      for (int u = 0; u < AHEAD; u++) {
          const int step = step0 + u < a.NCS ? step0 + u : a.NCS - 1;
          const int c = a.reverse ? a.NCS - 1 - step : step;
          gams[u] = step > 0 ? carry_gamma(a, poff, goff, a.reverse ? c + 1 : c) : 0.f;
          d0s[u] = *reinterpret_cast<const f32x4*>(src + (size_t)c * D * D);
          d1s[u] = *reinterpret_cast<const f32x4*>(src + (size_t)c * D * D + 4);
          nin[u] = vec ? nst[(size_t)c * D] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < AHEAD; u++) {
        const int step = step0 + u;
        if (step >= a.NCS) break;
        const int c = a.reverse ? a.NCS - 1 - step : step;
        const float gam = gams[u];
        run0 = run0 * gam + d0s[u];
        run1 = run1 * gam + d1s[u];
#pragma unroll
        for (int e = 0; e < 4; e++) {   // (see chunk_carry_t_kernel: the fp32 value is fixed before any conversion)
            asm volatile("" : "+v"(run0[e]));
            asm volatile("" : "+v"(run1[e]));
        }
        Pair o, rest;
        const bool split = a.Cst_lo || a.CstT_lo;   // split mode: the state as two terms
        if (split) {
            Tr<T>::cvt4_split(run0, o.lo, rest.lo);
            Tr<T>::cvt4_split(run1, o.hi, rest.hi);
        } else {
            o.lo = Tr<T>::cvt4(run0);
            o.hi = Tr<T>::cvt4(run1);
        }
        if (a.Cst) {
            *reinterpret_cast<Pair*>(reinterpret_cast<T*>(a.Cst) + koff + (size_t)c * D * D) = o;
            if (a.Cst_lo) *reinterpret_cast<Pair*>(reinterpret_cast<T*>(a.Cst_lo) + koff + (size_t)c * D * D) = rest;
        }
        if (a.CstT) {
            // value-major copy, element by element (the small shapes only: at D = 128 and 256 in 16 bits
            // chunk_carry_t_kernel turns the blocks round in LDS)
            T* t = reinterpret_cast<T*>(a.CstT) + hbase + (size_t)c * D * D + k;
            T* tl = a.CstT_lo ? reinterpret_cast<T*>(a.CstT_lo) + hbase + (size_t)c * D * D + k : nullptr;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const size_t r = (size_t)state_row(v8 + e) * D;
                t[r] = e < 4 ? o.lo[e & 3] : o.hi[e & 3];
                if (tl) tl[r] = e < 4 ? rest.lo[e & 3] : rest.hi[e & 3];
            }
        }
        if (vec) {
            nrun = nrun * gam + nin[u];
            nst[(size_t)c * D] = nrun;
        }
      }
    }
}

// Both carries leave the contraction of two sets of states (ChunkArgs::dot_with) as one sum per block of 32 values x 32 keys,
// added up in one order -- the four elements of a group, the eight groups of a row, the 32 rows, each as a balanced tree -- so that
// dF is the same bits whichever of them the number of heads selects.  (Nothing is contracted to a multiply-add here: the two
// kernels would not agree on which.)
__device__ __forceinline__ float dot_group(f32x4 x, f32x4 y) {
#pragma clang fp contract(off)
    const f32x4 p = x * y;
    return (p[0] + p[1]) + (p[2] + p[3]);
}

// The carry of the shapes of chunk_sum_small_kernel, and of the others where few workgroups would run (carry_in_small_blocks): a workgroup takes 32 keys x 32 values of a head's state, sixteen chunks'
// sums at a time in registers (one trip to memory per sixteen steps, whatever the number of heads), writes either layout or
// both -- the value-major one through LDS, in whole 64- or 128-byte pieces of a row -- and forms the contraction with another
// set of states (ChunkArgs::dot_with) on the way.
// Four steps share a barrier: their states go to LDS one after the other and come back turned round side by side.  With a barrier per
// step it was a chain of LDS round trips and lane reductions: with the contraction 91 us -> 60 at 64 heads x 31 states x 128 x 128 (16 bits),
// 10.1 -> 7.5 at 8 x 2 x 256 x 256 in split mode, 8.8 -> 6.7 at 8 x 7 x 128 x 128 (fp32).
// (Before: 2 to 8 workgroups per head, four steps at a time, the value-major copy element by element, and a kernel of its own
// for the contraction: 14.6 + 4.7 us at B1 H4 S2048 D64 fp32.)
// DOT: 0 no contraction, 1 with states of one term, 2 of two (their fragments cost registers, and registers workgroups per CU)
template <typename T, int D, int DOT>
__global__ __launch_bounds__(256) void chunk_carry_small_kernel(ChunkArgs a) {
    constexpr int AHEAD = 16, GROUP = 4, MAXC = 1024;   // (S <= 131072 in chunks of at least 128)
    typedef typename Tr<T>::vec4 V4;
    __shared__ __attribute__((aligned(16))) float tile[2][GROUP][32][36];   // [parity of the group][step]
    __shared__ float gams[MAXC];
    __shared__ float red[2][GROUP][4];
    const int bh = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kb = blockIdx.x / (D / 32), vb = blockIdx.x % (D / 32);
    const int row = tid >> 3, c4 = 4 * (tid & 7);   // row of the block (key; value in the turned one) and first of four columns
    const size_t poff = (size_t)bh * a.NG * GRAN, goff = (size_t)bh * a.NG, hbase = (size_t)bh * a.NCS * D * D;
    const float* src = a.dC + hbase + (size_t)(32 * kb + row) * D + 32 * vb + c4;
    const size_t koff = hbase + (size_t)state_row(32 * kb + row) * D + 32 * vb + c4;   // key-major
    const size_t voff = hbase + (size_t)state_row(32 * vb + row) * D + 32 * kb + c4;   // value-major
    float* nst = a.Nst + (size_t)bh * a.NCS * D + tid;
    const bool vec = blockIdx.x == 0 && tid < D;
    auto chunk_of = [&](int step) { return a.reverse ? a.NCS - 1 - step : step; };
    f32x4 d[AHEAD];
    V4 y[DOT ? AHEAD : 1], yl[DOT == 2 ? AHEAD : 1];
    float nin[AHEAD];
    auto request = [&](int step0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            const int c = chunk_of(step0 + u < a.NCS ? step0 + u : a.NCS - 1);
            const size_t co = (size_t)c * D * D;
            d[u] = *reinterpret_cast<const f32x4*>(src + co);
            if constexpr (DOT > 0) {
                y[u] = *reinterpret_cast<const V4*>(reinterpret_cast<const T*>(a.dot_with) + voff + co);
                if constexpr (DOT == 2) yl[u] = *reinterpret_cast<const V4*>(reinterpret_cast<const T*>(a.dot_with_lo) + voff + co);
            }
            nin[u] = vec ? nst[(size_t)c * D] : 0.f;
        }
    };
    request(0);
    for (int step = tid; step < a.NCS; step += 256)
        gams[step] = step > 0 ? carry_gamma(a, poff, goff, a.reverse ? chunk_of(step) + 1 : chunk_of(step)) : 0.f;
    __syncthreads();
    const bool split = a.Cst_lo || a.CstT_lo;
    f32x4 run = {0.f, 0.f, 0.f, 0.f};
    float nrun = 0.f;
    auto put = [&](void* hi_base, void* lo_base, size_t off, f32x4 x, V4& hi, V4& lo) __attribute__((always_inline)) {
        if (split) Tr<T>::cvt4_split(x, hi, lo);
        else hi = Tr<T>::cvt4(x);
        if (hi_base) *reinterpret_cast<V4*>(reinterpret_cast<T*>(hi_base) + off) = hi;
        if (lo_base) *reinterpret_cast<V4*>(reinterpret_cast<T*>(lo_base) + off) = lo;
    };
    auto put_dots = [&](int first) {   // of a group's steps, behind the barrier that follows their partial sums
        if constexpr (DOT > 0) {
            if (tid < GROUP && first + tid < a.NCS) {
                const float* const r = red[(first / GROUP) & 1][tid];
                a.dot_part[((size_t)bh * a.NCS + chunk_of(first + tid)) * gridDim.x + blockIdx.x] = (r[0] + r[1]) + (r[2] + r[3]);
            }
        }
    };
    for (int step0 = 0; step0 < a.NCS; step0 += AHEAD) {
        if (step0 > 0) request(step0);
#pragma unroll
        for (int u0 = 0; u0 < AHEAD; u0 += GROUP) {
            const int first = step0 + u0, par = (first / GROUP) & 1;
            if (first < a.NCS) {
            V4 hi, lo;
#pragma unroll
            for (int g = 0; g < GROUP; g++) {
                const int step = first + g;
                if (step < a.NCS) {
                    const float gam = gams[step];
                    run = run * gam + d[u0 + g];
#pragma unroll
                    for (int e = 0; e < 4; e++) asm volatile("" : "+v"(run[e]));   // (see chunk_carry_t_kernel)
                    if (a.Cst) put(a.Cst, a.Cst_lo, koff + (size_t)chunk_of(step) * D * D, run, hi, lo);
                    if (a.CstT) {
#pragma unroll
                        for (int e = 0; e < 4; e++) tile[par][g][c4 + e][row] = run[e];
                    }
                    if (vec) {
                        nrun = nrun * gam + nin[u0 + g];
                        nst[(size_t)chunk_of(step) * D] = nrun;
                    }
                }
            }
            if (a.CstT) {   // (uniform) turned round in LDS
                __syncthreads();
                if (first > 0) put_dots(first - GROUP);
#pragma unroll
                for (int g = 0; g < GROUP; g++) {
                    const int step = first + g;
                    if (step < a.NCS) {
                        const f32x4 x = *reinterpret_cast<const f32x4*>(&tile[par][g][row][c4]);
                        put(a.CstT, a.CstT_lo, voff + (size_t)chunk_of(step) * D * D, x, hi, lo);
                        if constexpr (DOT > 0) {   // the state as it is written (the sum of its terms in split mode)
                            f32x4 xs = __builtin_convertvector(hi, f32x4), ys = __builtin_convertvector(y[u0 + g], f32x4);
                            if (split) xs += __builtin_convertvector(lo, f32x4);
                            if constexpr (DOT == 2) ys += __builtin_convertvector(yl[u0 + g], f32x4);
                            const float dot = wave_reduce<OpAdd>(dot_group(xs, ys));   // (a wave: eight rows of eight groups)
                            if (lane == 0) red[par][g][wave] = dot;
                        }
                    }
                }
            }
            }
        }
    }
    if constexpr (DOT > 0) {
        __syncthreads();
        put_dots((a.NCS - 1) / GROUP * GROUP);
    }
}

// The same carry with the states written transposed, [value][key], for the dQ pass (which contracts the state over the
// value index): a workgroup takes 64 values x 64 keys, reads the chunk sums along the value index (coalesced), and
// turns the block round in LDS so that the rows leave 128 bytes at a time.  Rows in the contraction order of the row
// kernel, like the untransposed states.
template <typename T, int D, bool DOT, bool KM>
__global__ __launch_bounds__(256, 4) void chunk_carry_t_kernel(ChunkArgs a) {
    __shared__ __attribute__((aligned(16))) T tile[2][64][64 + 8];   // [hi | lo (split mode)]
    const int bh = blockIdx.y, tid = threadIdx.x;
    const bool split = a.CstT_lo != nullptr;
    const int vb = blockIdx.x % (D / 64), kb = blockIdx.x / (D / 64);
    const int vl = tid & 63, kq = tid >> 6;
    const size_t poff = (size_t)bh * a.NG * GRAN, goff = (size_t)bh * a.NG;
    const int L = a.L;
    const int orow = tid >> 2, opiece = tid & 3;
    const int vrow = 64 * vb + orow;
    T* dst = reinterpret_cast<T*>(a.CstT) + (size_t)bh * a.NCS * D * D + (size_t)((vrow & ~15) | perm16(vrow & 15)) * D + 64 * kb + 16 * opiece;
    f32x8 run[2];
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int e = 0; e < 8; e++) run[g][e] = 0.f;
    float* nst = a.Nst + (size_t)bh * a.NCS * D + tid;   // the vector states, in place, by the first workgroup of a head
    const bool vec = blockIdx.x == 0 && tid < D;
    float nrun = 0.f;
    __shared__ float red[4][2];
    const int lane = tid & 63, wave = tid >> 6;
    // (the kernel moves 4 bytes in and 2 to 4 out per element and, where it is chosen, fills the chip and runs at memory speed:
    // nothing to gain from requesting a step's chunk sums ahead of time)
    for (int step = 0; step < a.NCS; step++) {
        const int c = a.reverse ? a.NCS - 1 - step : step;
        const float gam = step > 0 ? carry_gamma(a, poff, goff, a.reverse ? c + 1 : c) : 0.f;
        if (vec) {
            nrun = nrun * gam + nst[(size_t)c * D];
            nst[(size_t)c * D] = nrun;
        }
        const float* src = a.dC + ((size_t)bh * a.NCS + c) * D * D + 64 * vb + vl;
        typedef typename Tr<T>::frag V8;
#pragma unroll
        for (int g = 0; g < 2; g++) {
            f32x8 d;
#pragma unroll
            for (int e = 0; e < 8; e++) d[e] = src[(size_t)(64 * kb + 8 * (kq + 4 * g) + e) * D];
            run[g] = run[g] * gam + d;
            // (the fp32 value is fixed here: left to itself the compiler may fold this multiply-add into a conversion to
            // fp16 further down -- one rounding instead of two -- in one kernel and not in its twin, and the two carries
            // must give the same bits)
#pragma unroll
            for (int e = 0; e < 8; e++) asm volatile("" : "+v"(run[g][e]));
            if constexpr (KM) {   // key-major copy: lanes of a wave hold consecutive values of one key, 128 bytes per store
                const size_t koff = ((size_t)bh * a.NCS + c) * D * D + 64 * vb + vl;
                T* kd = reinterpret_cast<T*>(a.Cst) + koff;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int k = 64 * kb + 8 * (kq + 4 * g) + e;
                    const T hi = (T)run[g][e];
                    kd[(size_t)((k & ~15) | perm16(k & 15)) * D] = hi;
                    if (a.Cst_lo) (reinterpret_cast<T*>(a.Cst_lo) + koff)[(size_t)((k & ~15) | perm16(k & 15)) * D] = (T)(run[g][e] - (float)hi);
                }
            }
            typedef typename Tr<T>::vec4 V4;
            struct Pair { V4 lo, hi; };
            Pair o;
            if (split) {   // the state as two terms: the second holds what rounding to the element type loses
                Pair rest;
                Tr<T>::cvt4_split(__builtin_shufflevector(run[g], run[g], 0, 1, 2, 3), o.lo, rest.lo);
                Tr<T>::cvt4_split(__builtin_shufflevector(run[g], run[g], 4, 5, 6, 7), o.hi, rest.hi);
                *reinterpret_cast<Pair*>(&tile[1][vl][8 * (kq + 4 * g)]) = rest;
            } else {
                o.lo = Tr<T>::cvt4(__builtin_shufflevector(run[g], run[g], 0, 1, 2, 3));
                o.hi = Tr<T>::cvt4(__builtin_shufflevector(run[g], run[g], 4, 5, 6, 7));
            }
            *reinterpret_cast<Pair*>(&tile[0][vl][8 * (kq + 4 * g)]) = o;
        }
        __syncthreads();
        const uint4 p0 = *reinterpret_cast<const uint4*>(&tile[0][orow][16 * opiece]), p1 = *reinterpret_cast<const uint4*>(&tile[0][orow][16 * opiece + 8]);
        *reinterpret_cast<uint4*>(dst + (size_t)c * D * D) = p0;
        *reinterpret_cast<uint4*>(dst + (size_t)c * D * D + 8) = p1;
        if constexpr (DOT) {   // <state c as it is written (the sum of its terms in split mode), the other set's state c>
            f32x8 x0 = __builtin_convertvector(__builtin_bit_cast(V8, p0), f32x8), x1 = __builtin_convertvector(__builtin_bit_cast(V8, p1), f32x8);
            // the other set's state c at the places this thread has just written (four workgroups share a CU: their
            // steps hide this round trip)
            const size_t doff = (size_t)(dst - reinterpret_cast<T*>(a.CstT)) + (size_t)c * D * D;
            const T* other = reinterpret_cast<const T*>(a.dot_with) + doff;
            f32x8 y0 = __builtin_convertvector(*reinterpret_cast<const V8*>(other), f32x8);
            f32x8 y1 = __builtin_convertvector(*reinterpret_cast<const V8*>(other + 8), f32x8);
            if (split) {
                x0 += __builtin_convertvector(*reinterpret_cast<const V8*>(&tile[1][orow][16 * opiece]), f32x8);
                x1 += __builtin_convertvector(*reinterpret_cast<const V8*>(&tile[1][orow][16 * opiece + 8]), f32x8);
            }
            if (a.dot_with_lo) {
                const T* other_lo = reinterpret_cast<const T*>(a.dot_with_lo) + doff;
                y0 += __builtin_convertvector(*reinterpret_cast<const V8*>(other_lo), f32x8);
                y1 += __builtin_convertvector(*reinterpret_cast<const V8*>(other_lo + 8), f32x8);
            }
            auto low = [](const f32x8& x) { return __builtin_shufflevector(x, x, 0, 1, 2, 3); };
            auto high = [](const f32x8& x) { return __builtin_shufflevector(x, x, 4, 5, 6, 7); };
            // a lane: four groups of a row; two lanes: the row of a block; a wave: sixteen rows of two blocks side by side
            float dot = (dot_group(low(x0), low(y0)) + dot_group(high(x0), high(y0))) + (dot_group(low(x1), low(y1)) + dot_group(high(x1), high(y1)));
            dot += dpp_f<0xb1>(0.f, dot);                 // quad_perm: the other lane of the pair
            dot += dpp_f<0x114>(0.f, dot);                // row_shr:4, row_shr:8
            dot += dpp_f<0x118>(0.f, dot);
            auto at = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, dot), l)); };
            const float left = (at(13) + at(29)) + (at(45) + at(61)), right = (at(15) + at(31)) + (at(47) + at(63));
            if (lane == 0) { red[wave][0] = left; red[wave][1] = right; }
        }
        if (split) {
            T* dlo = reinterpret_cast<T*>(a.CstT_lo) + (dst - reinterpret_cast<T*>(a.CstT));
            *reinterpret_cast<uint4*>(dlo + (size_t)c * D * D) = *reinterpret_cast<const uint4*>(&tile[1][orow][16 * opiece]);
            *reinterpret_cast<uint4*>(dlo + (size_t)c * D * D + 8) = *reinterpret_cast<const uint4*>(&tile[1][orow][16 * opiece + 8]);
        }
        __syncthreads();
        // (the waves' sums were written between the two barriers; the next ones follow the next barrier)
        if (DOT && tid < 4) {   // block (values 32 (2 vb + tid / 2) .., keys 32 (2 kb + tid % 2) ..)
            const int vh = tid >> 1, kh = tid & 1;
            a.dot_part[((size_t)bh * a.NCS + c) * (D / 32) * (D / 32) + (2 * kb + kh) * (D / 32) + 2 * vb + vh] = red[2 * vh][kh] + red[2 * vh + 1][kh];
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// The same states in ONE pass, bit for bit those of the two kernels above: a workgroup owns 64 keys x VW values of a head's
// state and walks the head's chunks in their order (forward: first to last; reverse: last to first).  Two sets of
// accumulators: the chunk's own sum, and the running state that takes it at the chunk's end (state = gamma * state + sum) and is
// written in the element type.  No fp32 chunk sums travel through memory (4 + 4 bytes per state element in the two-kernel form), no
// second launch.  WPH workgroups per head; chunk_seq_serves decides.
//
// Eight waves, two on every SIMD.  Waves 0..3 multiply straight out of the stages: the positions' weights go onto the V fragments in
// registers (rounded to the element type as chunk_sum_kernel rounds its weighted V rows); a wave owns 32 values, so that at
// D = 256 a weighted fragment serves two products.  Operands are requested two contraction steps ahead and weighed one step ahead,
// across the tiles.  They write the states and own every global store.  Waves 4 and 5 copy: the tiles (64 positions: K's 64
// columns, V's VW columns) and the positions' gate rows by direct global->LDS loads, the tiles PF ahead into NS = PF + 1 stages, the gate
// rows one further ahead; and form the positions' weights, two tiles ahead.  Waves 6 and 7 add up the vector state from K.  (All
// four copying and adding up in turn: a wave sits 600 cycles per tile in the issue of its copies, and what it does behind them came on top,
// 1900 cycles per tile where the products need 1100.)  One barrier per tile; behind it tiles t and t + 1 and the weights
// of both are there.  The copies are counted by hand: a copying wave issues exactly NI direct loads per tile and no other vector
// memory operation, and waits with vmcnt((PF - 2) * NI) -- everything but the newest PF - 2 tiles -- before the barrier
// that hands a tile on; a compiled kernel that uses scratch memory is not launched (launch_chunk_t then takes the two kernels).
template <typename T, int D>
struct SeqCfg {
    static constexpr int KR = 64, VW = D / 2;
    static constexpr int NKB = VW / 64;                                // key blocks of a multiplying wave
    static constexpr int KP = GRAN * KR * (int)sizeof(T) / 16 / 128, VP = GRAN * VW * (int)sizeof(T) / 16 / 128;   // direct loads per copying wave and tile: K, V
    static constexpr int NI = KP + VP + 2;                             // ... and two gate rows
    static constexpr int MAX_STEPS = 256;                              // chunk states per head
    static constexpr int NPG = 2048 / D;                               // groups of rows of the vector sum (as in chunk_sum_kernel)
    static constexpr size_t K_BYTES = (size_t)GRAN * KR * sizeof(T), V_BYTES = (size_t)GRAN * VW * sizeof(T), AUX_BYTES = 4 * GRAN * sizeof(float);
    static constexpr size_t STAGE_BYTES = K_BYTES + V_BYTES + AUX_BYTES;
    static constexpr size_t SW_BYTES = 4 * 2 * GRAN * sizeof(float);   // [tile modulo 4][matrix, vector][position]
    static constexpr size_t RED_BYTES = 2 * NPG * 32 * sizeof(float);  // [parity of the step][group][key]
    static constexpr size_t TABLE_BYTES = MAX_STEPS * (sizeof(double) + 2 * sizeof(float));
    static constexpr size_t FIXED_BYTES = SW_BYTES + RED_BYTES + TABLE_BYTES;
    // tiles requested ahead: as many stages as LDS holds
    static constexpr int FIT = (int)((160 * 1024 - FIXED_BYTES) / STAGE_BYTES), NS = FIT < 8 ? FIT : 8, PF = NS - 1;
    static_assert(PF >= 3 && (PF - 2) * NI < 64, "the counted wait must fit vmcnt's six bits");
    static constexpr size_t LDS_BYTES = NS * STAGE_BYTES + FIXED_BYTES;
    static constexpr int WPH = (D / KR) * (D / VW);                    // workgroups per head
};

// KM, VM: key-major and value-major states are written (ChunkArgs::Cst, CstT); DOT: the contraction with another set on the way; STRICT: split
// mode (ChunkArgs::precise): the weighted values and the states as two terms
template <typename T, int D, bool KM, bool VM, bool DOT, bool STRICT>
__global__ __launch_bounds__(512) void chunk_seq_kernel(ChunkArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
    using R = Tr<T>;
    using Cfg = SeqCfg<T, D>;
    typedef typename R::frag frag;
    typedef typename R::vec4 V4;
    static_assert(R::HALF && (D == 128 || D == 256), "16-bit types, D = 128 or 256");
    constexpr int VW = Cfg::VW, NKB = Cfg::NKB, KW = R::KW, NS = Cfg::NS, PF = Cfg::PF, NI = Cfg::NI, NPG = Cfg::NPG;
    constexpr int SB = (int)Cfg::STAGE_BYTES, KB = (int)Cfg::K_BYTES, AUX = (int)(Cfg::K_BYTES + Cfg::V_BYTES);
    using ZK = Swz<T, 64>;
    using ZV = Swz<T, VW>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float* const sw = reinterpret_cast<float*>(smem + NS * SB);     // [4][2][64]
    float* const red = sw + 4 * 2 * GRAN;                           // [2][NPG][32]
    double* const tGend = reinterpret_cast<double*>(red + 2 * NPG * 32);
    float* const tbend = reinterpret_cast<float*>(tGend + Cfg::MAX_STEPS);
    float* const tgam = tbend + Cfg::MAX_STEPS;

    const bool feeder = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) != 0;
    const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, c32 = lane & 31;
    // the workgroups of a head on one XCD (they read the same K and V columns), heads dealt round the eight XCDs
    int w, bh;
    if ((a.BH & 7) == 0) { const int q = blockIdx.x >> 3; w = q % Cfg::WPH; bh = (blockIdx.x & 7) + 8 * (q / Cfg::WPH); }
    else { w = blockIdx.x % Cfg::WPH; bh = blockIdx.x / Cfg::WPH; }
    const int kq = w >> 1, vh = w & 1;
    const int S = a.S, L = a.L, NT = L / GRAN, NCS = a.NCS;
    const size_t poff = (size_t)bh * a.NG * GRAN, goff = (size_t)bh * a.NG;
    const bool rev = a.reverse != 0;
    // step s of the walk: forward chunk s (state s); reverse the positions of chunk NCS - s (state NCS - 1 - s), of which
    // the first, the sequence's last chunk, may be short
    const int NT0 = rev ? (S - NCS * L + GRAN - 1) / GRAN : NT;
    const int NTOT = NT0 + (NCS - 1) * NT;
    auto state_of = [&](int s) { return rev ? NCS - 1 - s : s; };
    auto step_base = [&](int s) { return rev ? (NCS - s) * L : s * L; };
    // per step: the reference exponent of its weights and the decay into it
    for (int s = threadIdx.x; s < NCS; s += 512) {
        const int c = state_of(s), pe = (c + 1) * L - 1;   // forward: the chunk's last position; reverse: the last position before the chunk
        tbend[s] = a.beta2[poff + pe];
        tGend[s] = a.G2[goff + pe / GRAN];
        tgam[s] = s > 0 ? carry_gamma(a, poff, goff, rev ? c + 1 : c) : 0.f;
    }

    // Places in the walk, each advanced tile by tile: the step, how many of its tiles are left (this one included), the stage (bytes), and what
    // its user needs of the position.  Between steps only the reverse walk jumps, from the end of a chunk to the start of the one before.
    const int jump0 = -(NT0 * GRAN + L), jump = -(NT * GRAN + L);   // (the first step may be a short one)
    struct Place { int s, left, st; };
    const Place start{0, NT0, 0};
    auto next = [&](Place& c, auto&& jumped) __attribute__((always_inline)) {
        c.st = c.st == (NS - 1) * SB ? 0 : c.st + SB;
        if (__builtin_expect(--c.left == 0, 0)) {
            if (rev) jumped(c.s == 0 ? jump0 : jump);
            c.s++;
            c.left = NT;
        }
    };
    if (feeder && wave < 2) {   // ---- copies
        const size_t rsK = (size_t)a.lk.ss, rsV = (size_t)a.lv.ss;
        const T* const zeros = reinterpret_cast<const T*>(&zero_piece);
        const T* Kh = reinterpret_cast<const T*>(a.K) + a.lk.head(bh) + 64 * kq;
        const T* Vh = reinterpret_cast<const T*>(a.V) + a.lv.head(bh) + VW * vh;
        TileDma<T, 64, GRAN, 128> kdma;
        TileDma<T, VW, GRAN, 128> vdma;
        kdma.init(tid);
        vdma.init(tid);
        const auto krows = kdma.rows(tid, (unsigned)(rsK * sizeof(T)));
        const auto vrows = vdma.rows(tid, (unsigned)(rsV * sizeof(T)));
        static_assert(TileDma<T, 64, GRAN, 128>::PER_WAVE == Cfg::KP && TileDma<T, VW, GRAN, 128>::PER_WAVE == Cfg::VP, "direct loads per tile");
        // gate rows of a tile: 0 alpha (forward) or beta (reverse), 1 and 2 the dQ pass's 1/n and db (reverse; the forward repeats
        // alpha), 3 the granule's G (two dwords; the other lanes read them again).  Wave 0 brings rows 0 and 1, wave 1 rows 2 and 3.
        const float* const row0 = (rev ? a.beta2 : a.alpha2) + poff + lane;
        const float* ap0 = wave == 0 ? row0 : (rev ? a.db + poff + lane : row0);
        const float* ap1 = wave == 0 ? (rev ? a.inv_n + poff + lane : row0) : reinterpret_cast<const float*>(a.G2 + goff) + (lane & 1);
        const int ap1step = wave == 0 ? GRAN : 2;   // floats per tile
        dma_wait();   // (from here on this wave's vmcnt counts direct loads only)

        Place pi = start, pa = start, pw = start;   // the next tile to request, the next gate rows, the next tile to form weights for
        int pos_i = step_base(0), pos_w = pos_i;
        const T* kp = Kh + (size_t)pos_i * rsK;
        const T* vp = Vh + (size_t)pos_i * rsV;
        ap0 += pos_i;
        ap1 += pos_i / GRAN * ap1step;
        const size_t kstep = GRAN * rsK, vstep = GRAN * rsV;
        auto next_i = [&]() __attribute__((always_inline)) {
            pos_i += GRAN; kp += kstep; vp += vstep;
            next(pi, [&](int d) { pos_i += d; kp += (long long)d * (long long)rsK; vp += (long long)d * (long long)rsV; });
        };
        auto next_a = [&]() __attribute__((always_inline)) {
            ap0 += GRAN; ap1 += ap1step;
            next(pa, [&](int d) { ap0 += d; ap1 += d / GRAN * ap1step; });
        };
        auto issue_aux = [&]() __attribute__((always_inline)) {
            const unsigned to = __builtin_amdgcn_readfirstlane(lds_offset_of(smem + pa.st + AUX)) + wave * 512;
            dma4(ap0, to);
            dma4(ap1, to + 256);
        };
        auto issue = [&]() __attribute__((always_inline)) {
            T* const ks = reinterpret_cast<T*>(smem + pi.st);
            T* const vs = reinterpret_cast<T*>(smem + pi.st + KB);
            if (__builtin_expect(pos_i + GRAN <= S, 1)) {
                kdma.issue(ks, kp, krows);
                vdma.issue(vs, vp, vrows);
            } else {   // the sequence's last tile: rows past the end are zeros
                tile_dma_rolled<T, 64, GRAN, 128>(ks, Kh, pos_i, S, tid, rsK, zeros);
                tile_dma_rolled<T, VW, GRAN, 128>(vs, Vh, pos_i, S, tid, rsV, zeros);
            }
        };
        // the positions' weights of tile n (see chunk_sum_kernel), by the two waves in turns
        const float log2scale = -0.5f * __log2f((float)D);
        struct Gate { float x0, x1, x2, bend; double xg, Gend; } g{};
        auto gate_rows = [&]() __attribute__((always_inline)) {
            const float* const ax = reinterpret_cast<const float*>(smem + pw.st + AUX);
            g = Gate{ax[lane], ax[GRAN + lane], ax[2 * GRAN + lane], tbend[pw.s], *reinterpret_cast<const double*>(ax + 3 * GRAN), tGend[pw.s]};
        };
        auto weigh = [&](int n) __attribute__((always_inline)) {
            float wm, w2;
            if (rev) {
                const float rho = fast_exp2(g.bend - g.x0 + (float)(g.xg - g.Gend) + log2scale);
                wm = rho * g.x1;
                w2 = rho * g.x2;
            } else {
                wm = w2 = fast_exp2(g.x0 - g.bend + (float)(g.Gend - g.xg) + log2scale);
            }
            if (pos_w + lane >= S) wm = w2 = 0.f;
            float* const o = sw + (n & 3) * 2 * GRAN + lane;
            o[0] = wm;
            o[GRAN] = w2;
        };
        auto next_w = [&]() __attribute__((always_inline)) {
            pos_w += GRAN;
            next(pw, [&](int d) { pos_w += d; });
        };
        issue_aux();
        next_a();
        int t = 0;
        for (; t < PF && t < NTOT; t++) {   // (behind the last tile its own gate rows again: the count stays the same)
            issue();
            next_i();
            issue_aux();
            if (t + 2 < NTOT) next_a();
        }
        __syncthreads();   // the tables are there
        if (NTOT >= PF) dma_wait_but<(PF - 2) * NI>(); else dma_wait();
        __syncthreads();   // tiles 0 and 1 have landed, and the gate rows up to tile 2
        if (wave == 0) { gate_rows(); weigh(0); }
        next_w();
        if (NTOT > 1) {
            if (wave == 1) { gate_rows(); weigh(1); }
            next_w();
        }
        __syncthreads();   // their weights are there
        for (t = 0; t < NTOT; t++) {
            const bool more = t + PF < NTOT, ahead = t + 2 < NTOT, mine = wave == (t & 1);
            if (ahead && mine) gate_rows();
            __builtin_amdgcn_sched_barrier(0);
            if (more) {   // (into the stage of tile t - 1)
                issue();
                next_i();
                issue_aux();
                if (t + PF + 2 < NTOT) next_a();
            }
            __builtin_amdgcn_sched_barrier(0);
            if (ahead) {
                if (mine) weigh(t + 2);
                next_w();
            }
            if (more) dma_wait_but<(PF - 2) * NI>(); else dma_wait();
            __syncthreads();   // tile t + 2 has landed
        }
    } else if (feeder) {   // ---- the vector state
        const int ft = tid - 128;
        Place pv = start;   // the tile to add up
        // The vector sum of the workgroup's half of its 64 keys, in the order of chunk_sum_kernel: NPG partial sums per key, each over
        // every NPG-th row.  A lane takes KPL keys of one group of rows.
        constexpr int KPL = NPG / 4, RPT = GRAN / NPG;   // keys per lane, rows per lane and tile
        typedef T KVec __attribute__((ext_vector_type(KPL)));
        const int kl = KPL * (ft % (32 / KPL)), pg = ft / (32 / KPL);
        float nacc[KPL];
#pragma unroll
        for (int e = 0; e < KPL; e++) nacc[e] = 0.f;
        __syncthreads();   // the tables are there
        __syncthreads();   // tiles 0 and 1 have landed, and the gate rows up to tile 2
        __syncthreads();   // their weights are there
        KVec x[RPT], xn[RPT];
        float wr[RPT], wn[RPT];
        auto request = [&](int st, int t) __attribute__((always_inline)) {   // (stage in bytes)
#pragma unroll
            for (int it = 0; it < RPT; it++) {
                xn[it] = *reinterpret_cast<const KVec*>(smem + st + ZK::off(pg + NPG * it, 32 * vh + kl));
                wn[it] = sw[(t & 3) * 2 * GRAN + GRAN + pg + NPG * it];
            }
        };
        request(0, 0);
        for (int t = 0; t < NTOT; t++) {
#pragma unroll
            for (int it = 0; it < RPT; it++) { x[it] = xn[it]; wr[it] = wn[it]; }
            request(pv.st == (NS - 1) * SB ? 0 : pv.st + SB, t + 1);   // (behind the sequence's last tile what lies there, unused)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int it = 0; it < RPT; it++)
#pragma unroll
                for (int e = 0; e < KPL; e++) nacc[e] = fmaf((float)x[it][e], wr[it], nacc[e]);
            if (__builtin_expect(pv.left == 1, 0)) {   // the step's last tile: the partial sums go to a multiplying wave
                float* const r = red + ((pv.s & 1) * NPG + pg) * 32 + kl;
#pragma unroll
                for (int e = 0; e < KPL; e++) { r[e] = nacc[e]; nacc[e] = 0.f; }
            }
            next(pv, [](int) {});
            __syncthreads();
        }
    } else {
        const int wv = NKB == 2 ? wave : wave >> 1, wk = NKB == 2 ? 0 : wave & 1;   // the wave's 32 values; its (first) 32 keys
        f32x16 acc[NKB], run[NKB];
#pragma unroll
        for (int kb = 0; kb < NKB; kb++)
#pragma unroll
            for (int x = 0; x < 16; x++) { acc[kb][x] = 0.f; run[kb][x] = 0.f; }
        // per-lane byte offsets of the transposing reads (see swz_frag_transposed), contraction step 0; a step further lies 16 tile rows
        // on (the swizzle key has a period of 16 rows)
        const int tj = lane & 15, tsub = (lane >> 4) & 1;
        int koff[NKB][2], voff[2];
#pragma unroll
        for (int hi = 0; hi < 2; hi++) {
#pragma unroll
            for (int kb = 0; kb < NKB; kb++) koff[kb][hi] = ZK::off(4 * h + (tj >> 2) + 8 * hi, 32 * (wk + kb) + 16 * tsub + 4 * (tj & 3));
            voff[hi] = ZV::off(4 * h + (tj >> 2) + 8 * hi, 32 * wv + 16 * tsub + 4 * (tj & 3));
        }
        auto read_tr = [&](const char* base, const int (&off)[2]) __attribute__((always_inline)) {
            s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(base + off[0]));
            s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_PTR(s16x4))(base + off[1]));
            return __builtin_bit_cast(frag, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        };
        constexpr int NSTEP = GRAN / KW;
        static_assert(NSTEP == 4, "two registers of weights");
        struct Weighed { frag hi, lo; };   // (lo: split mode)
        frag kf[NSTEP][NKB], vf[NSTEP];
        Weighed vw;
        // The weights of a tile in two registers: a V fragment holds, for the lane's value, positions 16 s4 + 4 h + (0..3) and
        // 16 s4 + 8 + 4 h + (0..3) as elements 0..7, and element e of step s4 finds its weight in lane 8 (s4 & 1) + e of its row of 16
        // lanes, register s4 / 2 (one DPP operand; as two 16-byte reads per step the weights were a third of all LDS traffic).
        const int wl = lane & 15, wpos = 16 * (wl >> 3) + 4 * h + (wl & 3) + 8 * ((wl >> 2) & 1);
        float wr[2], wnext[2];
        auto request_weights = [&](int t) __attribute__((always_inline)) {
            const float* const wp = sw + (t & 3) * 2 * GRAN + wpos;
            wnext[0] = wp[0];
            wnext[1] = wp[32];
        };
        auto request = [&](int st, int s4) __attribute__((always_inline)) {   // the operands of contraction step s4 of the tile in stage st
            const char* const ks = smem + st * SB;
            vf[s4] = read_tr(ks + KB + KW * s4 * ZV::ROW_BYTES, voff);
#pragma unroll
            for (int kb = 0; kb < NKB; kb++) kf[s4][kb] = read_tr(ks + KW * s4 * ZK::ROW_BYTES, koff[kb]);
        };
        auto weighed = [&](auto s4_tag, const float (&wt)[2]) __attribute__((always_inline)) {
            constexpr int s4 = decltype(s4_tag)::value, l0 = 8 * (s4 & 1);
            float x[8];
            unpack8<T>(__builtin_bit_cast(u32x4, vf[s4]), x);
            const float wv4 = wt[s4 >> 1];
            auto weight = [&](auto e) __attribute__((always_inline)) {   // row_newbcast
                return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, wv4), 0x150 + l0 + decltype(e)::value, 0xf, 0xf, true));
            };
            static_for<8>([&](auto e) __attribute__((always_inline)) { x[decltype(e)::value] *= weight(e); });
            struct Pair { V4 lo, hi; } p, rest;
            Weighed out{};
            if constexpr (STRICT) {
                R::cvt4_split(f32x4{x[0], x[1], x[2], x[3]}, p.lo, rest.lo);
                R::cvt4_split(f32x4{x[4], x[5], x[6], x[7]}, p.hi, rest.hi);
                out.lo = __builtin_bit_cast(frag, rest);
            } else {
                p.lo = R::cvt4(f32x4{x[0], x[1], x[2], x[3]});
                p.hi = R::cvt4(f32x4{x[4], x[5], x[6], x[7]});
            }
            out.hi = __builtin_bit_cast(frag, p);
            return out;
        };
        const int vg = VW * vh + 32 * wv + c32;        // the lane's value
        const int krow0 = 64 * kq + 32 * wk + 8 * h;   // state row of its first key: that of key 32 kb + 8 g4 + 4 h lies 32 kb + 16 (g4 / 2) + 4 (g4 % 2) on
        const size_t hbase = (size_t)bh * NCS * D * D, toff = hbase + (size_t)state_row(vg) * D + 64 * kq + 32 * wk + 4 * h;
        const unsigned odd = lane & 1, sel = odd ? 0x03020706u : 0x05040100u;
        T* const dst_t = reinterpret_cast<T*>(a.CstT) + toff;
        T* const dst_k = reinterpret_cast<T*>(a.Cst) + hbase + (size_t)(krow0 + odd) * D + (vg & ~1);
        // (low-order terms: as far behind the others as the arrays are apart)
        const ptrdiff_t t_lo = STRICT && VM ? reinterpret_cast<T*>(a.CstT_lo) - reinterpret_cast<T*>(a.CstT) : 0;
        const ptrdiff_t k_lo = STRICT && KM ? reinterpret_cast<T*>(a.Cst_lo) - reinterpret_cast<T*>(a.Cst) : 0;
        const ptrdiff_t o_lo = STRICT && DOT ? reinterpret_cast<const T*>(a.dot_with_lo) - reinterpret_cast<const T*>(a.dot_with) : 0;
        const T* const other = reinterpret_cast<const T*>(a.dot_with) + toff;
        V4 y[DOT ? NKB : 1][4], yl[DOT && STRICT ? NKB : 1][4];
        float nrun = 0.f;
        auto carry_vector = [&](int s) __attribute__((always_inline)) {   // by one wave, behind the barrier that follows the step's last tile
            float sum = 0.f;
#pragma unroll
            for (int g = 0; g < NPG; g++) sum += red[((s & 1) * NPG + g) * 32 + c32];
            nrun = nrun * tgam[s] + sum;
            if (h == 0) a.Nst[((size_t)bh * NCS + state_of(s)) * D + 64 * kq + 32 * vh + c32] = nrun;
        };
        __syncthreads();
        __syncthreads();
        __syncthreads();   // tiles 0 and 1 have landed and their weights are there
        request(0, 0);
        request(0, 1);
        request_weights(0);
        wr[0] = wnext[0]; wr[1] = wnext[1];
        vw = weighed(std::integral_constant<int, 0>{}, wr);
        int st = 0, t = 0;
        for (int s = 0; s < NCS; s++) {
            const int nt = s == 0 ? NT0 : NT;
            const size_t so = (size_t)state_of(s) * D * D;
            if (s > 0 && wave == 3) carry_vector(s - 1);
            if constexpr (DOT) {   // (used at the end of the step)
#pragma unroll
                for (int kb = 0; kb < NKB; kb++)
#pragma unroll
                    for (int g4 = 0; g4 < 4; g4++) {
                        y[kb][g4] = *reinterpret_cast<const V4*>(other + so + 32 * kb + 8 * g4);
                        if constexpr (STRICT) yl[kb][g4] = *reinterpret_cast<const V4*>(other + o_lo + so + 32 * kb + 8 * g4);
                    }
            }
            for (int tt = 0; tt < nt; tt++) {
                const int stn = st + 1 == NS ? 0 : st + 1;
                static_for<NSTEP>([&](auto tag) __attribute__((always_inline)) {
                    constexpr int s4 = decltype(tag)::value;
                    // (behind the sequence's last tile what lies in the next stage, unused)
                    if constexpr (s4 + 2 < NSTEP) {
                        request(st, s4 + 2);
                    } else {
                        if constexpr (s4 + 2 == NSTEP) request_weights(t + 1);
                        request(stn, s4 + 2 - NSTEP);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int kb = 0; kb < NKB; kb++) R::mma(acc[kb], kf[s4][kb], vw.hi);
                    if constexpr (STRICT) {
#pragma unroll
                        for (int kb = 0; kb < NKB; kb++) R::mma(acc[kb], kf[s4][kb], vw.lo);
                    }
                    if constexpr (s4 + 1 < NSTEP) vw = weighed(std::integral_constant<int, s4 + 1>{}, wr);
                    else vw = weighed(std::integral_constant<int, 0>{}, wnext);
                    __builtin_amdgcn_sched_barrier(0);
                });
                wr[0] = wnext[0]; wr[1] = wnext[1];
                if (tt == nt - 1) {   // the step's state leaves
                    const float gam = tgam[s];
#pragma unroll
                    for (int kb = 0; kb < NKB; kb++) {
                        run[kb] = run[kb] * gam + acc[kb];
#pragma unroll
                        for (int x = 0; x < 16; x++) {
                            asm volatile("" : "+v"(run[kb][x]));   // (see chunk_carry_t_kernel: the fp32 value is fixed before any conversion)
                            acc[kb][x] = 0.f;
                        }
                        float part[4];
#pragma unroll
                        for (int g4 = 0; g4 < 4; g4++) {
                            const f32x4 four = f32x4{run[kb][4 * g4], run[kb][4 * g4 + 1], run[kb][4 * g4 + 2], run[kb][4 * g4 + 3]};
                            V4 hi, lo{};
                            if constexpr (STRICT) R::cvt4_split(four, hi, lo); else hi = R::cvt4(four);
                            if constexpr (VM) {
                                *reinterpret_cast<V4*>(dst_t + so + 32 * kb + 8 * g4) = hi;
                                if constexpr (STRICT) *reinterpret_cast<V4*>(dst_t + t_lo + so + 32 * kb + 8 * g4) = lo;
                            }
                            if constexpr (KM) {   // two keys x two values per dword: a lane of even value stores the first key of a pair, its neighbour the second
                                T* const dk = dst_k + so + (size_t)(32 * kb + 16 * (g4 >> 1) + 4 * (g4 & 1)) * D;
                                auto store_pairs = [&](T* to, const V4& x) __attribute__((always_inline)) {
                                    struct U2 { unsigned k01, k23; };
                                    const U2 own = __builtin_bit_cast(U2, x);
                                    const unsigned n01 = __builtin_amdgcn_mov_dpp((int)own.k01, 0xb1, 0xf, 0xf, false), n23 = __builtin_amdgcn_mov_dpp((int)own.k23, 0xb1, 0xf, 0xf, false);
                                    *reinterpret_cast<unsigned*>(to) = __builtin_amdgcn_perm(n01, own.k01, sel);
                                    *reinterpret_cast<unsigned*>(to + 2 * D) = __builtin_amdgcn_perm(n23, own.k23, sel);
                                };
                                store_pairs(dk, hi);
                                if constexpr (STRICT) store_pairs(dk + k_lo, lo);
                            }
                            if constexpr (DOT) {   // (the states as they are written: in split mode the sums of their terms)
                                f32x4 xs = __builtin_convertvector(hi, f32x4), ys = __builtin_convertvector(y[kb][g4], f32x4);
                                if constexpr (STRICT) { xs += __builtin_convertvector(lo, f32x4); ys += __builtin_convertvector(yl[kb][g4], f32x4); }
                                part[g4] = sum_halves(dot_group(xs, ys));
                            }
                        }
                        if constexpr (DOT) {   // (the tree of dot_group's comment: groups of four keys, then the 32 values)
                            float dot = (part[0] + part[1]) + (part[2] + part[3]);
                            dot += dpp_f<0xb1>(0.f, dot);    // quad_perm 1 0 3 2
                            dot += dpp_f<0x4e>(0.f, dot);    // quad_perm 2 3 0 1
                            dot += dpp_f<0x141>(0.f, dot);   // row_half_mirror
                            dot += dpp_f<0x140>(0.f, dot);   // row_mirror
                            dot += __shfl_xor(dot, 16);
                            if (lane == 0) a.dot_part[((size_t)bh * NCS + state_of(s)) * (D / 32) * (D / 32) + (2 * kq + wk + kb) * (D / 32) + (VW / 32) * vh + wv] = dot;
                        }
                    }
                }
                st = stn;
                t++;
                __syncthreads();
            }
        }
        if (wave == 3) carry_vector(NCS - 1);
    }
#endif
}

// Whether the one-pass kernel serves a launch: a table's worth of states, split mode at D = 256 only, and where nothing asks for one form or the other by how
// full its workgroups leave the chip (one per CU, each as long as its walk).  Rounds of workgroups three quarters full at the least: whatever the number of states.  One round
// that is emptier: up to as many states as it has thirty-twos of workgroups.  us, the two kernels / one pass, forward, forward that keeps states, backward, whole
// passes (bf16; heads x states):
//   D = 256   4 x 3: 31.5, 32.0, 68.8 / 37.3, 39.8, 74.7   8 x 2: 33.2, 33.5, 70.7 / 31.8, 34.0, 68.2   8 x 3: 37.6, 38.3, 76.8 / 38.0, 40.9, 77.5
//             12 x 3: 50.7, 51.8, 105 / 46.8, 49.5, 100   16 x 7: 83.4, 85.1, 191.4 / 89.1, 94.6, 190.8   20 x 3: 64.3, 66.7, 145.5 / 57.8, 61.1, 138.3
//             24 x 7: 119, 127, 297 / 106, 111, 279   32 x 2: 54.0, 55.0, 118 / 43.1, 45.1, 105   32 x 7: 152, 156, 369 / 130, 138, 346
//             36 x 3: 86.0, 87.8, 215 / 96.6, 102, 225   40 x 3: 86.9, 88.9, 244.5 / 89.9, 94.4, 245.3   48 x 7: 226, 239, 541 / 209, 228, 532   64 x 3: 144, 147, 341 / 122, 130, 327
//   D = 128   16 x 2: 29.6, 30.0, 53.5 / 28.7, 29.7, 51.1   16 x 3: 32.6, 33.1, 65.6 / 34.4, 35.6, 67.0   24 x 3: 39.1, 39.8, 91.1 / 38.3, 39.4, 88.7   32 x 7: 62.7, 64.2, 157 / 71.8, 74.1, 160
//             48 x 3: 51.4, 51.7, 122 / 48.6, 49.7, 117   48 x 15: 172, 178, 448 / 169, 179, 446   64 x 2: 42.0, 43.9, 99.9 / 37.0, 38.2, 91.0   64 x 31: 465, 489, 1165 / 434, 454, 1138
//             72 x 7: 126, 131, 336 / 140, 145, 343   96 x 7: 169, 176, 442 / 171, 178, 436   128 x 7: 223, 238, 581 / 211, 221, 567
//   Split mode, D = 256 (two products per fragment, twice the states to write; one round from three eighths full on)   8 x 2: 42.0, 43.4, 89.9 / 42.8, 48.2, 92.6
//             12 x 3: 70.4, 72.5, 148 / 63.6, 70.6, 142   16 x 7: 116, 124, 266 / 127, 143, 280   24 x 7: 172, 194, 406 / 151, 179, 394   32 x 2: 73.1, 78.5, 158 / 59.8, 68.1, 145
//             32 x 7: 207, 231, 491 / 182, 215, 480   64 x 3: 193, 216, 463 / 175, 203, 453    (D = 128 64 x 3: 76.1, 84.2, 212 / 75.6, 82.9, 213   96 x 7: 224, 254, 646 / 237, 267, 664)
int g_state_kernel = 0;   // 0 = the rule, 1 = chunk sums + carry, 2 = one pass where it can serve
template <typename T, int D>
static bool chunk_seq_serves(const ChunkArgs& a, int form) {   // form: see g_state_kernel
    using Cfg = SeqCfg<T, D>;
    if ((a.precise && D == 128) || a.NCS > Cfg::MAX_STEPS || (a.Cst && a.dot_part) || form == 1) return false;
    constexpr long long CUS = 256;
    const long long wgs = (long long)a.BH * Cfg::WPH, rounds = (wgs + CUS - 1) / CUS;
    return form == 2 || 4 * wgs >= 3 * CUS * rounds || (rounds == 1 && 32ll * a.NCS <= wgs && (!a.precise || 8 * wgs >= 3 * CUS));
}
template <typename T, int D, bool STRICT, bool KM, bool VM, bool DOT>
static int launch_chunk_seq_t(const ChunkArgs& a, hipStream_t st) {
    using Cfg = SeqCfg<T, D>;
    if (int rc = no_scratch_once<chunk_seq_kernel<T, D, KM, VM, DOT, STRICT>>()) return rc;
    if (hipError_t e = lds_limit_once<chunk_seq_kernel<T, D, KM, VM, DOT, STRICT>>(160 * 1024); e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((chunk_seq_kernel<T, D, KM, VM, DOT, STRICT>), dim3(a.BH * Cfg::WPH), dim3(512), Cfg::LDS_BYTES, st, a);
    return (int)hipGetLastError();
}
template <typename T, int D, bool STRICT>
static int launch_chunk_seq(const ChunkArgs& a, hipStream_t st) {
    if (a.dot_part) {
        if (!a.CstT || !a.dot_with || STRICT != (a.dot_with_lo != nullptr)) return MLSTM_EINVAL;
        return launch_chunk_seq_t<T, D, STRICT, false, true, true>(a, st);
    }
    if (a.Cst && a.CstT) return launch_chunk_seq_t<T, D, STRICT, true, true, false>(a, st);
    return a.Cst ? launch_chunk_seq_t<T, D, STRICT, true, false, false>(a, st) : launch_chunk_seq_t<T, D, STRICT, false, true, false>(a, st);
}

template <typename T, int D, bool STRICT>
static int launch_chunk_sum(const ChunkArgs& a, hipStream_t st) {
    using Cfg = ChunkCfg<T, D, STRICT>;
    if (a.L > Cfg::MAX_L) return MLSTM_ESHAPE;
    const dim3 grid(a.BH * a.NCS * (D / Cfg::VW));
    // Workgroups of the narrow kernel up to which it is the faster one (us, bf16, chunk_sum_kernel / narrow):
    //   D = 256   32: 15.5 / 7.9   128: 16.2 / 8.4   384: 17.6 / 11.9   640: 18.0 / 16.5   768: 18.3 / 16.9   896: 18.6 / 19.7
    //   D = 128   96: 10.7 / 8.0   192: 11.2 / 8.2   384: 11.3 / 11.8   768: 13.1 / 17.1
    //   D = 256 in split mode   128: 23.2 / 9.8   256: 24.2 / 11.4   512: 24.2 / 19.1   768: 24.9 / 26.7
    using N = ChunkNarrowCfg<T, STRICT>;
    const int narrow = a.BH * a.NCS * (D / N::W) * (D / N::W);
    if (a.L == N::L && narrow <= (D == 128 ? 256 : (STRICT ? 512 : 768))) {
        if (hipError_t e = lds_limit_once<chunk_sum_narrow_kernel<T, D, STRICT>>((int)N::LDS_BYTES); e != hipSuccess) return (int)e;
        hipLaunchKernelGGL((chunk_sum_narrow_kernel<T, D, STRICT>), dim3(narrow), dim3(256), N::LDS_BYTES, st, a);
        return 0;
    }
    const size_t lds = Cfg::TILE_BYTES + 2 * (size_t)a.L * sizeof(float);
    // (the unrolled variant of split mode at D = 256 does not fit the 256 registers of a wave and would spill)
    constexpr bool UNROLLED_FITS = !(STRICT && D == 256);
    if (UNROLLED_FITS && a.L == 8 * GRAN) {   // the default chunk length
        constexpr int NTT = UNROLLED_FITS ? 8 : 0;
        if (hipError_t e = lds_limit_once<chunk_sum_kernel<T, D, NTT, STRICT>>(160 * 1024); e != hipSuccess) return (int)e;
        hipLaunchKernelGGL((chunk_sum_kernel<T, D, NTT, STRICT>), grid, dim3(512), lds, st, a);
    } else {
        if (hipError_t e = lds_limit_once<chunk_sum_kernel<T, D, 0, STRICT>>(160 * 1024); e != hipSuccess) return (int)e;
        hipLaunchKernelGGL((chunk_sum_kernel<T, D, 0, STRICT>), grid, dim3(512), lds, st, a);
    }
    return 0;
}

// 16-bit D = 128 and 256: the carry in blocks of 32 x 32, sixteen steps per trip to memory, or in blocks of 64 x 64, a trip per
// step but rows of 128 bytes.  The second moves memory faster where it fills the chip and the states are few; otherwise it is its trips
// one after the other.  Workgroups of the second form, states: both carries of a training step in us, 64 x 64 / 32 x 32 (bf16):
//   D = 128   64, 4: 21.3 / 11.1    128, 7: 33.8 / 20.8   192, 7: 37.7 / 24.9   256, 4: 24.4 / 25.1   256, 7: 39.0 / 31.2   256, 15: 99.8 / 54.1
//             256, 31: 207 / 118    512, 7: 61.2 / 53.7   512, 15: 122 / 112    512, 31: 240 / 213
//   D = 256   192, 3: 16.3 / 13.8   256, 3: 16.6 / 17.9   256, 7: 35.6 / 30.0   256, 15: 72.9 / 52.2  384, 7: 45.5 / 42.9   512, 3: 22.5 / 33.8
//             512, 7: 50.8 / 52.6   512, 15: 128 / 116    512, 31: 248 / 236    1024, 15: 195 / 228
static bool carry_in_small_blocks(const ChunkArgs& a, int D) {
    const int wgs = a.BH * (D / 64) * (D / 64);
    return wgs <= 192 || (wgs <= 384 && a.NCS >= 6) || (wgs <= 512 && a.NCS >= 12);
}

template <typename T, int D>
static int launch_chunk_carry_small(const ChunkArgs& a, hipStream_t st) {
    const dim3 cgrid((D / 32) * (D / 32), a.BH);
    if (a.dot_part && a.dot_with_lo) hipLaunchKernelGGL((chunk_carry_small_kernel<T, D, 2>), cgrid, dim3(256), 0, st, a);
    else if (a.dot_part) hipLaunchKernelGGL((chunk_carry_small_kernel<T, D, 1>), cgrid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((chunk_carry_small_kernel<T, D, 0>), cgrid, dim3(256), 0, st, a);
    return (int)hipGetLastError();
}

template <typename T, int D>
static int launch_chunk_t(const ChunkArgs& a, hipStream_t st) {
    if (a.precise && ((a.Cst && !a.Cst_lo) || (a.CstT && !a.CstT_lo))) return MLSTM_EINVAL;
    const int form = g_state_kernel;
    if (chunk_seq_serves<T, D>(a, form)) {
        int rc;
        if constexpr (D == 256) rc = a.precise ? launch_chunk_seq<T, D, true>(a, st) : launch_chunk_seq<T, D, false>(a, st);
        else rc = launch_chunk_seq<T, D, false>(a, st);
        // (not launched because the compiler gave the kernel scratch memory: the two kernels give the same bits; refused only where the form is named)
        if (rc != MLSTM_EBUILD || form == 2) return rc;
    }
    if (int rc = a.precise ? launch_chunk_sum<T, D, true>(a, st) : launch_chunk_sum<T, D, false>(a, st)) return rc;
    // one carry kernel: the value-major one writes both layouts and the vector states
    if (a.dot_part && !(a.CstT && a.dot_with)) return MLSTM_EINVAL;
    // (the variants of the value-major carry: with the contraction, with the key-major copy, with neither; both at once do
    // not fit the registers of four workgroups per CU, and nothing asks for both)
    if (a.CstT && a.dot_part && a.Cst) return MLSTM_EINVAL;
    if (carry_in_small_blocks(a, D)) return launch_chunk_carry_small<T, D>(a, st);
    const dim3 cgrid((D / 64) * (D / 64), a.BH);
    if (a.CstT && a.dot_part) hipLaunchKernelGGL((chunk_carry_t_kernel<T, D, true, false>), cgrid, dim3(256), 0, st, a);
    else if (a.CstT && a.Cst) hipLaunchKernelGGL((chunk_carry_t_kernel<T, D, false, true>), cgrid, dim3(256), 0, st, a);
    else if (a.CstT) hipLaunchKernelGGL((chunk_carry_t_kernel<T, D, false, false>), cgrid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((chunk_carry_kernel<T, D>), dim3(D * D / 8 / 256, a.BH), dim3(256), 0, st, a);
    return (int)hipGetLastError();
}

// the small shapes: sums straight from memory, one carry for both layouts and the contraction
template <typename T, int D>
static int launch_chunk_small(const ChunkArgs& a, hipStream_t st) {
    if (a.precise && ((a.Cst && !a.Cst_lo) || (a.CstT && !a.CstT_lo))) return MLSTM_EINVAL;
    if (!a.precise && (a.Cst_lo || a.CstT_lo)) return MLSTM_EINVAL;
    if (a.dot_part && !(a.CstT && a.dot_with)) return MLSTM_EINVAL;
    if (a.NCS > 1024) return MLSTM_ESHAPE;
    if constexpr (std::is_same<T, __bf16>::value) {   // (other chunk lengths, which only mlstm_set_chunk_length asks for, go to the kernel below)
        using C = ChunkTermsCfg;
        if (a.L == C::L && !a.precise) {
            if (hipError_t e = lds_limit_once<chunk_sum_terms_kernel>((int)C::LDS_BYTES); e != hipSuccess) return (int)e;
            hipLaunchKernelGGL(chunk_sum_terms_kernel, dim3(a.BH * a.NCS), dim3(256), C::LDS_BYTES, st, a);
            return launch_chunk_carry_small<T, D>(a, st);
        }
    }
    hipLaunchKernelGGL((chunk_sum_small_kernel<T, D>), dim3(a.BH * a.NCS * (D / 32)), dim3(256), 0, st, a);
    return launch_chunk_carry_small<T, D>(a, st);
}

// Sum of dD over all pairs (query behind the end of chunk c, key up to it): the forward state at that boundary
// contracted with the reverse state, <C~_c, E_c> + n~_c . g_c.  Rounding errors of the two matrices' 16-bit entries
// average out over the D^2 products.
template <typename T>
__global__ __launch_bounds__(1024) void anchor_kernel(const T* __restrict__ A, const T* __restrict__ B, const T* __restrict__ Al,
                                                     const T* __restrict__ Bl, const float* __restrict__ va, const float* __restrict__ vb,
                                                     float* __restrict__ anchor, int D, int NCS) {
    __shared__ float part[16];
    const int c = blockIdx.x, bh = blockIdx.y, tid = threadIdx.x;
    const size_t base = ((size_t)bh * NCS + c) * D * D;
    typedef T V8 __attribute__((ext_vector_type(8)));
    float acc = 0.f;
    for (int e = 8 * tid; e < D * D; e += 8 * 1024) {
        f32x8 x = __builtin_convertvector(*reinterpret_cast<const V8*>(A + base + e), f32x8);
        f32x8 y = __builtin_convertvector(*reinterpret_cast<const V8*>(B + base + e), f32x8);
        if (Al) {   // split mode: both states as hi + lo (the sums are exact in fp32: 8 + 8 significant bits at most)
            x += __builtin_convertvector(*reinterpret_cast<const V8*>(Al + base + e), f32x8);
            y += __builtin_convertvector(*reinterpret_cast<const V8*>(Bl + base + e), f32x8);
        }
        acc += ((x[0] * y[0] + x[1] * y[1]) + (x[2] * y[2] + x[3] * y[3])) + ((x[4] * y[4] + x[5] * y[5]) + (x[6] * y[6] + x[7] * y[7]));
    }
    if (tid < D) acc += va[((size_t)bh * NCS + c) * D + tid] * vb[((size_t)bh * NCS + c) * D + tid];
    acc = wave_scan_inclusive<OpAdd>(acc);
    if ((tid & 63) == 63) part[tid >> 6] = acc;
    __syncthreads();
    // (both states carry the factor 1 / sqrt(D) of the scores; dD has it once)
    if (tid == 0) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < 16; w++) sum += part[w];
        anchor[(size_t)bh * NCS + c] = sum * sqrtf((float)D);
    }
}

int launch_anchor(int dtype, int D, const void* A, const void* B, const void* A_lo, const void* B_lo, const float* va, const float* vb,
                  float* anchor, int BH, int NCS, hipStream_t st) {
    if ((A_lo == nullptr) != (B_lo == nullptr)) return MLSTM_EINVAL;
    if (dtype == MLSTM_BF16)
        hipLaunchKernelGGL(anchor_kernel<__bf16>, dim3(NCS, BH), dim3(1024), 0, st, (const __bf16*)A, (const __bf16*)B, (const __bf16*)A_lo,
                           (const __bf16*)B_lo, va, vb, anchor, D, NCS);
    else if (dtype == MLSTM_F16)
        hipLaunchKernelGGL(anchor_kernel<_Float16>, dim3(NCS, BH), dim3(1024), 0, st, (const _Float16*)A, (const _Float16*)B,
                           (const _Float16*)A_lo, (const _Float16*)B_lo, va, vb, anchor, D, NCS);
    else if (dtype == MLSTM_F32)
        hipLaunchKernelGGL(anchor_kernel<float>, dim3(NCS, BH), dim3(1024), 0, st, (const float*)A, (const float*)B, (const float*)A_lo,
                           (const float*)B_lo, va, vb, anchor, D, NCS);
    else return MLSTM_ESHAPE;
    return (int)hipGetLastError();
}

int launch_chunk_states(int dtype, int D, const ChunkArgs& a, hipStream_t st) {
    // NCS complete chunks, and at least one position behind them
    if (a.NCS <= 0 || a.L % 128 != 0 || (size_t)a.L * a.NCS >= (size_t)a.S || (size_t)a.L * (a.NCS + 1) < (size_t)a.S) return MLSTM_EINVAL;
    if (dtype == MLSTM_BF16 && D == 128) return launch_chunk_t<__bf16, 128>(a, st);
    if (dtype == MLSTM_BF16 && D == 256) return launch_chunk_t<__bf16, 256>(a, st);
    if (dtype == MLSTM_F16 && D == 128) return launch_chunk_t<_Float16, 128>(a, st);
    if (dtype == MLSTM_F16 && D == 256) return launch_chunk_t<_Float16, 256>(a, st);
    if (dtype == MLSTM_BF16 && D == 64) return launch_chunk_small<__bf16, 64>(a, st);
    if (dtype == MLSTM_F16 && D == 64) return launch_chunk_small<_Float16, 64>(a, st);
    if (dtype == MLSTM_F32 && D == 64) return launch_chunk_small<float, 64>(a, st);
    if (dtype == MLSTM_F32 && D == 128) return launch_chunk_small<float, 128>(a, st);
    return MLSTM_ESHAPE;
}

int set_state_kernel(int variant) {
    if (variant < 0 || variant > 2) return MLSTM_EINVAL;
    g_state_kernel = variant;
    return 0;
}

}  // namespace mlstm
