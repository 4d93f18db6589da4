// sLSTM cell, forward and backward, fp32.  The reference lists the cell as an open item (README.md:9) and holds no code for
// it; this implements the published cell (Beck et al., "xLSTM: Extended Long Short-Term Memory", arXiv:2405.04517,
// section 2.2, with the stabilised exponential gating of appendix A.2), per head (block-diagonal recurrent matrices):
//     i~, f~, z~, o~ = Wx_t[g] + R_g h_{t-1} + b_g
//     m_t  = max(log f_t + m_{t-1}, i~)                 log f_t = f~ (exponential gate) or logsigmoid(f~)
//     i'_t = exp(i~ - m_t),  f'_t = exp(log f_t + m_{t-1} - m_t)
//     c_t  = f'_t c_{t-1} + i'_t tanh(z~),  n_t = f'_t n_{t-1} + i'_t,  h_t = sigmoid(o~) c_t / n_t
// The recurrence through h makes the cell sequential in t, so the kernels are latency machines, not throughput ones: one
// workgroup per (batch, head) walks the sequence with the head's four recurrent matrices in registers.
//   slstm_forward_kernel   eight lanes per two units, each with an eighth of the units' rows of all four R_g: partial
//                          pre-activations from h_{t-1} (LDS), one gate's sum per lane; every lane then updates the cell of its
//                          unit.  Gate values and (c, n, m) are kept for the backward.  Helper waves bring the inputs and write the outputs.
//   slstm_backward_kernel  back through time: rows of 16 lanes form R^T delta_{t+1} for their four units (a sixteenth of the
//                          gradient vector per lane, summed over the row), which is what step t+1 sent back to h_t; the
//                          lanes of a unit's quad turn (dh_t + that, dc, dn) into one pre-activation gradient each (= dWx_t).
//                          Helper waves form the factors of that from the saved values and write dWx out.
//                          The stabiliser m is a common scale of c and n that h does not depend on, so it is held constant.
//   slstm_dr_kernel        dR_g = sum_{b,t} dWx_t[g] h_{t-1}^T and db_g = sum_{b,t} dWx_t[g]: off the sequential path, in
//                          slices of (b, t) whose partial sums a second kernel adds in a fixed order.
// Layouts: wx, dwx [B,S,4,NH,DH] (gates i, f, z, o); r, dr [NH,4,DH,DH] (r[h][g][j][k]: unit j from unit k); b, db [NH,4,DH];
// h, dh [B,S,NH,DH]; saved [B,S,7,NH,DH] (i~, log f, tanh(z~), sigmoid(o~), c, n, m).
#include <hip/hip_runtime.h>
#include <stddef.h>
#include "../../include/mlstm_hip.h"
#include "mlstm_device.h"
#include "mlstm_kernels.h"

namespace slstm {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// The nonlinearities from the hardware's exp2 / reciprocal (a few instructions each, relative error around 1e-6): they sit
// on the critical path of every step of a sequential kernel.
__device__ __forceinline__ float fast_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896340736f); }
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// Inputs of a step come from memory several steps ahead, as direct-to-LDS loads into a ring (a trip to memory is several
// steps long, and a step must not wait for one).  The loads are issued and waited for by hand, by helper waves that issue at least a known
// number of memory operations in every interval between two barriers, in the same order, so that
// "the loads of step t have landed" is a counted wait -- memory operations of a wave complete in the order issued, and a count that is
// too low only waits for more.  The helpers' own code has only stores besides, for which the compiler places no waits.  (Left to the
// compiler, ordinary loads into a ring of registers ended in a wait for everything at every step.)
constexpr int PF = 8;
// (a row's address is uniform, the lane's place in it an offset in bytes)
__device__ __forceinline__ void ring_load(const float* row, unsigned lane_off, unsigned lds_off) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(lane_off), "s"(row), "s"(lds_off) : "memory", "m0");
}

// Sum over the four lanes of a quad (lanes 4a .. 4a+3), the same bits in all four: two exchanges inside the quad.
template <int CTRL>
__device__ __forceinline__ float quad_perm(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float quad_sum(float x) {
    x += quad_perm<0xB1>(x);   // lanes 1, 0, 3, 2
    x += quad_perm<0x4E>(x);   // lanes 2, 3, 0, 1
    return x;
}
// the value of lane q of a quad (three selects; is0..is2: q == 0, 1, 2)
__device__ __forceinline__ float pick(bool is0, bool is1, bool is2, float a, float b, float c, float d) {
    float x = is2 ? c : d;
    x = is1 ? b : x;
    return is0 ? a : x;
}

// A quad of lanes owns a unit j, an octet two of them: lane p of the octet keeps, for all four gates of both units, part p (an
// eighth) of their rows of R_g and forms its part of the eight pre-activations from its part of h_{t-1}.  Lane q of a quad holds
// gate q ^ s of its own unit, and q ^ 3 ^ s of the other, as its s-th, so that seven exchanges with an add each (the octet's mirror
// image, then the quad) leave the whole sum of gate q in lane q, which adds the input last; it applies that gate's nonlinearity
// (one exp2, one reciprocal, one logarithm serve the three kinds side by side), the quad exchanges the four results -- i~ before there is an
// exponential, each from where it is formed, so that the selects that make one value per lane of them are needed for the saved state alone --
// and every lane updates the cell, all four alike (c, n, m are kept four times, the same bits).  A step has no hand-over between waves but h itself: one LDS write,
// one barrier (h in two buffers, taken in turns).
// What bounds it is the serial chain of a step, 300 ns or some 720 cycles (DH = 64): the trip of h through LDS and the barrier about
// 250, 64 multiply-adds at 4 cycles on the one wave of a SIMD, the gates 200.  Eighths and not quarters because the LDS reads of
// h (32 DH floats a step) were the longest part of that trip.  Row broadcasts in the place of wide LDS reads were
// slower (DH = 128: 831 to 889 us): a broadcast, alone or as an operand of the multiply-add, costs as much as one.
// Global memory belongs to helper waves: they bring the steps' inputs into a ring, PF steps ahead, and write out what a step keeps, which the
// walk leaves in LDS in the NEXT step, while that waits for h.  With its own stores and ring loads in that place a step issued 28 instructions
// there, more than the wait hides.
// Forward, B16 NH4, us, quarters / eighths / helpers: DH = 64, S = 2048 716 / 690 / 613; DH = 128, S = 1024 627 / 559 / 553 (545 without the saved state); DH = 32,
// S = 1024 285 / 281 / 246.  DH = 32, eighths / helpers, by workgroups: 256, S = 300 85 / 75; 512, S = 200 70.2 / 71.5 (two on a CU, the helpers of either on a
// SIMD with a walk of the other); 1024 110 / 84.
// With selects before the exchange / the exchange straight from the gates, without the saved state: DH = 64 614 / 602, DH = 128 537 / 530, DH = 32 245 / 240 and by
// workgroups (256, S = 300; 512, 200; 1024, 100) 74.5 / 72.8, 71.1 / 67.4, 38.6 / 36.6; with it 617 / 610, 558 / 549, 246 / 242 and 75.6 / 74.6, 71.9 / 70.6, 39.8 / 39.4.
// (The input as the first term of its lane's sum would save the add at the end, 4, 11 and 2 us of these, and round every multiply-add behind it at the
// size of the whole pre-activation: its error by root mean square 1.9, 2.3 and 2.9 times as large at DH = 32, 64 and 128.)
template <int DH>
struct FwdCfg {
    static constexpr int UW = DH > 64 ? DH / 64 : 1;   // helper waves: a 16-byte piece of a step's input per lane
    static constexpr int THREADS = 4 * DH + 64 * UW;
};
// WIDE: wx, h and saved are on 16-byte boundaries (their rows then are, too)
template <int DH, bool SAVE, bool FS, bool WIDE>
__global__ __launch_bounds__(FwdCfg<DH>::THREADS) void slstm_forward_kernel(const float* __restrict__ wx, const float* __restrict__ r,
                                                                            const float* __restrict__ bias, float* __restrict__ h,
                                                                            float* __restrict__ saved, int NH, int S) {
    using Cfg = FwdCfg<DH>;
    constexpr int KP = DH / 8, KS = KP < 16 ? KP : KP + 4;   // a part of h, and its place in LDS (eight parts, no bank twice)
    constexpr int SR = DH + 16;                              // a row of `stage` (the four rows that a wave writes: no bank twice)
    __shared__ __attribute__((aligned(16))) float hs[2][8 * KS];
    __shared__ __attribute__((aligned(16))) float ring[PF][4 * DH];             // wx of the next PF steps: [slot][unit / 4][gate][unit % 4]
    __shared__ __attribute__((aligned(16))) float stage[SAVE ? 2 : 1][SAVE ? 8 * SR : 4];   // [step mod 2][i~, log f, z, o, c, n, m, unused][unit]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = blockIdx.x / NH, hd = blockIdx.x % NH;
    const size_t step_wx = (size_t)4 * NH * DH, step_h = (size_t)NH * DH, step_s = (size_t)7 * NH * DH;
    for (int e = tid; e < 8 * KS; e += Cfg::THREADS) hs[0][e] = 0.f;
    // Interval t lies between barriers t + 1 and t + 2 (the walk reads the first input between barriers 0 and 1); the walk's step t is in it.  Step t
    // takes h_{t-1} from hs[t & 1] and leaves h_t in the other; it writes what step t - 1 keeps to stage[(t - 1) & 1] and reads its successor's input
    // from the ring.
    if (wave < 4 * DH / 64) {
        const int j = tid >> 2, q = tid & 3, p = tid & 7;
        const bool is0 = q == 0, is1 = q == 1, is2 = q == 2;
        float ro[4][KP], rx[4][KP];   // part p of the rows of the own unit, [s: gate q ^ s], and of the octet's other one, [s: gate q ^ 3 ^ s]
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const float* own = r + (((size_t)hd * 4 + (q ^ s)) * DH + j) * DH + p * KP;
            const float* oth = r + (((size_t)hd * 4 + (q ^ 3 ^ s)) * DH + (j ^ 1)) * DH + p * KP;
#pragma unroll
            for (int k = 0; k < KP; k += 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(own + k), w = *reinterpret_cast<const f32x4*>(oth + k);
#pragma unroll
                for (int e = 0; e < 4; e++) { ro[s][k + e] = v[e]; rx[s][k + e] = w[e]; }
            }
        }
        const float bq = bias[((size_t)hd * 4 + q) * DH + j];
        // the gate's nonlinearity: e = exp2(coef |x|) (sigmoid: of x itself)
        const float coef = is2 ? -2.0f * 1.44269504088896340736f : -1.44269504088896340736f;
        const unsigned sign_off = q == 3 ? 0xffffffffu : 0x7fffffffu;
        const int h_at = j / KP * KS + j % KP, in_at = (j >> 2) * 16 + q * 4 + (j & 3), keep_at = q * SR + j;
        // (the stabiliser starts at -inf rather than the paper's 0: with c_0 = n_0 = 0 it only sets the scale of the first
        // step, and this way the first input gate is exp(0) whatever the first forget gate says)
        float c = 0.f, n = 0.f, m = -INFINITY, val = 0.f;
        auto keep = [&](int slot) __attribute__((always_inline)) {   // what a step keeps, from the registers it left it in
            if constexpr (SAVE) {
                stage[slot][keep_at] = val;
                stage[slot][keep_at + 4 * SR] = pick(is0, is1, true, c, n, m, m);
            }
        };
        __syncthreads();
        float wv = ring[0][in_at];
        __syncthreads();   // (its place may be refilled; every later one is read an interval ahead of that)
        auto step = [&](int u) __attribute__((always_inline)) {   // u = t mod PF
            const float* hcur = hs[u & 1] + p * KS;   // (PF is even: the buffers alternate across rounds too)
            constexpr int AHEAD = KP / 4 < 4 ? KP / 4 : 2;   // (reads under way: DH = 128 has registers for no more)
            f32x4 hv[KP / 4];
#pragma unroll
            for (int k = 0; k < AHEAD; k++) hv[k] = *reinterpret_cast<const f32x4*>(hcur + 4 * k);
            __builtin_amdgcn_sched_barrier(0);
            keep((u & 1) ^ 1);   // (at t = 0 nothing that is read)
            const float in = wv + bq;
            wv = ring[(u + 1) % PF][in_at];
            __builtin_amdgcn_sched_barrier(0);
            float a[4] = {0.f, 0.f, 0.f, 0.f}, x4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KP / 4; k++) {
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int s = 0; s < 4; s++) {
                        a[s] += ro[s][4 * k + e] * hv[k][e];
                        x4[s] += rx[s][4 * k + e] * hv[k][e];
                    }
                if (k + AHEAD < KP / 4) {   // (the sums so far are formed before the next read is issued)
                    asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(x4[0]), "+v"(x4[1]), "+v"(x4[2]), "+v"(x4[3]));
                    __builtin_amdgcn_sched_barrier(0);
                    hv[k + AHEAD] = *reinterpret_cast<const f32x4*>(hcur + 4 * (k + AHEAD));
                }
            }
            // own unit: what the octet's mirror lane (7 - p, of gate q ^ 3) has of it, then gate q from lanes q, q ^ 1, q ^ 2, q ^ 3
#pragma unroll
            for (int s = 0; s < 4; s++) a[s] += quad_perm<0x141>(x4[s]);   // row_half_mirror
            // (what the other lanes need goes to them as each lane has it, whether it is that lane's gate or not; the selects are off the chain)
            const float x = ((a[0] + quad_perm<0xB1>(a[1])) + (quad_perm<0x4E>(a[2]) + quad_perm<0x1B>(a[3]))) + in;
            const float it = quad_perm<0x00>(x);
            const float e = __builtin_amdgcn_exp2f(coef * __builtin_bit_cast(float, __builtin_bit_cast(unsigned, x) & sign_off));
            const float d = 1.0f + e, rd = fast_rcp(d);
            const float th = __builtin_copysignf((1.0f - e) * rd, x);                                                  // tanh
            const float ls = FS ? fmaf(__builtin_amdgcn_logf(d), -0.69314718055994530942f, fminf(x, 0.0f)) : x;        // log sigmoid
            const float logf = quad_perm<0x55>(ls), z = quad_perm<0xAA>(th), o = quad_perm<0xFF>(rd);
            val = pick(is0, is1, is2, x, ls, th, rd);   // i~, log f, z, o (here: with the other selects, where the step waits for h, it costs 20 us of 600)
            const float fm = logf + m, mn = fmaxf(fm, it);
            const float ip = fast_exp(it - mn), fp = fast_exp(fm - mn);
            n = fp * n + ip;
            c = fp * c + ip * z;
            m = mn;
            hs[(u & 1) ^ 1][h_at] = o * c * fast_rcp(n);   // (the quad's four lanes write the same bits)
            __syncthreads();
        };
        int t = 0;
        for (; t + PF <= S; t += PF) {
#pragma unroll
            for (int u = 0; u < PF; u++) step(u);
        }
#pragma unroll
        for (int u = 0; u < PF - 1; u++)
            if (t + u < S) step(u);
        keep((S - 1) & 1);
        __syncthreads();
        return;
    }
    // ---- helpers.  In interval t they request input row t + PF, write out h_{t-1} and what step t - 2 keeps, and wait for row t + 2.
    const int hl = tid - 4 * DH, hwave = wave - 4 * DH / 64;
    // Input: piece hl of a row's 4 DH floats is gate hl % 4 of units 4 (hl / 4) ..; without 16-byte boundaries a load brings a float of 64 places.
    constexpr int LOADS = WIDE ? 1 : (4 * DH / Cfg::UW) / 64;
    unsigned in_off[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
        const int piece = WIDE ? hl : 64 * hwave + (64 * i + lane) / 4, e = WIDE ? 0 : lane & 3;
        in_off[i] = 4u * (unsigned)(((piece & 3) * NH + hd) * DH + 4 * (piece >> 2) + e);
    }
    const float* wnext = wx + (size_t)b * S * step_wx;   // the row that is requested next (past the end of the sequence the last one again)
    const unsigned ring_base = __builtin_amdgcn_readfirstlane(mlstm::lds_offset_of(&ring[0][0]) + hwave * 1024);
    int row = 0;
    auto request = [&](int slot) __attribute__((always_inline)) {
        const unsigned at = ring_base + slot * (4 * DH * 4);
        if constexpr (WIDE) {
            if (hl < DH)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(in_off[0]), "s"(wnext), "s"(at) : "memory", "m0");
        } else {
#pragma unroll
            for (int i = 0; i < LOADS; i++) ring_load(wnext, in_off[i], at + 256 * i);
        }
        if (++row < S) wnext += step_wx;
    };
    // Output: 16-byte pieces of the seven rows of the saved state, then of h
    constexpr int PIECES = SAVE ? 2 * DH / (64 * Cfg::UW) : 1, PR = DH / 4;
    const float *from[PIECES], *next[PIECES];   // (of this interval's buffer and of the other)
    char* to[PIECES];
    size_t stride[PIECES];
    bool is_h[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; i++) {
        const int piece = hl + 64 * Cfg::UW * i, v = SAVE ? piece / PR : 7, u4 = 4 * (piece % PR);
        is_h[i] = v == 7;
        if (SAVE && v < 7) {
            from[i] = &stage[0][v * SR + u4];
            next[i] = &stage[SAVE ? 1 : 0][v * SR + u4];
            to[i] = reinterpret_cast<char*>(saved + (size_t)b * S * step_s + ((size_t)v * NH + hd) * DH + u4);
            stride[i] = step_s * 4;
        } else {
            from[i] = &hs[0][u4 / KP * KS + u4 % KP];
            next[i] = &hs[1][u4 / KP * KS + u4 % KP];
            to[i] = reinterpret_cast<char*>(h + (size_t)b * S * step_h + (size_t)hd * DH + u4);
            stride[i] = step_h * 4;
        }
    }
    auto put_out = [&](bool with_state, bool with_h) __attribute__((always_inline)) {   // (once per interval)
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
            if ((is_h[i] ? with_h : with_state) && (SAVE || hl < PR)) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(from[i]);
                if constexpr (WIDE) *reinterpret_cast<f32x4*>(to[i]) = v;
                else {
#pragma unroll
                    for (int e = 0; e < 4; e++) reinterpret_cast<float*>(to[i])[e] = v[e];
                }
                to[i] += stride[i];
            }
            const float* const now = from[i];
            from[i] = next[i];
            next[i] = now;
        }
    };
#pragma unroll 1
    for (int u = 0; u < PF; u++) request(u);
    mlstm::dma_wait();
    __syncthreads();
    __syncthreads();   // the walk has read row 0
    // Rows PF on: row t + 2 was requested in interval t + 2 - PF, and the PF - 2 intervals since have a request each and, from interval 2 on, the stores
    // (without the saved state those of h, of the first helper wave alone): one interval fewer is waited for.  What may stay under way counts only
    // operations that are certain to be issued: the loads are asm, one each, but a piece that is stored float by float need not be four stores (the
    // compiler makes one of 16 bytes of it, which may lie on any boundary of four).  Counted as four the wait never came to bear.
    constexpr int OPS = LOADS + PIECES;
    static_assert((PF - 3) * OPS < 64, "a count that the wait can hold");
    auto wait = [&]() __attribute__((always_inline)) {
        if (SAVE || hwave == 0) mlstm::dma_wait_but<(PF - 3) * OPS>();
        else mlstm::dma_wait_but<(PF - 3) * LOADS>();
    };
    int t = 0;
    for (; t < 2 && t < S; t++) {
        request(t);
        put_out(false, t > 0);
        wait();
        __syncthreads();
    }
    for (int slot = t; t < S; t++) {
        put_out(true, true);
        request(slot);
        slot = (slot + 1) % PF;
        wait();
        __syncthreads();
    }
    put_out(S > 1, true);
    __syncthreads();
    put_out(true, false);
}

// Back through time with the same quads, but what step t + 1 sends back to h_t -- R^T delta_{t+1}, a vector of 4 DH gradients
// against DH outputs -- is formed by rows of 16 lanes: the four quads of a row own four units k, and lane p of the row takes
// a sixteenth of the gradient vector for all four of them (DH / 4 gradients x 4 columns of R: DH registers, DH multiply-adds,
// but only DH / 4 floats of LDS reads where a lane that served one unit alone read DH: the LDS pipeline was what the step
// waited for).  Quad Q of the row holds unit (Q + s) mod 4 as its s-th, so that three rotations with an add each bring a unit's
// sums to its own quad, and the exchange inside the quad finishes them.
// Everything else a step computes is linear in dh_t: with dc, dn what comes back to c_t and n_t, lane q of a quad needs
//     dc = dh A + dc',  dn = dh B + dn',  its gradient = P dc + Q dn  (q = 3: O dh)
// and A, B, P, Q, O are made of saved values only, so that five instructions lie between dh_t and the gradient that is handed on
// (delta in two buffers, taken in turns: one barrier per step).
// What bounded a step was instruction issue: 157 instructions on the one wave of a SIMD, 4 to 5 cycles each, of which only 100 are on
// the chain; the rest -- the factors, the ring of their inputs, the stores -- do not fit behind a trip to LDS of 130 cycles.  They
// belong to waves of their own: helper group g of NGRP, a lane per unit, serves every NGRP-th step, its work spread over the
// intervals between as many barriers, and leaves a step's factors in LDS ahead of it.  (A lane per unit, where each of the quad's
// lanes formed the same factors: the helpers issue a fraction of what they replace.  Work of more than some 250 ns in one
// interval makes the step wait for it: addresses that walk, and 16-byte loads of several rows at a time.)
// Now a step is bounded by R^T delta alone: the same kernel whose helpers only met the barriers took 515 of its 519 us.
// Backward, us, without / with the helpers: B16 NH4, DH = 64, S = 2048 824 / 519; DH = 32, S = 1024 317 / 209; DH = 128, S = 1024
// 682 / 528; 256 and 512 workgroups (DH = 64, S = 500; S = 300) 212 / 144, 172 / 125; DH = 32 at 1024 workgroups and S = 200, where
// 3.6 TB/s are moved, 86.6 / 88.7.
constexpr int BWD_SAVED = 10;   // rows of the saved state that a step's factors are made of: i~, log f, z, o, c, n, m of the step, c, n, m of the one before it in time
template <int DH>
struct BwdCfg {
    static constexpr int UW = DH > 64 ? DH / 64 : 1;      // waves per helper group
    static constexpr int NGRP = DH > 64 ? 2 : 4;
    static constexpr int THREADS = 4 * DH + NGRP * UW * 64;
    static constexpr int RING = 4;                         // jobs of a group under way
    static constexpr int SLOTS = 4;                        // steps whose factors are in LDS
};

// WIDE: saved is on a 16-byte boundary (its rows then are, too): four floats per lane and load
template <int DH, bool FS, bool WIDE>
__global__ __launch_bounds__(BwdCfg<DH>::THREADS) void slstm_backward_kernel(const float* __restrict__ dh, const float* __restrict__ r,
                                                                             const float* __restrict__ saved, float* __restrict__ dwx, int NH,
                                                                             int S) {
    using Cfg = BwdCfg<DH>;
    constexpr int PE = DH / 4;       // gradients per lane: a sixteenth of the 4 DH (in the order unit * 4 + gate)
    constexpr int PS = PE + 4;       // ... and four floats, so that the 16 parts of a row's read start in different banks
    constexpr int UW = Cfg::UW, NGRP = Cfg::NGRP, RING = Cfg::RING, SLOTS = Cfg::SLOTS, UL = DH < 64 ? DH : 64;   // UL: units per helper wave
    constexpr int RPL = WIDE ? 256 / UL : 1, NLOAD = (BWD_SAVED + RPL - 1) / RPL;   // rows per load, loads per job
    static_assert((RING - 2) * (NLOAD + 1) < 64, "a count that the wait can hold");
    struct Lds {   // (what the steps read comes first: within an offset of the instructions)
        float delta[2][16 * PS];             // [buffer][part][unit * 4 + gate within the part]
        float shared_of[SLOTS][DH][4];       // A, B, f', dh of a unit
        float own_of[SLOTS][DH][4][2];       // P, Q of gates 0..2; O
        float ring[NGRP * UW][RING][(BWD_SAVED + 1) * UL];   // of a job: ten rows of the saved state, dh
    };
    __shared__ __attribute__((aligned(16))) Lds lds;
    auto& delta = lds.delta;
    auto& shared_of = lds.shared_of;
    auto& own_of = lds.own_of;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = blockIdx.x / NH, hd = blockIdx.x % NH;
    const size_t step_wx = (size_t)4 * NH * DH, step_h = (size_t)NH * DH, step_s = (size_t)7 * NH * DH;
    for (int e = tid; e < 16 * PS; e += Cfg::THREADS) delta[0][e] = 0.f;   // (nothing comes back to the last step)
    // step n (of S, counted down in time) is row S - 1 - n; its gradients go to buffer (n & 1) ^ 1, its factors lie in slot n % SLOTS
    if (wave < 4 * DH / 64) {
        const int k = tid >> 2, q = tid & 3;
        const int part = tid & 15, k4 = (tid >> 4) * 4;   // the lane's part of the gradient vector; the first of its row's four units
        const int urow = k & 3;                           // which of the row's units is this lane's own
        float rc[PE][4];   // [gradient of the part][s]: R_g[j][k4 + (urow + s) mod 4] for the part's (j, g)
#pragma unroll
        for (int e = 0; e < PE; e++) {
            const int f = part * PE + e, j = f >> 2, g = f & 3;
            const f32x4 v = *reinterpret_cast<const f32x4*>(r + (((size_t)hd * 4 + g) * DH + j) * DH + k4);
#pragma unroll
            for (int s = 0; s < 4; s++) rc[e][s] = pick(urow == 0, urow == 1, urow == 2, v[s], v[(s + 1) & 3], v[(s + 2) & 3], v[(s + 3) & 3]);
        }
        const int mine_at = ((4 * k + q) / PE) * PS + (4 * k + q) % PE;   // where this lane's gradient goes in a delta buffer
        float dc_next = 0.f, dn_next = 0.f;
        __syncthreads();
        auto step = [&](auto u_tag) __attribute__((always_inline)) {
            constexpr int u = decltype(u_tag)::value;
            const float* dcur = delta[u & 1] + part * PS;
            constexpr int AHEAD = PE / 4 < 4 ? PE / 4 : 4;   // (reads under way: DH = 128 has registers for no more)
            f32x4 dl[PE / 4];
#pragma unroll
            for (int e = 0; e < AHEAD; e++) dl[e] = *reinterpret_cast<const f32x4*>(dcur + 4 * e);
            const f32x4 sh = *reinterpret_cast<const f32x4*>(shared_of[u % SLOTS][k]);   // (a quad reads one address)
            const float2 pq = *reinterpret_cast<const float2*>(own_of[u % SLOTS][k][q]);
            __builtin_amdgcn_sched_barrier(0);
            float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < PE / 4; e++) {
#pragma unroll
                for (int f = 0; f < 4; f++)
#pragma unroll
                    for (int x = 0; x < 4; x++) a[x] += rc[4 * e + f][x] * dl[e][f];
                if (e + AHEAD < PE / 4) {   // (the sums so far are formed before the next read is issued)
                    asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]));
                    __builtin_amdgcn_sched_barrier(0);
                    dl[e + AHEAD] = *reinterpret_cast<const f32x4*>(dcur + 4 * (e + AHEAD));
                }
            }
            // (row_ror: lane i takes from lane i - 4s of its row, whose s-th unit is this quad's own)
            const float dhrec = quad_sum((a[0] + quad_perm<0x124>(a[1])) + (quad_perm<0x128>(a[2]) + quad_perm<0x12C>(a[3])));
            const float d_h = sh[3] + dhrec;
            const float dc = fmaf(d_h, sh[0], dc_next), dn = fmaf(d_h, sh[1], dn_next);   // (the shorter way from d_h)
            const float lin = fmaf(dc, pq.x, dn * pq.y);
            delta[(u & 1) ^ 1][mine_at] = q == 3 ? d_h * pq.x : lin;
            dc_next = dc * sh[2];
            dn_next = dn * sh[2];
            mlstm::pin(dc_next); mlstm::pin(dn_next);
            __syncthreads();
        };
        static_assert(SLOTS == 4, "the steps are unrolled by the slots");
        int n = 0;
        for (; n + 4 <= S; n += 4) {
            step(std::integral_constant<int, 0>{});
            step(std::integral_constant<int, 1>{});
            step(std::integral_constant<int, 2>{});
            step(std::integral_constant<int, 3>{});
        }
        if (n < S) { step(std::integral_constant<int, 0>{}); n++; }
        if (n < S) { step(std::integral_constant<int, 1>{}); n++; }
        if (n < S) step(std::integral_constant<int, 2>{});
        return;
    }
    // ---- helpers: job i of a group is step g + NGRP i
    const int hw = wave - 4 * DH / 64, g = hw / UW, u0 = (hw % UW) * 64, unit = u0 + (lane < UL ? lane : 0);
    const bool there = lane < UL;
    const unsigned row_bytes = (unsigned)(step_h * 4), state_bytes = (unsigned)(step_s * 4);   // (from row to row of a state, from state to state)
    const unsigned lane_off = 4u * (unsigned)(hd * DH + unit);
    float* const myring = &lds.ring[hw][0][0];
    const unsigned ring_base = __builtin_amdgcn_readfirstlane(mlstm::lds_offset_of(myring));
    // Rows 0..6 are those of state t, 7..9 rows 4..6 of the state before it; offsets count from that one.  A lane's piece of load l (WIDE: 16 bytes,
    // RPL rows a load) and whether it is of state t.
    constexpr int JOB = (BWD_SAVED + 1) * UL, PIECES = WIDE ? NLOAD : 1, LAST_LANES = (BWD_SAVED - (NLOAD - 1) * RPL) * UL / 4;
    unsigned off[PIECES];
    bool of_t[PIECES];
    if constexpr (WIDE) {
#pragma unroll
        for (int l = 0; l < PIECES; l++) {
            int v = l * RPL + lane / (UL / 4);
            v = v < BWD_SAVED ? v : BWD_SAVED - 1;
            of_t[l] = v < 7;
            off[l] = (unsigned)(v < 7 ? v : v - 3) * row_bytes + (v < 7 ? state_bytes : 0u) + 4u * (unsigned)(hd * DH + u0 + 4 * (lane % (UL / 4)));
        }
    }
    int tf = S - 1 - g;                                                       // the row that is requested next
    const float* sf = saved + ((size_t)b * S + tf - 1) * step_s;              // the state before it (not read where tf < 1)
    const float* df = dh + ((size_t)b * S + tf) * step_h;
    const float* const s_first = saved + (size_t)b * S * step_s;
    const float* const d_first = dh + (size_t)b * S * step_h;
    unsigned at = ring_base;
    auto fetch = [&]() __attribute__((always_inline)) {   // (steps past the last one: row 0; there is no state before that: its own)
        const bool inside = tf >= 1;
        const float* const base = inside ? sf : s_first;
        if constexpr (WIDE) {
#pragma unroll
            for (int l = 0; l < PIECES; l++) {
                const unsigned o = inside || !of_t[l] ? off[l] : off[l] - state_bytes;
                if (l < PIECES - 1 || lane < LAST_LANES)
                    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(o), "s"(base), "s"(at + 1024 * l) : "memory", "m0");
            }
        } else if (there) {
#pragma unroll
            for (int v = 0; v < BWD_SAVED; v++)
                ring_load(base, lane_off + (unsigned)(v < 7 ? v : v - 3) * row_bytes + (v < 7 && inside ? state_bytes : 0u), at + 4 * UL * v);
        }
        if (there) ring_load(tf >= 0 ? df : d_first, lane_off, at + 4 * UL * BWD_SAVED);
        tf -= NGRP;
        sf -= NGRP * step_s;
        df -= NGRP * step_h;
        at = at == ring_base + (RING - 1) * JOB * 4 ? ring_base : at + JOB * 4;
    };
    float in[BWD_SAVED], dht = 0.f;
    auto take = [&](int i) __attribute__((always_inline)) {
        const float* const from = myring + (i & (RING - 1)) * JOB + (there ? lane : 0);
#pragma unroll
        for (int v = 0; v < BWD_SAVED; v++) in[v] = from[v * UL];
        dht = from[BWD_SAVED * UL];
        if (g + NGRP * i >= S - 1) { in[7] = 0.f; in[8] = 0.f; in[9] = -INFINITY; }
    };
    float A = 0.f, B = 0.f, O = 0.f, fp = 0.f, P0 = 0.f, Q0 = 0.f, P1 = 0.f, Q1 = 0.f, P2 = 0.f;
    auto factors = [&]() __attribute__((always_inline)) {
        const float it = in[0], logf = in[1], z = in[2], o = in[3], ct = in[4], nt = in[5], mt = in[6];
        const float ip = fast_exp(it - mt);
        fp = fast_exp(logf + in[9] - mt);
        const float inv_n = fast_rcp(nt), psi = ct * inv_n;
        A = o * inv_n; B = -A * psi; O = psi * o * (1.0f - o);
        // d i~ = (dc z + dn) i',  d f~ = (dc c_{t-1} + dn n_{t-1}) f' (sigmoid gate: sigmoid(-f~) = 1 - exp(log f)),  d z~ = dc i' (1 - z^2)
        const float fs = FS ? fp * (1.0f - fast_exp(logf)) : fp;
        P0 = z * ip; Q0 = ip;
        P1 = in[7] * fs; Q1 = in[8] * fs;
        P2 = ip * (1.0f - z * z);
    };
    auto put = [&](int i) __attribute__((always_inline)) {
        if (there) {
            const int slot = (g + NGRP * i) & (SLOTS - 1);
            *reinterpret_cast<f32x4*>(shared_of[slot][unit]) = f32x4{A, B, fp, dht};
            *reinterpret_cast<f32x4*>(own_of[slot][unit][0]) = f32x4{P0, Q0, P1, Q1};
            *reinterpret_cast<f32x4*>(own_of[slot][unit][2]) = f32x4{P2, 0.f, O, 0.f};
        }
    };
    const int grad_at = (4 * unit / PE) * PS + 4 * unit % PE;
    unsigned gate_off[4];
#pragma unroll
    for (int x = 0; x < 4; x++) gate_off[x] = lane_off + (unsigned)x * row_bytes;
    auto store = [&](int n) __attribute__((always_inline)) {   // the gradients of step n
        const f32x4 v = *reinterpret_cast<const f32x4*>(delta[(n & 1) ^ 1] + grad_at);
        char* const row = reinterpret_cast<char*>(dwx + ((size_t)b * S + (S - 1 - n)) * step_wx);
        if (there) {
#pragma unroll
            for (int x = 0; x < 4; x++) *reinterpret_cast<float*>(row + gate_off[x]) = v[x];
        }
    };
#pragma unroll 1
    for (int i = 0; i < RING; i++) fetch();
    mlstm::dma_wait();
    take(0);
    factors();
    put(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (slot 0 has been read)
    if (g == 0) fetch();
    __syncthreads();
    // Interval n lies between barriers n and n + 1, beside step n.  A group's turn for job i (of step g + NGRP i) begins NGRP intervals ahead: the values
    // out of the ring; the factors; these to LDS, one interval at least before they are read; then the loads of the job RING on, into the same
    // place, and the store of step n - 1.  A job's loads are waited for with those of one job less than are younger still under way (stores
    // only make the wait longer).
    int n = 0;
    for (; n < g && n < S; n++) {   // (the end of the turn whose job 0 is done)
        if (n == g - 1) {
            fetch();
            if (n > 0) store(n - 1);
        }
        __syncthreads();
    }
    for (int job = 1; n < S; job++) {
        mlstm::dma_wait_but<(RING - 2) * (NLOAD + 1)>();
        take(job);
        if constexpr (NGRP == 2) { factors(); put(job); }
        __syncthreads();
        if (++n == S) break;
        if constexpr (NGRP == 4) {
            factors();
            __syncthreads();
            if (++n == S) break;
            put(job);
            __syncthreads();
            if (++n == S) break;
        }
        fetch();
        store(n - 1);
        __syncthreads();
        n++;
    }
    if ((S - g) % NGRP == NGRP - 1 || (S < g && S == g - 1)) store(S - 1);
}

constexpr int dr_parts(int DH) { return DH <= 64 ? 4 : 1; }   // waves that share a slice's pairs (slstm_dr_kernel's PARTS)
constexpr int dr_lds(int DH) { return DH <= 64 ? 4 * (DH * DH + DH) * (int)sizeof(float) : 0; }
// dR[h][g][j][k] and db[h][g][j] over one slice of the (b, t) pairs, on the matrix units: per head and gate this is the
// product of dWx[g] ([pairs] x DH, taken transposed) with h_{t-1} ([pairs] x DH), the pairs being the inner dimension.
// Every fp32 operand is three bf16 terms (mlstm::Tr<float>: 24 significant bits); a lane holds row or column l % 32 at eight
// successive pairs, 8 (l / 32) + e of a round's sixteen, so both
// come straight from global memory, one dword per lane, rows of 128 bytes; nothing passes through LDS.  One workgroup per
// (head, gate, slice), four waves: up to DH = 64 every wave forms the whole DH x DH block over a quarter of the slice's
// pairs (chunks of 16, taken in turns), and the four add up in LDS, a quarter of the block each; at DH = 128 every wave forms one 64 x 64
// quadrant over all the pairs.
// B16 NH4 S2048 DH64: 70 us on v_mfma_f32_32x32x2_f32, bound by its 512 cycles per 32 x 32 x 16 block; 57 on three bf16 terms (192, and the splits),
// with 33 MB of partial sums, one per wave, and a place in the sequence looked up and tested for every load; 46 now that only rounds that meet the start of a
// sequence or the end of the slice do that, and the others load from uniform rows: 134 MB of dWx and four readings of h (by gate, 34 MB each out of the caches).
template <int DH>
__global__ __launch_bounds__(256, 2) void slstm_dr_kernel(const float* __restrict__ dwx, const float* __restrict__ h, float* __restrict__ part_r,
                                                       float* __restrict__ part_b, int B, int NH, int S, int nslice) {
    using mlstm::f32x16;
    constexpr int W = DH < 64 ? DH : 64;   // a wave's block is W x W
    constexpr int T = W / 32;               // in T x T tiles
    constexpr int PARTS = dr_parts(DH);     // waves that share a block, each with its part of the pairs
    constexpr int U = 8, CH = 2 * U;        // pairs per lane and round, pairs per round
    typedef mlstm::Tr<float> X;
    const int hg = blockIdx.x, hd = hg / 4, g = hg % 4, slice = blockIdx.y;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, hh = lane >> 5;
    const int part = PARTS > 1 ? wave : 0, quad = PARTS > 1 ? 0 : wave;
    const int j0 = (quad >> 1) * 64, k0 = (quad & 1) * 64;   // the block's corner
    const long long total = (long long)B * S, per = (total + nslice - 1) / nslice;
    const long long lo = slice * per, hi = lo + per < total ? lo + per : total;
    const size_t step_wx = (size_t)4 * NH * DH, step_h = (size_t)NH * DH;
    // (a lane's place inside a pair of rows, as one 32-bit offset in bytes: the rows' own addresses are the same for the whole wave)
    const unsigned la = 4u * (unsigned)(U * hh * step_wx + ((size_t)g * NH + hd) * DH + j0 + l32);
    const unsigned lb = 4u * (unsigned)(U * hh * step_h + (size_t)hd * DH + k0 + l32);
    auto at = [](const float* row, unsigned off) __attribute__((always_inline)) { return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(row) + off); };
    f32x16 acc[T][T];
    float bsum[T];
#pragma unroll
    for (int x = 0; x < T; x++) {
        bsum[x] = 0.f;
#pragma unroll
        for (int y = 0; y < T; y++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[x][y][e] = 0.f;
    }
    X::frag a[2][T], bv[2][T];
    // the operands of the round that starts at pair p0, t0 steps into its sequence (this lane's first pair: 8 hh on)
    auto load = [&](int set, long long p0, int t0) __attribute__((always_inline)) {
        const float* const ra = dwx + p0 * (long long)step_wx;
        const float* const rb = h + (p0 - 1) * (long long)step_h;
        if (p0 + CH <= hi && t0 > 0 && t0 + CH <= S) {
#pragma unroll
            for (int e = 0; e < U; e++)
#pragma unroll
                for (int x = 0; x < T; x++) {
                    a[set][x][e] = at(ra + e * step_wx + 32 * x, la);
                    bv[set][x][e] = at(rb + e * step_h + 32 * x, lb);
                }
            return;
        }
#pragma unroll
        for (int e = 0; e < U; e++) {
            const long long pp = p0 + U * hh + e;
            int t = t0 + U * hh + e;
            if (t >= S) t %= S;
            const bool in = pp < hi, prev = in && t != 0;   // (h_{-1} = 0: the first step of a sequence adds nothing to dR)
#pragma unroll
            for (int x = 0; x < T; x++) {
                a[set][x][e] = in ? at(ra + e * step_wx + 32 * x, la) : 0.f;
                bv[set][x][e] = prev ? at(rb + e * step_h + 32 * x, lb) : 0.f;
            }
        }
    };
    long long p0 = lo + (long long)part * CH;
    int t0 = (int)(p0 % S);
    if (p0 < hi) load(0, p0, t0);
    // one round on operand set `set` (a constant at each call); the next round's operands are under way while it multiplies
    auto round = [&](int set) __attribute__((always_inline)) {
        const long long pn = p0 + (long long)PARTS * CH;
        int tn = t0 + PARTS * CH;
        if (tn >= S) tn %= S;
        if (pn < hi) load(set ^ 1, pn, tn);
        X::terms ta[T], tb[T];
#pragma unroll
        for (int x = 0; x < T; x++) {
#pragma unroll
            for (int e = 0; e < U; e++) bsum[x] += a[set][x][e];
            ta[x] = X::split(a[set][x]);
            tb[x] = X::split(bv[set][x]);
        }
#pragma unroll
        for (int x = 0; x < T; x++)
#pragma unroll
            for (int y = 0; y < T; y++) X::mma(acc[x][y], ta[x], tb[y]);
        p0 = pn;
        t0 = tn;
    };
    while (p0 < hi) {
        round(0);
        if (p0 >= hi) break;
        round(1);
    }
    // db: a lane's sum covers its half of the pairs (inner index l / 32) for row l % 32
#pragma unroll
    for (int x = 0; x < T; x++) bsum[x] += __shfl_xor(bsum[x], 32);
    // accumulator register e of a lane: column l % 32, row 8 (e / 4) + 4 (l / 32) + e % 4 of its tile
    float* const out = part_r + (((size_t)slice * NH * 4 + hg) * DH) * DH;
    float* const out_b = part_b + ((size_t)slice * NH * 4 + hg) * DH;
    // an element that is not finite, in fp32 multiply-adds straight from memory (see not_finite in mlstm_device.h)
    auto exact = [&](int j, int k) {
        float sum = 0.f;
#pragma unroll 1
        for (long long pp = lo; pp < hi; pp++)
            if (pp % S != 0) sum += dwx[pp * step_wx + ((size_t)g * NH + hd) * DH + j] * h[(pp - 1) * step_h + (size_t)hd * DH + k];
        return sum;
    };
    if constexpr (PARTS > 1) {
        constexpr int Q = T * T * 4, QW = Q / PARTS;   // groups of four registers, of those a wave's to add up
        extern __shared__ __attribute__((aligned(16))) f32x4 sums[];   // [wave][group][lane], then [wave][row]: sums of dWx
        float* const sums_b = reinterpret_cast<float*>(sums + PARTS * Q * 64);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const f32x16& v = acc[q / 4 / T][q / 4 % T];
            const int e = 4 * (q % 4);
            sums[(wave * Q + q) * 64 + lane] = f32x4{v[e], v[e + 1], v[e + 2], v[e + 3]};
        }
        if (hh == 0) {
#pragma unroll
            for (int x = 0; x < T; x++) sums_b[wave * DH + 32 * x + l32] = bsum[x];
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < QW; n++) {
            const int q = wave * QW + n, j = 32 * (q / 4 / T) + 8 * (q % 4) + 4 * hh, k = 32 * (q / 4 % T) + l32;
            const f32x4* const from = sums + q * 64 + lane;
            f32x4 v = (from[0] + from[Q * 64]) + (from[2 * Q * 64] + from[3 * Q * 64]);
            float seen = 0.f;
#pragma unroll
            for (int e = 0; e < 4; e++) seen = mlstm::not_finite(seen, v[e]);
            if (__any(seen != 0.f)) {
#pragma unroll 1
                for (int e = 0; e < 4; e++) out[(size_t)(j + e) * DH + k] = exact(j + e, k);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) out[(size_t)(j + e) * DH + k] = v[e];
            }
        }
        if ((int)threadIdx.x < DH)
            out_b[threadIdx.x] = (sums_b[threadIdx.x] + sums_b[DH + threadIdx.x]) + (sums_b[2 * DH + threadIdx.x] + sums_b[3 * DH + threadIdx.x]);
    } else {
        float seen = 0.f;
#pragma unroll
        for (int x = 0; x < T; x++)
#pragma unroll
            for (int y = 0; y < T; y++)
#pragma unroll
                for (int e = 0; e < 16; e++) seen = mlstm::not_finite(seen, acc[x][y][e]);
        if (__any(seen != 0.f)) {
#pragma unroll 1
            for (int n = lane; n < W * W; n += 64) out[(size_t)(j0 + n / W) * DH + k0 + n % W] = exact(j0 + n / W, k0 + n % W);
        } else {
#pragma unroll
            for (int x = 0; x < T; x++)
#pragma unroll
                for (int y = 0; y < T; y++)
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        out[(size_t)(j0 + 32 * x + 8 * (e / 4) + 4 * hh + e % 4) * DH + k0 + 32 * y + l32] = acc[x][y][e];
        }
        if (k0 == 0 && hh == 0) {
#pragma unroll
            for (int x = 0; x < T; x++) out_b[j0 + 32 * x + l32] = bsum[x];
        }
    }
}

// out[e] = sum over the partial sums, in a fixed order: 64 elements per workgroup and turn, four threads per element with every
// fourth partial sum each, their four sums added in order.  Behind the elements of dR come those of db (a launch of its own: 7 us).  (More than one
// turn only where a workgroup per 64 elements would be more threads than a launch holds.)
struct Reduce { const float* part; float* out; size_t n; };
__global__ __launch_bounds__(256) void slstm_reduce_kernel(Reduce r, Reduce b, int nslice) {
    __shared__ float red[4][64];
    const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
    const size_t wgs = (r.n + 63) / 64, all = wgs + (b.n + 63) / 64;
    for (size_t wg = blockIdx.x; wg < all; wg += gridDim.x) {
        const bool first = wg < wgs;
        const float* const part = first ? r.part : b.part;
        float* const out = first ? r.out : b.out;
        const size_t n = first ? r.n : b.n, e = (first ? wg : wg - wgs) * 64 + x;
        float s0 = 0.f, s1 = 0.f;
        if (e < n) {
            int i = y;
            for (; i + 4 < nslice; i += 8) { s0 += part[(size_t)i * n + e]; s1 += part[(size_t)(i + 4) * n + e]; }
            if (i < nslice) s0 += part[(size_t)i * n + e];
        }
        red[y][x] = s0 + s1;
        __syncthreads();
        if (y == 0 && e < n) out[e] = (red[0][x] + red[1][x]) + (red[2][x] + red[3][x]);
        __syncthreads();
    }
}

int slices_for(int B, int NH, int S) {
    const size_t total = (size_t)B * S;
    size_t n = 512 / ((size_t)NH * 4);   // about two workgroups for each of the 256 compute units
    if (n < 1) n = 1;
    if (n > (total + 255) / 256) n = (total + 255) / 256;   // at least 256 (b, t) pairs per slice
    return (int)(n < 1 ? 1 : n);
}

// A launch holds fewer than 2^32 threads: a batch of more sequences in several, launch(first sequence, how many).
template <typename F>
int over_batch(int B, int NH, int threads, F&& launch) {
    const long long fit = (long long)(0xffffffffu / (unsigned)threads) / NH, most = fit > 1 ? fit : 1;
    for (long long b0 = 0; b0 < B; b0 += most)
        if (int rc = launch(b0, (int)(B - b0 < most ? B - b0 : most))) return rc;
    return 0;
}

// (the step kernels count their waits for the input ring by hand: see no_scratch_once)
template <int DH, bool SAVE, bool FS>
int forward_launch(const float* wx, const float* r, const float* b, float* h, float* saved, int B, int NH, int S, hipStream_t st) {
    auto launch = [&](auto wide) {
        constexpr auto kernel = slstm_forward_kernel<DH, SAVE, FS, decltype(wide)::value>;
        if (int rc = mlstm::no_scratch_once<kernel>()) return rc;
        return over_batch(B, NH, FwdCfg<DH>::THREADS, [&](long long b0, int n) {
            const size_t at = (size_t)b0 * S * NH * DH;
            hipLaunchKernelGGL(kernel, dim3(n * NH), dim3(FwdCfg<DH>::THREADS), 0, st, wx + 4 * at, r, b, h + at, SAVE ? saved + 7 * at : nullptr, NH, S);
            return (int)hipGetLastError();
        });
    };
    const size_t at = reinterpret_cast<size_t>(wx) | reinterpret_cast<size_t>(h) | reinterpret_cast<size_t>(saved);
    return at & 15 ? launch(std::false_type{}) : launch(std::true_type{});
}

template <int DH>
int forward_t(const float* wx, const float* r, const float* b, float* h, float* saved, int B, int NH, int S, int fs, hipStream_t st) {
    if (saved && fs) return forward_launch<DH, true, true>(wx, r, b, h, saved, B, NH, S, st);
    if (saved) return forward_launch<DH, true, false>(wx, r, b, h, saved, B, NH, S, st);
    if (fs) return forward_launch<DH, false, true>(wx, r, b, h, saved, B, NH, S, st);
    return forward_launch<DH, false, false>(wx, r, b, h, saved, B, NH, S, st);
}

template <int DH, bool FS, bool WIDE>
int backward_launch_w(const float* dh, const float* r, const float* saved, float* dwx, int B, int NH, int S, hipStream_t st) {
    if (int rc = mlstm::no_scratch_once<slstm_backward_kernel<DH, FS, WIDE>>()) return rc;
    return over_batch(B, NH, BwdCfg<DH>::THREADS, [&](long long b0, int n) {
        const size_t at = (size_t)b0 * S * NH * DH;
        hipLaunchKernelGGL((slstm_backward_kernel<DH, FS, WIDE>), dim3(n * NH), dim3(BwdCfg<DH>::THREADS), 0, st, dh + at, r, saved + 7 * at, dwx + 4 * at, NH, S);
        return (int)hipGetLastError();
    });
}
template <int DH, bool FS>
int backward_launch(const float* dh, const float* r, const float* saved, float* dwx, int B, int NH, int S, hipStream_t st) {
    return reinterpret_cast<size_t>(saved) & 15 ? backward_launch_w<DH, FS, false>(dh, r, saved, dwx, B, NH, S, st)
                                                : backward_launch_w<DH, FS, true>(dh, r, saved, dwx, B, NH, S, st);
}

template <int DH>
int backward_t(const float* dh, const float* h, const float* r, const float* saved, float* dwx, float* dr, float* db, int B, int NH, int S,
               int fs, char* ws, hipStream_t st) {
    if (int rc = fs ? backward_launch<DH, true>(dh, r, saved, dwx, B, NH, S, st) : backward_launch<DH, false>(dh, r, saved, dwx, B, NH, S, st)) return rc;
    const int ns = slices_for(B, NH, S);
    const size_t nr = (size_t)NH * 4 * DH * DH, nb = (size_t)NH * 4 * DH;
    float* part_r = reinterpret_cast<float*>(ws);
    float* part_b = part_r + (size_t)ns * nr;
    if constexpr (dr_lds(DH) > 0)
        if (hipError_t e = mlstm::lds_limit_once<slstm_dr_kernel<DH>>(dr_lds(DH)); e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(slstm_dr_kernel<DH>, dim3(NH * 4, ns), dim3(256), dr_lds(DH), st, dwx, h, part_r, part_b, B, NH, S, ns);
    const size_t wgs = (nr + 63) / 64 + (nb + 63) / 64, most = 1 << 23;
    hipLaunchKernelGGL(slstm_reduce_kernel, dim3((unsigned)(wgs < most ? wgs : most)), dim3(256), 0, st, Reduce{part_r, dr, nr}, Reduce{part_b, db, nb}, ns);
    return (int)hipGetLastError();
}

bool good_dh(int DH) { return DH == 32 || DH == 64 || DH == 128; }

}  // namespace slstm

extern "C" {

size_t slstm_saved_bytes(int B, int NH, int S, int DH) {
    if (B <= 0 || NH <= 0 || S <= 0 || !slstm::good_dh(DH)) return 0;
    return (size_t)B * S * 7 * NH * DH * sizeof(float);
}

size_t slstm_workspace_bytes(int B, int NH, int S, int DH) {
    if (B <= 0 || NH <= 0 || S <= 0 || !slstm::good_dh(DH)) return 0;
    return (size_t)slstm::slices_for(B, NH, S) * NH * 4 * ((size_t)DH * DH + DH) * sizeof(float);
}

int slstm_forward_ex(const float* wx, const float* r, const float* b, float* h, float* saved, int B, int NH, int S, int DH,
                     int forget_sigmoid, void* stream) {
    if (!wx || !r || !b || !h || B <= 0 || NH <= 0 || S <= 0) return MLSTM_EINVAL;
    if (!slstm::good_dh(DH)) return MLSTM_ESHAPE;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int fs = forget_sigmoid ? 1 : 0;
    switch (DH) {
        case 32: return slstm::forward_t<32>(wx, r, b, h, saved, B, NH, S, fs, st);
        case 64: return slstm::forward_t<64>(wx, r, b, h, saved, B, NH, S, fs, st);
        default: return slstm::forward_t<128>(wx, r, b, h, saved, B, NH, S, fs, st);
    }
}

int slstm_backward_ex(const float* dh, const float* h, const float* r, const float* saved, float* dwx, float* dr, float* db, int B,
                      int NH, int S, int DH, int forget_sigmoid, void* workspace, size_t workspace_bytes, void* stream) {
    if (!dh || !h || !r || !saved || !dwx || !dr || !db || B <= 0 || NH <= 0 || S <= 0) return MLSTM_EINVAL;
    if (!slstm::good_dh(DH)) return MLSTM_ESHAPE;
    // (the kernels' offsets inside nine rows of dWx are 32 bits)
    if ((size_t)NH * DH > 0xffffffffu / (9 * 4 * sizeof(float))) return MLSTM_ESHAPE;
    if (!workspace || workspace_bytes < slstm_workspace_bytes(B, NH, S, DH)) return MLSTM_EWORKSPACE;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int fs = forget_sigmoid ? 1 : 0;
    char* ws = reinterpret_cast<char*>(workspace);
    switch (DH) {
        case 32: return slstm::backward_t<32>(dh, h, r, saved, dwx, dr, db, B, NH, S, fs, ws, st);
        case 64: return slstm::backward_t<64>(dh, h, r, saved, dwx, dr, db, B, NH, S, fs, ws, st);
        default: return slstm::backward_t<128>(dh, h, r, saved, dwx, dr, db, B, NH, S, fs, ws, st);
    }
}

}  // extern "C"
