// Gate pre-pass of the matmul form and of the scan form: everything that depends only on (f, i).
//
// Reference semantics: logsigmoid + cumulative sum of the forget gate and the row maximum of the log-decay
// matrix (mlstm_matmul.py:57-59,73-84; mlstm_scan.py:48-69 computes the same m by a max-plus scan).
//
// With lf = logsigmoid(f), Fc = cumsum(lf), a_j = i_j - Fc_j and A_i = max_{j<=i} a_j the stabilised decay is
//     D_ij - m_i = a_j - A_i,        m_i = Fc_i + A_i,
// so the row maximum is a prefix maximum and the tile kernels need no online rescaling.  Fc grows to 1e3..1e4
// in magnitude, so it is never stored in fp32: each 64-position granule g keeps an fp64 base G_g (Fc before the
// granule) and positions store granule-relative values
//     alpha_j = i_j - (Fc_j - G_g(j)),     beta_i = A_i + G_g(i),
// whence  a_j - A_i = alpha_j - beta_i + (G_g(i) - G_g(j))  with one fp64 subtraction per tile pair.
// alpha, beta and G are stored pre-multiplied by log2(e) (the kernels use exp2); m in natural units.
// alpha and beta have a row stride of ceil(S/64)*64 per head (padded to whole granules).
#include "mlstm_gates.h"

namespace mlstm {

constexpr int GATES_MAX_GRANULES = 2048;  // S <= 131072
constexpr int GATES_WAVES = 16;           // waves per workgroup, a granule each at a time

// Sequences of up to 16 * GPW granules (GPW = 1, 2, 4: S <= 4096) in one launch: a workgroup writes `per` granules (a power of two of up to 16) and
// forms the totals of all granules up to those by itself, one per wave and turn.  What bounds it is instruction issue on one CU, some 90
// instructions per granule for the totals and as many for the outputs; all loads are issued before the first scan.  us, one
// workgroup of 16 waves per head with GPW = 4 whatever the length, and the prefix by lane shuffles / now, one head: S = 64 3.9 / 2.8, 640 4.6 / 3.3,
// 1000 5.0 / 3.4; eight: 2048 7.4 / 5.7, 4096 10.9 / 8.0.  With as many workgroups as CUs the totals formed several times over cost more than
// the outputs saved, hence per = 16 there (32 heads x 4096 10.0 / 8.2; 256 x 1000 6.4 / 5.3 on 16, 5.8 on 4).
template <typename TG, int GPW>
__global__ __launch_bounds__(1024) void gates_kernel_reg(const TG* __restrict__ F, const TG* __restrict__ I, float* __restrict__ alpha2,
                                                        float* __restrict__ beta2, double* __restrict__ G2, float* __restrict__ M,
                                                        float* __restrict__ ek2, float* __restrict__ amax2, int S, int NG, int per, Lay lg, int form,
                                                        SavedStamp stamp) {
    stamp_apply(stamp, blockIdx.x == 0 && blockIdx.y == 0, threadIdx.x);
    __shared__ double sT[GATES_WAVES * GPW];
    __shared__ double sP[GATES_WAVES * GPW];
    // (the last granules first: they take longest)
    const int bh = blockIdx.x, first = per * (int)(gridDim.y - 1 - blockIdx.y), seg = first / GATES_WAVES, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const size_t gs = (size_t)lg.ss;
    const TG* f = F + lg.head(bh);
    const TG* ig = I + lg.head(bh);
    GateIn in[GPW];
    const int gown = wave + GATES_WAVES * seg, t = gown * GRAN + lane;
    const bool mine = gown >= first && gown < first + per && gown < NG, ok = t < S;
    const size_t pos = (size_t)bh * NG * GRAN + t, gidx = (size_t)bh * NG + gown;
    float c = 0.f, loc = 0.f;
#pragma unroll
    for (int k = 0; k < GPW; k++) in[k] = gate_in(f, ig, gs, (wave + GATES_WAVES * k) * GRAN + lane, S, form);
#pragma unroll
    for (int k = 0; k < GPW; k++) {
        const int g = wave + GATES_WAVES * k, tk = g * GRAN + lane;
        if (g < first + per && g < NG) {
            c = wave_scan_inclusive<OpAdd>(tk < S ? forget_log(in[k], tk, form) : 0.0f);
            const float al = tk < S ? in[k].i - c : -INFINITY;
            const float tot = last_lane(c);
            float p;
            if (mine && k == seg) {
                const GateLocal v = gates_local(al, ok, lane);
                store_local(v, pos, gidx, lane, alpha2, ek2, amax2);
                loc = v.loc;
                p = v.p;
            } else {
                p = wave_reduce<OpMax>(al);
            }
            if (lane == 0) { sT[g] = (double)tot; sP[g] = (double)p; }
        }
    }
    // (c is now that of the last granule passed, the wave's own)
    __syncthreads();
    if (!mine) return;
    {   // the prefix, by every wave for itself (a wave alone, with the others waiting for it, takes as long, and a barrier)
        const int ng = gown + 1;
        double incl, excl, mx;
        granule_scan(lane < ng ? sT[lane] : 0.0, lane < ng ? sP[lane] : -INFINITY, 0.0, lane, incl, excl, mx);
        const double before = before_lane(mx, lane);
        const double Gg = readlane_d(excl, gown);
        store_global(gates_global(c, loc, ok, Gg, readlane_d(before, gown)), ok, Gg, pos, (size_t)bh * S + t, gidx, lane, beta2, G2, M);
    }
}

// Longer sequences in two launches of a workgroup per 16 granules, each granule's totals formed once.  us, one workgroup per
// head / now: one head of 8192 positions 16.6 / 8.0, 64 heads of 8192 20.1 / 12.0, of 16384 37.5 / 17.2 (at 4096 one launch of 8 is level with these two):
//   gates_local_kernel   alpha2 and the key weights, which need no other granule; in beta2 the prefix maxima of alpha, in M the cumulative
//                        sums, both of the granule alone and in natural units; totals: sum of the log-sigmoids and maximum of alpha per granule
//   gates_carry_kernel   the granules before, and with them beta2, M and G2
template <typename TG>
__global__ __launch_bounds__(1024) void gates_local_kernel(const TG* __restrict__ F, const TG* __restrict__ I, float* __restrict__ alpha2,
                                                          float* __restrict__ beta2, float2* __restrict__ totals, float* __restrict__ M,
                                                          float* __restrict__ ek2, float* __restrict__ amax2, int S, int NG, Lay lg, int form,
                                                          SavedStamp stamp) {
    stamp_apply(stamp, blockIdx.x == 0 && blockIdx.y == 0, threadIdx.x);
    const int bh = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int g = blockIdx.y * GATES_WAVES + __builtin_amdgcn_readfirstlane(tid >> 6), t = g * GRAN + lane;
    if (g >= NG) return;
    const size_t gs = (size_t)lg.ss;
    const bool ok = t < S;
    const GateIn in = gate_in(F + lg.head(bh), I + lg.head(bh), gs, t, S, form);
    const float c = wave_scan_inclusive<OpAdd>(ok ? forget_log(in, t, form) : 0.0f), al = ok ? in.i - c : -INFINITY;
    const float tot = last_lane(c);
    const size_t pos = (size_t)bh * NG * GRAN + t, gidx = (size_t)bh * NG + g;
    const GateLocal v = gates_local(al, ok, lane);
    if (lane == 0) totals[gidx] = make_float2(tot, v.p);
    store_local(v, pos, gidx, lane, alpha2, ek2, amax2);
    beta2[pos] = v.loc;
    if (ok) M[(size_t)bh * S + t] = c;
}
__global__ __launch_bounds__(1024) void gates_carry_kernel(const float2* __restrict__ totals, float* __restrict__ beta2, double* __restrict__ G2,
                                                          float* __restrict__ M, int S, int NG) {
    constexpr int GROUPS = GATES_MAX_GRANULES / 64;   // of 64 granules
    __shared__ double sSum[GROUPS], sMax[GROUPS], sG[GATES_WAVES], sR[GATES_WAVES];
    const int bh = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int first = blockIdx.y * GATES_WAVES, mygroup = first / 64;   // (the workgroup's granules lie in one group)
    const float2* tp = totals + (size_t)bh * NG;
    const int g = first + wave, t = g * GRAN + lane;
    const bool mine = g < NG, ok = mine && t < S;
    const size_t pos = (size_t)bh * NG * GRAN + t, mpos = (size_t)bh * S + t;
    const float loc = mine ? beta2[pos] : 0.f, c = ok ? M[mpos] : 0.f;
    double tot[2], p[2];   // of groups wave and wave + 16
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int n = 64 * (wave + GATES_WAVES * k) + lane;
        const bool there = wave + GATES_WAVES * k <= mygroup && n < NG;
        const float2 x = there ? tp[n] : make_float2(0.f, -INFINITY);
        tot[k] = (double)x.x;
        p[k] = (double)x.y;
    }
#pragma unroll
    for (int k = 0; k < 2; k++)
        if (wave + GATES_WAVES * k <= mygroup) {
            const double incl = wave_scan_inclusive_d<AddD>(tot[k], lane);
            if (lane == 63) sSum[wave + GATES_WAVES * k] = incl;
        }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int group = wave + GATES_WAVES * k;
        if (group <= mygroup) {
            double run = 0.0, incl, excl, mx;
            for (int n = 0; n < group; n++) run += sSum[n];
            granule_scan(tot[k], p[k], run, lane, incl, excl, mx);
            if (lane == 63) sMax[group] = mx;
            const int own = 64 * group + lane - first;
            const double before = before_lane(mx, lane);
            if (group == mygroup && own >= 0 && own < GATES_WAVES) { sG[own] = excl; sR[own] = before; }
        }
    }
    __syncthreads();
    if (!mine) return;
    double rmax = -INFINITY;
    for (int n = 0; n < mygroup; n++) rmax = fmax(rmax, sMax[n]);
    const double Gg = sG[wave];
    store_global(gates_global(c, loc, ok, Gg, fmax(rmax, sR[wave])), ok, Gg, pos, mpos, (size_t)bh * NG + g, lane, beta2, G2, M);
}

template <typename TG>
static hipError_t launch_gates_t(const void* F, const void* I, float* alpha2, float* beta2, double* G2, float* M, float* ek2,
                                 float* amax2, void* scratch, int BH, int S, hipStream_t st, const Lay& lg, int form, const SavedStamp& stamp) {
    const int NG = (S + GRAN - 1) / GRAN;
    const TG *f = (const TG*)F, *i = (const TG*)I;
    const int per = (long long)BH * ((NG + 3) / 4) <= 256 ? 4 : GATES_WAVES, parts = (NG + per - 1) / per;
    if (NG <= GATES_WAVES)
        hipLaunchKernelGGL((gates_kernel_reg<TG, 1>), dim3(BH, parts), dim3(1024), 0, st, f, i, alpha2, beta2, G2, M, ek2, amax2, S, NG, per, lg, form, stamp);
    else if (NG <= 2 * GATES_WAVES)
        hipLaunchKernelGGL((gates_kernel_reg<TG, 2>), dim3(BH, parts), dim3(1024), 0, st, f, i, alpha2, beta2, G2, M, ek2, amax2, S, NG, per, lg, form, stamp);
    else if (NG <= 4 * GATES_WAVES)
        hipLaunchKernelGGL((gates_kernel_reg<TG, 4>), dim3(BH, parts), dim3(1024), 0, st, f, i, alpha2, beta2, G2, M, ek2, amax2, S, NG, per, lg, form, stamp);
    else {
        const dim3 grid(BH, (NG + GATES_WAVES - 1) / GATES_WAVES);
        float2* const totals = static_cast<float2*>(scratch);
        hipLaunchKernelGGL(gates_local_kernel<TG>, grid, dim3(1024), 0, st, f, i, alpha2, beta2, totals, M, ek2, amax2, S, NG, lg, form, stamp);
        hipLaunchKernelGGL(gates_carry_kernel, grid, dim3(1024), 0, st, totals, beta2, G2, M, S, NG);
    }
    return hipGetLastError();
}

hipError_t launch_gates(int gate_dtype, const void* F, const void* I, float* alpha2, float* beta2, double* G2, float* M, float* ek2,
                        float* amax2, void* scratch, int BH, int S, hipStream_t st, const Lay& lg, int form, const SavedStamp* stamp_in) {
    const SavedStamp stamp = stamp_in ? *stamp_in : SavedStamp{};
    if ((S + GRAN - 1) / GRAN > GATES_MAX_GRANULES) return hipErrorInvalidValue;
    if (form == MLSTM_GATE_CUMSUM && gate_dtype != MLSTM_F32) return hipErrorInvalidValue;   // (16-bit types cannot hold the sum)
    switch (gate_dtype) {
        case MLSTM_F32: return launch_gates_t<float>(F, I, alpha2, beta2, G2, M, ek2, amax2, scratch, BH, S, st, lg, form, stamp);
        case MLSTM_F16: return launch_gates_t<_Float16>(F, I, alpha2, beta2, G2, M, ek2, amax2, scratch, BH, S, st, lg, form, stamp);
        case MLSTM_BF16: return launch_gates_t<__bf16>(F, I, alpha2, beta2, G2, M, ek2, amax2, scratch, BH, S, st, lg, form, stamp);
    }
    return hipErrorInvalidValue;
}

}  // namespace mlstm
