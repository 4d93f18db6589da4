// What the gate pre-pass (mlstm_gates.hip) and a row kernel that forms the gates of its head by itself (mlstm_roww.hip) have in common:
// see the head of mlstm_gates.hip for the quantities.
#pragma once
#include "mlstm_device.h"
#include "mlstm_kernels.h"

namespace mlstm {

// the DPP scans of mlstm_device.h on doubles, two moves per step
template <int CTRL>
__device__ __forceinline__ double dpp_d(double old, double src) {
    const long long o = __builtin_bit_cast(long long, old), x = __builtin_bit_cast(long long, src);
    const int lo = __builtin_amdgcn_update_dpp((int)o, (int)x, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(x >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double readlane_d(double v, int lane) {
    const long long x = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_readlane((int)x, lane), hi = __builtin_amdgcn_readlane((int)(x >> 32), lane);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
struct AddD { static __device__ __forceinline__ double id() { return 0.0; } static __device__ __forceinline__ double f(double a, double b) { return a + b; } };
struct MaxD { static __device__ __forceinline__ double id() { return -INFINITY; } static __device__ __forceinline__ double f(double a, double b) { return fmax(a, b); } };
template <typename Op>
__device__ __forceinline__ double wave_scan_inclusive_d(double v, int lane) {
    v = Op::f(v, dpp_d<0x111>(Op::id(), v));
    v = Op::f(v, dpp_d<0x112>(Op::id(), v));
    v = Op::f(v, dpp_d<0x114>(Op::id(), v));
    v = Op::f(v, dpp_d<0x118>(Op::id(), v));
    const double r0 = readlane_d(v, 15), r1 = Op::f(r0, readlane_d(v, 31)), r2 = Op::f(r1, readlane_d(v, 47));
    double c = Op::id();
    if (lane >= 16) c = r0;
    if (lane >= 32) c = r1;
    if (lane >= 48) c = r2;
    return Op::f(c, v);
}

// fp64 prefix over up to 64 granules, one per lane: inclusive sum of their totals, exclusive sum G behind `run`, and the running maximum of (P - G) up to and
// with a granule (before_lane: over the EARLIER ones).  The totals of 64 logarithms are floats: their sums are exact in fp64, in any order, unless they
// lie 2^18 apart.  (By log-step lane shuffles, an LDS round trip each, the two scans took 0.9 us; these take 0.2.)
__device__ __forceinline__ void granule_scan(double tot, double p, double run, int lane, double& incl, double& excl, double& mx) {
    incl = wave_scan_inclusive_d<AddD>(tot, lane);
    excl = run + (incl - tot);                               // G of this granule
    mx = wave_scan_inclusive_d<MaxD>(p - excl, lane);        // with this granule's candidate for later ones
}
__device__ __forceinline__ double before_lane(double mx, int lane) {   // maximum over the earlier granules of these 64
    double x = dpp_d<0x111>(-INFINITY, mx);
    const double r0 = readlane_d(mx, 15), r1 = readlane_d(mx, 31), r2 = readlane_d(mx, 47);
    if (lane == 16) x = r0;
    if (lane == 32) x = r1;
    if (lane == 48) x = r2;
    return x;
}

// What a granule's positions have without the granules before it, from the in-granule cumulative sum c and alpha (natural units): the prefix
// maximum of alpha; alpha2 (rows are padded to whole granules: alpha = -inf there, so padded keys weigh nothing); and the
// factorised weights for blocks of 32 keys that lie entirely below the diagonal: with c0 the block maximum of
// alpha, exp2(alpha_j - beta_i + dG) = exp2(alpha_j - c0) * exp2(c0 - beta_i + dG); both factors are <= 1 there,
// so the product under- or overflows only where the weight itself does.
// One scan over the lanes gives all maxima: of the granule (p), of either half (rounding a product with log2(e) keeps their order), and up to a lane.
struct GateLocal { float loc, p, alpha2, ek2, c0; };
__device__ __forceinline__ GateLocal gates_local(float al, bool ok, int lane) {
    GateLocal v;
    float x = al;   // (as wave_scan_inclusive)
    x = fmaxf(x, dpp_f<0x111>(-INFINITY, x));
    x = fmaxf(x, dpp_f<0x112>(-INFINITY, x));
    x = fmaxf(x, dpp_f<0x114>(-INFINITY, x));
    x = fmaxf(x, dpp_f<0x118>(-INFINITY, x));
    auto at = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l)); };
    const float r0 = at(15), lo = fmaxf(r0, at(31)), r2 = at(47), hi = fmaxf(r2, at(63));
    float before = -INFINITY;
    if (lane >= 16) before = r0;
    if (lane >= 32) before = lo;
    if (lane >= 48) before = fmaxf(lo, r2);
    v.loc = fmaxf(before, x);
    v.p = fmaxf(lo, hi);
    const float al2 = product_apart(al, LOG2E);   // (rounded, also where the block maximum is taken off it)
    v.alpha2 = ok ? al2 : -INFINITY;
    v.c0 = product_apart(lane < 32 ? lo : hi, LOG2E);
    v.ek2 = (ok && v.c0 > -INFINITY) ? fast_exp2(al2 - v.c0) : 0.0f;
    return v;
}
__device__ __forceinline__ void store_local(const GateLocal& v, size_t pos, size_t gidx, int lane, float* alpha2, float* ek2, float* amax2) {
    alpha2[pos] = v.alpha2;
    ek2[pos] = v.ek2;
    if ((lane & 31) == 0) amax2[gidx * 2 + (lane >> 5)] = v.c0;
}
// and with G and R of the granule: beta2 and the stabiliser
struct GateGlobal { float beta2, m; };
__device__ __forceinline__ GateGlobal gates_global(float c, float loc, bool ok, double Gg, double Rg) {
    const float carry = (float)(Rg + Gg);  // max over earlier granules of (alpha_j - G_g(j)) + G_g ; -inf for g == 0
    const float be = fmaxf(loc, carry);
    return GateGlobal{ok ? be * LOG2E : 0.0f, c + be};
}
__device__ __forceinline__ void store_global(const GateGlobal& v, bool ok, double Gg, size_t pos, size_t mpos, size_t gidx, int lane, float* beta2, double* G2, float* M) {
    beta2[pos] = v.beta2;
    if (ok) M[mpos] = v.m;
    if (lane == 0) G2[gidx] = Gg * LOG2E_D;
}

// log-sigmoid of the forget gate at position t from what the caller's F holds (see launch_gates): the pre-activation,
// the log-sigmoid itself, or its cumulative sum over the head (then the difference of two neighbours)
struct GateIn { float x, before, i; };
template <typename TG>
__device__ __forceinline__ GateIn gate_in(const TG* f, const TG* ig, size_t ss, int t, int S, int form) {   // (positions past the end: the last one's)
    t = t < S ? t : S - 1;
    GateIn v;
    v.x = (float)f[(size_t)t * ss];
    v.i = (float)ig[(size_t)t * ss];
    v.before = form == MLSTM_GATE_CUMSUM && t > 0 ? (float)f[(size_t)(t - 1) * ss] : 0.f;
    return v;
}
__device__ __forceinline__ float forget_log(const GateIn& v, int t, int form) {
    if (form == MLSTM_GATE_RAW) return log_sigmoid(v.x);
    if (form == MLSTM_GATE_LOGSIGMOID) return v.x;
    return t > 0 ? v.x - v.before : v.x;
}
__device__ __forceinline__ float last_lane(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63)); }

}  // namespace mlstm
