// Internal launch interface between the C ABI (mlstm_api.hip) and the kernel translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include "../../include/mlstm_hip.h"

namespace mlstm {

inline size_t dtype_size(int dt) { return dt == MLSTM_F32 ? 4 : 2; }

// Raises a kernel's dynamic LDS limit, once per process and kernel; the initialisation of a function-local static is
// thread-safe, so concurrent first calls do not race.  Returns the status of that one call.
template <auto KERN>
inline hipError_t lds_limit_once(int bytes) {
    static const hipError_t rc = hipFuncSetAttribute(reinterpret_cast<const void*>(KERN), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    return rc;
}
// For kernels that wait in every step for memory that is counted by hand (s_waitcnt vmcnt(n) with n the operations the SOURCE issues behind the
// ones it waits for).  Operations that the count does not know, the compiler's own for a spilled register among them, never let a load pass
// as landed that has not: they only push counted ones out of the newest n, and the wait takes in copies that were meant to stay under
// way.  In a step that is all latency that is its whole point gone, so the kernel is not launched (MLSTM_EBUILD) if it was compiled to use any
// scratch memory at all; where others give the same results (launch_chunk_t), they take its place.  Asked once per process and kernel.
template <auto KERN>
inline int no_scratch_once() {
    static const int rc = [] {
        hipFuncAttributes attr;
        const hipError_t e = hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(KERN));
        if (e != hipSuccess) return (int)e;
        return attr.localSizeBytes == 0 ? 0 : MLSTM_EBUILD;
    }();
    return rc;
}
constexpr int GATE_GRANULE = 64;  // positions per gate granule (== mlstm::GRAN in the device code)

// Where a [B,NH,S,D] (or [B,NH,S]) tensor of the caller's keeps position s of head bh = b * NH + h: at element
// b * sb + h * sh + s * ss (+ the column: the last dimension is contiguous).  Everything the library owns (workspace,
// statistics m and b, chunk states) is dense.
struct Lay {
    long long sb, sh, ss;
    int NH;
    __host__ __device__ size_t head(int bh) const { return (size_t)((long long)(bh / NH) * sb + (long long)(bh % NH) * sh); }
};
inline Lay dense_layout(int NH, long long S, long long D) { return Lay{(long long)NH * S * D, S * D, D, NH}; }
// dense [B,NH,S,D]?  (The tile kernels keep a variant with the strides as compile-time constants for that case: run-time
// strides cost them address arithmetic in loops that are bound by instruction issue.)
inline bool is_dense(const Lay& l, long long S, long long D) { return l.ss == D && l.sh == S * D && l.sb == (long long)l.NH * S * D; }

// Eight words that one kernel of the forward leaves at the head of a caller-kept buffer (dst) and one kernel of the backward
// compares with what it finds there (src; a difference sets bit 1 of *err): rides along in kernels that run anyway.
struct SavedStamp {
    int* dst = nullptr;
    const int* src = nullptr;
    int* err = nullptr;
    int v[8] = {};
};
#if defined(__HIPCC__)
__device__ __forceinline__ void stamp_apply(const SavedStamp& s, bool first_block, int tid) {
    if (!first_block || tid >= 8) return;
    if (s.dst) s.dst[tid] = s.v[tid];
    if (s.src && s.src[tid] != s.v[tid]) atomicOr(s.err, 2);
}
#endif

// Gate pre-pass: alpha2, beta2 [BH, NG*64] fp32 (NG = ceil(S/64), rows padded), G2 [BH, NG] fp64, M [BH,S] fp32.
// ek2 [BH, NG*64] = exp2(alpha2 - block max), amax2 [BH, NG*2] = the maxima of alpha2 over blocks of 32 positions.
// lg: layout of F and I.  gate_form: what F holds (MLSTM_GATE_RAW: the forget gate's pre-activation, _LOGSIGMOID: its
// log-sigmoid, _CUMSUM: the cumulative sum of that over the positions of a head).
// scratch: 8 BH NG bytes (on an 8-byte boundary), written and read where S > 4096.
hipError_t launch_gates(int gate_dtype, const void* F, const void* I, float* alpha2, float* beta2, double* G2, float* M, float* ek2,
                        float* amax2, void* scratch, int BH, int S, hipStream_t st, const Lay& lg, int gate_form, const SavedStamp* stamp = nullptr);
inline hipError_t launch_gates(int gate_dtype, const void* F, const void* I, float* alpha2, float* beta2, double* G2, float* M, float* ek2,
                               float* amax2, void* scratch, int BH, int S, hipStream_t st) {
    return launch_gates(gate_dtype, F, I, alpha2, beta2, G2, M, ek2, amax2, scratch, BH, S, st, dense_layout(BH, S, 1), MLSTM_GATE_RAW);
}

extern bool g_force_generic;  // see mlstm_force_generic_kernels
constexpr int DEFAULT_SPIN_LIMIT = 1 << 22;   // iterations of 64 cycles and an LDS read each: a fraction of a second

struct RowArgs {
    const void* X;    // row operand held in registers: Q (forward) or dH (dQ pass)      [BH,S,D]
    const void* Y1;   // contracted over D with X:       K (forward) or V (dQ pass)
    const void* Y2;   // contracted over keys:           V (forward) or K (dQ pass)
    void* out;        // H (forward) or dQ
    // forward with an output gate: when O is set the kernel also writes silu(O) * H to out_gated (H itself, which the
    // backward needs, still goes to out)
    const void* O;
    void* out_gated;
    // long sequences in chunks: with chunk_len = L > 0 a row takes the keys of its own chunk of
    // L positions from Y1 / Y2 and everything before the chunk from the state at the end of the previous chunk
    // (launch_chunk_states).  L is a multiple of 128.
    int chunk_len;
    int n_states;         // states per head (chunks but the last)
    const void* Qrow;     // dQ pass in chunks: Q [BH,S,D] and
    float* rowinter;      //   [BH,S] out: q_i . dQ_i of the state part = the row sums of dD over the keys before the chunk
    const void* Cst;      // [BH][n_states][D][D] matrix states in the element type of X, rows in contraction order:
                          // key-major for the forward, value-major (ChunkArgs::CstT) for the dQ pass
    const void* Cst_lo;   // split mode: the states' low-order terms, same layout (the state enters its product as Cst + Cst_lo)
    const float* Nst;     // [BH][n_states][D] vector states
    const float* alpha2;
    const float* beta2;
    const double* G2;
    const float* ek2;     // factorised key weights and their block maxima (see launch_gates)
    const float* amax2;
    const float* M;       // forward: stabiliser, for the normaliser
    float* Bsum;          // forward: row sums b
    // dQ pass: the kernel derives 1/n and db per row from (dh, h, m, b) and also writes them, [BH, NG*64], for the
    // column kernel that runs after it
    const void* Hin;      // forward output h [BH,S,D]
    const float* Bin;     // forward row sums b [BH,S]
    float* inv_n;
    float* db;
    int BH, S, NG;
    // Split mode (16-bit types; rowx_kernel and row_kernel): the weights of the second product enter it as two terms, hi + lo,
    // each in the element type (two MFMAs per fragment), so that their rounding no longer limits the result.  The
    // forward then also leaves h - (h rounded) in out_lo; the dQ pass reads it back through Hin_lo for dh . h.
    int precise;
    void* out_lo;
    const void* Hin_lo;
    // eight-wave kernel: the producers' wait for their P buffer is bounded; a wait that expires sets *err (sticky,
    // see mlstm_kernel_error) and the kernel runs on to its end.  spin_limit < 0 (test aid) lets every wait expire.
    int* err;
    int spin_limit;
    // layouts of the caller's tensors: la for q, k, v (forward: X, Y1, Y2; dQ pass: Y1, Y2, Qrow and out),
    // lb for h, dh, o (forward: out, O, out_gated; dQ pass: X), lh for Hin (the caller's h, or a dense recomputed one)
    Lay la, lb, lh;
    // forward of a sequence that is not cut, where roww_kernel serves it (roww_serves): with gate_F set it forms the gates of its head by itself, from
    // F and I in layout lg, and leaves in alpha2, beta2, G2, ek2, amax2 and M what launch_gates would have
    const void* gate_F = nullptr;
    const void* gate_I = nullptr;
    int gate_dtype = 0, gate_form = 0;
    Lay lg{};
};
// mode 0 = forward (H, b), mode 1 = dQ
int launch_row_kernel(int mode, int dtype, int D, const RowArgs& a, hipStream_t st);
// fp32 on 32 rows per workgroup, the same bits, for launches that leave the chip part empty; D in {64, 128}
int launch_rowf_kernel(int mode, int D, const RowArgs& a, hipStream_t st);
// eight waves (producer / consumer pairs per SIMD); 16-bit types and D in {128, 256} only
int launch_row8_kernel(int mode, int dtype, int D, const RowArgs& a, hipStream_t st);
// the same bits on 64 or 32 rows per workgroup, for launches that leave the chip part empty; 16-bit types and D in {128, 256} only
int launch_roww_kernel(int mode, int dtype, int D, const RowArgs& a, hipStream_t st);
// split mode on 64 rows per workgroup, the bits of the four-wave kernel, for the same launches; not with an output gate
int launch_rowx_kernel(int mode, int dtype, int D, const RowArgs& a, hipStream_t st);
constexpr int RW_MOST_KEYS = 1024;   // keys a row of roww_kernel may meet: their scalars stay in LDS for the whole kernel
inline bool roww_serves(int dtype, int D, const RowArgs& a) {
    // (a wait bound of the caller's asks for the kernel that has the wait: mlstm_set_spin_limit)
    if (dtype == MLSTM_F32 || (D != 128 && D != 256) || a.precise || g_force_generic || a.spin_limit != DEFAULT_SPIN_LIMIT) return false;
    if ((a.chunk_len > 0 && a.chunk_len < a.NG * GATE_GRANULE ? a.chunk_len : a.NG * GATE_GRANULE) > RW_MOST_KEYS) return false;
    // While its workgroups (64 rows) number no more than the chip's CUs, roww_kernel: row8_kernel / roww_kernel, forward, us --
    // D = 128   10: 13.3 / 9.9   128 (uncut, 1000 positions): 20 / 14.9   256 (chunks of 512): 15.6 / 12.9
    // D = 256   10: 17.2 / 12.6   224 (chunks of 512): 23.1 / 18.4   256: 15.4 / 13.0
    // and beyond them, where sequences are not cut, as long as the workgroups left over, which are the lightest, end before the longest walk,
    // forward and dQ pass --
    // D = 128   320: 128 positions 8.2, 10.6 / 11.2, 13.0   256: 10.6, 12.6 / 11.8, 13.4   512: 13.6, 16.0 / 13.2, 15.7   1000: 21.1, 22.8 / 16.8, 18.7
    //           384: 512 positions 14.1, 16.1 / 14.8, 16.7   1000: 20.9, 22.3 / 18.6, 20.7   448: 1000 positions 21.0, 22.8 / 21.4, 23.4
    // D = 256   320: 256 positions 14.4, 19.2 / 14.5, 19.1   512: 18.9, 23.7 / 17.5, 21.4   1000: 28.4, 32.5 / 24.7, 26.5   384: 1000 28.5, 32.7 / 25.5, 28.8
    //           (in chunks of 512, 320: D = 128 16.4, 18.5 / 19.8, 23.6   D = 256 25.8, 30.4 / 29.2, 36.9)
    // (bf16; fp16, in chunks of 512, forward and dQ pass, 256: D = 128 17.5, 18.8 / 15.0, 16.7, D = 256 25.6, 29.2 / 21.1, 23.4)
    const long long roww_most = a.chunk_len > 0 ? 256 : 256 + 8 * a.NG;
    return (long long)a.BH * a.NG <= roww_most;
}
// (the four-wave kernel serves every other case: fp32, D = 64, split mode -- in chunks too --, large launches at D = 128 and the test switch)
inline int launch_row_best(int mode, int dtype, int D, const RowArgs& a, hipStream_t st) {
    // (what a kernel that forms the gates is to read is not there for any other, also where a switch was turned since that was decided)
    if (a.gate_F) return launch_roww_kernel(mode, dtype, D, a, st);
    if (dtype != MLSTM_F32 && (D == 128 || D == 256) && !g_force_generic) {
        int rc = MLSTM_ESHAPE;
        if (roww_serves(dtype, D, a)) rc = launch_roww_kernel(mode, dtype, D, a, st);
        // Split mode: row_kernel / rowx_kernel, forward and dQ pass, us (heads x positions: 2, 8 and 16 x 2048, 12 and 16 x 1500) --
        // D = 128   64: 19.0, 21.8 / 14.4, 16.4   256: 21.4, 23.2 / 16.3, 18.6   288: 21.0, 23.5 / 16.7, 20.6   384: 21.5, 24.1 / 22.0, 25.2   512: 22.6, 26.0 / 25.8, 29.3
        // D = 256   64: 34.6, 39.2 / 23.1, 27.0   256: 38.0, 42.3 / 25.6, 30.4   288: 37.3, 41.4 / 25.8, 32.1   384: 37.9, 41.8 / 33.4, 39.2   512: 40.1, 44.7 / 40.1, 46.3
        //           (8 heads, whose tiles share an XCD's cache one by one: 376, 8 x 3000, 38.2, 42.0 / 36.8, 44.2   512, 8 x 4096, 40.1, 44.7 / 46.7, 54.2)
        if ((long long)a.BH * a.NG <= (D == 128 ? 256 : 512) && a.precise) rc = launch_rowx_kernel(mode, dtype, D, a, st);
        // D = 128 beyond 512 of them, row_kernel, whose workgroups share a CU in pairs: row8_kernel / row_kernel, forward and dQ pass, us --
        //   512: 17.8, 20.5 / 17.2, 20.8   768: 27.2, 31.1 / 20.9, 25.4   1024: 30.0, 34.4 / 23.2, 28.4   2048: 49.1, 56.8 / 36.7, 45.0
        //   8192: 212, 245 / 141, 182      16384: 415, 489 / 275, 368     not in chunks, 1024: 35.2, 38.7 / 26.7, 29.8
        // (and as long as the granules a row may meet leave the LDS for two: uncut sequences of up to 118784 positions)
        const bool pairs = D == 128 && (long long)a.BH * a.NG > 512 && a.spin_limit == DEFAULT_SPIN_LIMIT && (a.chunk_len > 0 || a.NG <= 1856);
        if (rc == MLSTM_ESHAPE && !a.precise && !pairs) rc = launch_row8_kernel(mode, dtype, D, a, st);
        if (rc != MLSTM_ESHAPE) return rc;  // extremely long sequences do not fit its LDS budget
    }
    return launch_row_kernel(mode, dtype, D, a, st);
}

struct ColArgs {
    const void* Q; const void* K; const void* V; const void* dH;
    void* dK; void* dV;
    float* colsum;    // [BH,S] fp32 column sums of dD (= dI before the cast)
    float* rowpart;   // [BH,RS,S] fp32 partial row sums of dD, one slice per key tile (RS = NG), or, in chunks, per key
                      // tile of the position's own chunk (RS = chunk_len / 64: slice = key tile modulo RS)
    int RS;
    float* rowpart2 = nullptr;   // may be null: a second array of partials, for the kernel that keeps a tile's halves apart (colf_serves)
    const float* alpha2; const float* beta2; const double* G2;
    const float* inv_n; const float* db;
    int BH, S, NG;
    // long sequences in chunks: with chunk_len > 0 the keys walk the queries of their own chunk and
    // take the contribution of the queries behind it from the chunk's reverse states (ChunkArgs::reverse); rowpart is then
    // written for the key tiles of the query's own chunk only
    int chunk_len;
    int n_states;
    const void* Ev;          // [BH][n_states][D][D] reverse states, value-major (ChunkArgs::CstT of the reverse pass)
    const void* Ev_lo;       // split mode: their low-order terms
    const float* gvec;       // [BH][n_states][D]
    int precise;             // split mode (see RowArgs): G and W enter phase B as hi + lo
    Lay la, lb;              // layouts of Q, K, V, dK, dV (la) and of dH (lb)
};
int launch_col_kernel(int dtype, int D, const ColArgs& a, hipStream_t st);
// fp32 on 32 keys per workgroup, the same bits, for launches that leave the chip part empty; D in {64, 128}.  The row partials of a
// tile's first and second 32 keys go to rowpart and rowpart2 (launch_df adds them): launch_col_kernel takes it where rowpart2 is given
bool colf_serves(int dtype, int D, const ColArgs& a);
int launch_colf_kernel(int D, const ColArgs& a, hipStream_t st);
// phase A as 16x16x32 products on two query halves, the element-wise part of the first between the MFMAs of the second;
// 16-bit types at D = 128 and 256 only
int launch_col16_kernel(int dtype, int D, const ColArgs& a, hipStream_t st);
// weights kept in registers between the two phases (no G / W tiles in LDS); 16-bit types at D = 128 and 256, split mode included
int launch_cold_kernel(int dtype, int D, const ColArgs& a, hipStream_t st);
// the same on 64 keys per workgroup and eight waves, the same bits, for launches of few workgroups; keys that meet up to 1024 queries
int launch_colw_kernel(int dtype, int D, const ColArgs& a, hipStream_t st);
extern int g_col_variant;   // see mlstm_set_column_kernel: 0 = the library's choice, 1 = col16_kernel, 2 = cold_kernel, 3 = col_kernel
constexpr int CW_MOST_QUERIES = 1024;    // queries a key of colw_kernel may meet: their scalars stay in LDS for the whole kernel
// Workgroups of 64 keys up to which colw_kernel is the faster one.  It runs them in rounds of 256, one per CU; cold_kernel has one per 128 keys, one per CU too,
// but two at D = 128 outside split mode.  Up to 512 colw_kernel's two rounds are shorter than cold_kernel's one or two.  Of 513 to 768 it needs a third: a short one
// if the last tiles of a long head are in it (tiles go heaviest first), a whole one if heads are short or a sequence has a few chunks only, while cold_kernel is still in its
// second, which a short last chunk leaves nearly empty.  cold_kernel / colw_kernel, us, workgroups of 64 keys (heads):
//   D = 256, bf16, uncut   S = 64   579: 46 / 39   768: 50 / 44        S = 128   516: 42 / 40   580: 43 / 41   642: 43 / 44        S = 320   515: 41 / 45   768: 52 / 62
//     S = 512   512: 48 / 43   576: 50 / 52   768: 59 / 67     S = 640   580: 59 / 65   640: 60 / 63     S = 768   576: 66 / 64   648: 71 / 79     S = 1000   512: 76 / 62   576: 84 / 78   640: 81 / 80   768: 83 / 94
//     in chunks of 512   S = 1100   522: 59 / 61   594: 60 / 74   756: 75 / 85     S = 1536   600: 65 / 69   768: 76 / 76     S = 2048   512: 56 / 54   672: 76 / 75   768: 82 / 83     S = 4096   576: 76 / 70   768: 93 / 86
//     in split mode   S = 1000   576: 97 / 88   768: 98 / 107     S = 1100   594: 76 / 92     S = 2048   768: 107 / 104     S = 4096   768: 119 / 107
//   D = 256, fp16 (cold_kernel with some 95 registers spilled)   S = 320   515: 55 / 47   768: 68 / 64     S = 1100   594: 81 / 79   738: 98 / 91     S = 4096   768: 113 / 87     split mode   S = 1000   768: 102 / 102
//   D = 128, bf16 (fp16 alike), uncut   S = 200   512: 21.5 / 19.9   580: 24 / 26   768: 24 / 28     S = 320   515: 28 / 29   768: 30 / 39     S = 384   576: 30 / 29   642: 32 / 35     S = 448   644: 35 / 34   770: 37 / 42
//     S = 512   768: 40 / 38     S = 1000   512: 59 / 38   768: 63 / 56     in chunks   S = 1100   594: 42 / 42   756: 43 / 45     S = 1400   682: 43 / 42   770: 43 / 45     S = 1536   768: 46 / 42     S = 2048   768: 48 / 44
//     in split mode   S = 64   768: 32 / 29     S = 320   515: 29 / 34     S = 1000   512: 63 / 51   640: 64 / 68   768: 66 / 76     S = 1100   595: 45 / 52     S = 1800   667: 51 / 55     S = 2048   768: 59 / 58     S = 4096   768: 67 / 58
inline int colw_most_workgroups(int dtype, int D, const ColArgs& a) {
    const bool paired = D == 128 && !a.precise;   // (cold_kernel's, on a CU)
    if (dtype == MLSTM_F16 && D == 256) return 768;
    if (a.chunk_len > 0 && a.chunk_len < a.NG * GATE_GRANULE) return a.S >= (paired ? 3ll : 4ll) * a.chunk_len ? 768 : paired ? 640 : 512;
    if (paired) return a.NG <= 5 ? 512 : a.NG >= 8 ? 768 : 512 + 96 * (a.NG - 5);
    return a.NG == 1 ? 768 : a.NG == 2 ? 640 : a.NG < 12 ? 512 : 576;
}
inline bool colw_serves(int dtype, int D, const ColArgs& a) {
    if (dtype == MLSTM_F32 || (D != 128 && D != 256) || g_force_generic || g_col_variant != 0) return false;
    if ((a.chunk_len > 0 && a.chunk_len < a.NG * GATE_GRANULE ? a.chunk_len : a.NG * GATE_GRANULE) > CW_MOST_QUERIES) return false;
    return (long long)a.BH * a.NG <= colw_most_workgroups(dtype, D, a);
}
inline int launch_col_best(int dtype, int D, const ColArgs& a, hipStream_t st) {
    const bool half_big = dtype != MLSTM_F32 && (D == 128 || D == 256);
    int variant = g_force_generic ? 3 : g_col_variant;
    if (!half_big || variant < 0 || variant > 3) variant = 3;
    if (variant == 0) {
        if (colw_serves(dtype, D, a)) return launch_colw_kernel(dtype, D, a, st);
        variant = 2;   // (measured faster than col16_kernel at D = 128 and 256, chunked and not)
    }
    if (variant == 1 && a.precise) variant = 2;   // (col16_kernel has no split mode)
    if (variant == 1 || variant == 2) {
        int rc = variant == 1 ? launch_col16_kernel(dtype, D, a, st) : launch_cold_kernel(dtype, D, a, st);
        if (rc != MLSTM_ESHAPE) return rc;  // extremely long sequences do not fit their LDS budget
    }
    return launch_col_kernel(dtype, D, a, st);
}

struct DfArgs {
    const void* F; const float* colsum; const float* rowpart;
    void* dF; void* dI;
    int BH, S, NG;
    int RS;                  // row-partial slices per head (see ColArgs)
    const float* rowpart2;   // may be null: the partials of the tiles' second halves (see ColArgs)
    bool pairs;              // the slices are added up in pairs first (the order of a kernel whose tiles are twice as wide: see colw_serves)
    // in chunks: rowpart holds the slices of the key tiles of the position's own chunk only, rowinter the rest
    int chunk_len;
    const float* rowinter;
    const float* anchor;     // [BH][n_states]: the running sum of (col - row) at the first position of chunks 1, 2, ...
    int n_states;
    Lay lg;                  // layout of F, dF and dI
    int gate_form;           // what F holds (see launch_gates); dF is the gradient of that same quantity
    // chunk_len <= 1024: the anchors come as partial sums instead (ChunkArgs::dot_part of the reverse states) and the
    // vector states of both directions, and the kernel adds them up itself
    const float* anchor_part = nullptr;   // [BH][n_states][anchor_parts]
    int anchor_parts = 0;
    const float* anchor_va = nullptr;     // [BH][n_states][D] each
    const float* anchor_vb = nullptr;
    int D = 0;
    SavedStamp stamp;        // compared by the first workgroup (src), if set
};
int launch_df(int gate_dtype, const DfArgs& a, hipStream_t st);

// States at the ends of the first NCS chunks of L positions of every head (16-bit types, D = 128 or 256), for the
// chunked forward of RowArgs: dC is scratch, Nst and Cst receive the states.
struct ChunkArgs {
    const void* K;
    const void* V;        // [BH,S,D]
    const float* alpha2;
    const float* beta2;
    const double* G2;
    float* dC;            // [BH][NCS][D][D] fp32 scratch: the chunks' own sums
    float* Nst;           // [BH][NCS][D]
    void* Cst;            // [BH][NCS][D][D], key-major: the forward contracts it over the key index; may be null
    void* CstT;           // the same states value-major, for the dQ pass; may be null
    int BH, S, NG, L, NCS;
    // reverse states for the keys of a chunk, summed over the queries behind it: K = Q, V = dH,
    //   E_c = sum_{i > e_c} exp(A_{e_c} - A_i) q_i (dh_i / n_i)^T / sqrt(D)  (Cst / CstT),  g_c likewise with db_i (Nst);
    // inv_n and db are the per-row scalars the dQ pass leaves
    int reverse;
    const float* inv_n;
    const float* db;
    Lay lk, lv;           // layouts of K and V
    // Split mode: the weighted V rows enter the chunk sums as two terms (hi + lo, two MFMAs per fragment) and every state
    // is written as two terms as well: Cst_lo / CstT_lo receive state - (state rounded to the element type), rounded.
    int precise;
    void* Cst_lo;
    void* CstT_lo;
    // What writes the value-major states can contract them, as it writes them, with another set in the same layout (dot_with,
    // dot_with_lo: its low-order terms or null): dot_part[bh][c][block] receives the partial sums of <state_c, dot_with_c>, one
    // per block of 32 keys x 32 values (block = key block * D / 32 + value block).
    const void* dot_with = nullptr;
    const void* dot_with_lo = nullptr;
    float* dot_part = nullptr;
};
int launch_chunk_states(int dtype, int D, const ChunkArgs& a, hipStream_t st);
// test and measurement aid: 0 = the library's choice by the size of the launch, 1 = chunk sums and carry (two kernels),
// 2 = the one-pass kernel wherever it can serve
int set_state_kernel(int variant);

// anchor[bh][c] = <A_c, B_c> + va_c . vb_c over two sets of states in the same layout; A_lo, B_lo (both or neither): their low-order
// terms (split mode).  Only for chunks of more than 1024 positions, which mlstm_set_chunk_length alone asks for: with shorter ones the
// reverse carry leaves the anchors in parts.
int launch_anchor(int dtype, int D, const void* A, const void* B, const void* A_lo, const void* B_lo, const float* va, const float* vb,
                  float* anchor, int BH, int NCS, hipStream_t st);

// Backward of the output gate h_out = silu(o) * h, element-wise over n elements (n a multiple of 8):
//   dh = dh_out * silu(o)   (the upstream gradient of the ungated form),   d_o = dh_out * h * silu'(o).
int launch_gate_backward(int dtype, const void* dh_out, const void* o, const void* h, void* dh, void* d_o, size_t n, hipStream_t st);
// the same over [BH, S, D] tensors in layouts: dh_out, o, d_o in lx, h in lh, dh in ld
int launch_gate_backward_rows(int dtype, const void* dh_out, const void* o, const void* h, void* dh, void* d_o, int BH, int S, int D,
                              const Lay& lx, const Lay& lh, const Lay& ld, hipStream_t st);

struct ScanArgs {
    const float* q; const float* k; const float* v; const float* o;
    float* h;             // unnormalised numerator (first key range), then the output
    float* hpart;         // [parts-1, BH, S, D] numerators of the other key ranges
    int shared;           // key ranges 2p and 2p+1 add to one partial numerator p (parts = scan_key_parts)
    const float* alpha2; const float* beta2; const double* G2; const float* M;
    float* P;             // [BH, NC, 64, 64] in-chunk pair weights
    float* Nst;           // [BH, NC, D] vector state n~ at every chunk end
    int BH, S, D, NC;
    // What the last kernel writes to h: 0 = silu(o) * numerator / n (the scan form's output), 1 = numerator / n (ungated),
    // 2 = the numerator itself, sum_j exp(a_j - A_t) (q_t . k_j) / sqrt(D) v_j: the causal weighted sum the backward pass
    // reuses with other operands in the places of q, k and v, finished as `ep` says.  Bout (may be null): the normaliser
    // sums b_t, modes 0 and 1.
    int finish_mode;
    float* Bout;
    float* Hun;           // mode 0 only, may be null: numerator / n next to the gated output (what a backward wants kept)
    // rev (mode 2 only): q, k and v hold the sequence in its own order and the pipeline walks it from the end: position t
    // of the walk is row S-1-t of q, k and v.  Gate arrays, P, Nst, h and hpart are in walk order.
    int rev;
    // Mode 2 can carry a vector sum along with the matrix one (ep.vec):
    //   numerator_t = sum_{j<=t} exp(a_j - A_t) / sqrt(D) ((q_t . k_j) + rs_t cs_j) v_j
    // rs = ep.row_scale ([BH,S], walk order; null: 1), cs = col_scale ([BH,S], in the order of the rows of q, k, v; null: 1).
    // The pairs inside a chunk take the term into their weights P; the chunks before it come through Nst, which then holds
    // sum_j exp(a_j - A_end) / sqrt(D) cs_j v_j at the chunk ends.  What the last kernel then does with row t:
    //   x = numerator_t (+ rs_t decay_t Nst_{c-1}),  x *= exp2(wd_alpha2_j - wd_beta2_j)  (gate arrays of the output row j; may be null)
    //   out_j = x  with j = t, or S-1-t when out_rev             (out null: h, in place; out_rev needs out != h)
    //   dot_out_j = dot_with_j . x,  x_out_j = dot_out_j - dot_minus_j                              (each may be null)
    const float* col_scale;
    struct Epilogue {
        float* out; int out_rev;
        int vec; const float* row_scale;
        const float* wd_alpha2; const float* wd_beta2;
        const float* dot_with; float* dot_out; const float* dot_minus; float* x_out;
    } ep;
    // segments of the sequence that the state kernel runs side by side (filled in by launch_scan from scan_segments);
    // seg_state: scan_segment_state_bytes() bytes of scratch for the states at the segment ends, needed when nseg > 1
    float* seg_state;
    int nseg, seg_chunks;
};
int scan_key_splits(int BH, int D);
// Partial numerators of a walk: one per key range, or (shared) one per pair of them, where scan_can_share(BH, D)
bool scan_can_share(int BH, int D);
int scan_key_parts(int BH, int D, bool shared);
void scan_segments(int BH, int S, int D, int* nseg, int* seg_chunks);
size_t scan_segment_state_bytes(int BH, int S, int D);
// mark(kernel id, stream, begin?) brackets groups of launches for the optional event timing
int launch_scan(const ScanArgs& a, int KS, hipStream_t st, void (*mark)(int, hipStream_t, bool));
// n~ at every chunk end from the chunks' own sums, in place (ScanArgs::Nst, beta2, G2, BH, NC, D are read)
void launch_scan_ncarry(const ScanArgs& a, hipStream_t st);

// Backward of the scan form (mlstm_scan_bwd.hip): every pointer fp32, [B,NH,S,D] or [B,NH,S]; ws holds
// scan_backward_workspace_bytes(BH, S, D) bytes.  o == null: no output gate (dhg is the gradient of the ungated
// output, d_o is not written)
struct ScanBwdArgs {
    const float* dhg; const float* q; const float* k; const float* v; const float* f; const float* i; const float* o;
    float* dq; float* dk; float* dv; float* df; float* di; float* d_o;
    int BH, S, D;
    // the forward's ungated output and normaliser sums, if the caller kept them (both or neither): the forward is then not
    // run again
    const float* h_kept; const float* b_kept;
};
size_t scan_backward_workspace_bytes(int BH, int S, int D);
int launch_scan_backward(const ScanBwdArgs& a, char* ws, hipStream_t st, void (*mark)(int, hipStream_t, bool));
// dF_t = sigmoid(-f_t) * sum_{s<t} x_s over each head (x: [BH,S] fp32; dF_0 = 0): the scan of launch_df on its own
int launch_dfscan_plain(int gate_dtype, const void* F, const float* x, void* dF, int BH, int S, hipStream_t st);

}  // namespace mlstm
