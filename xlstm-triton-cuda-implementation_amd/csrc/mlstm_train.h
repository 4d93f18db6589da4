// The training step of the matmul form (with or without the output gate) as the host path behind torch calls it: a forward
// that leaves what its backward needs in ONE buffer of the caller's -- m, b, what mlstm_forward_save_lx saves (chunk states and
// gate pre-pass of a long sequence, the low-order part of h in split mode), and for sequences that do not run in chunks the
// gate pre-pass -- and the backward that reads it.  Same kernels and results as the entry points of include/mlstm_hip.h.
#pragma once
#include <stddef.h>
#include "../../include/mlstm_hip.h"

namespace mlstm {
size_t train_kept_bytes(int B, int NH, int S, int D, int dtype);
// o, h_gated, dh (then the gradient of h_gated) and d_o: the gated form, or all null; layout: null = dense tensors
int train_forward(const void* q, const void* k, const void* v, const void* f, const void* i, const void* o, void* h, void* h_gated, void* kept, size_t kept_bytes, int B,
                  int NH, int S, int D, int dtype, int gate_dtype, const mlstm_layout* layout, void* workspace, size_t workspace_bytes, void* stream);
int train_backward(const void* dh, const void* q, const void* k, const void* v, const void* f, const void* i, const void* o, const void* h,
                   const void* kept, size_t kept_bytes, void* dq, void* dk, void* dv, void* df, void* di, void* d_o, int B, int NH, int S, int D, int dtype,
                   int gate_dtype, const mlstm_layout* layout, void* workspace, size_t workspace_bytes, void* stream);
}  // namespace mlstm
