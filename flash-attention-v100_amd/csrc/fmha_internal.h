// What the PyTorch extension uses of the kernel library beside its public interface (fused_mha.h).
#ifndef FMHA_INTERNAL_H_
#define FMHA_INTERNAL_H_

#include "fused_mha.h"

extern "C" {

// fused_mha_forward_strided for callers without a backward pass: the logsumexp is not written.
int fmha_forward_without_lse(const void* query_ptr, const fused_mha_strides* query_strides, const void* key_ptr,
                             const fused_mha_strides* key_strides, const void* value_ptr,
                             const fused_mha_strides* value_strides, void* output_ptr, int batch, int head, int n, int d,
                             float scale, int causal, void* stream);

// fused_mha_backward_workspace_bytes for callers that can spare `room` bytes: the size of at most that (and at least the
// minimum) with which the backward is fastest.  0 for an invalid shape.
size_t fmha_backward_workspace_within(int batch, int head, int n, int d, size_t room);

// fused_mha_backward_workspace_bytes for one backward: the minimum where that needs no room for dS, since it does both passes in
// one launch or takes a work group for each slice.
size_t fmha_backward_workspace_for(int batch, int head, int n, int d, int causal);

// Bytes behind room for the dS of all slices with which a backward of this shape does both passes over dS in one launch; 0 where
// it does not.
size_t fmha_backward_count_bytes(int batch, int head, int n, int d, int causal);

// fused_mha_backward by its passes also where that takes a work group for each slice, and with a limit of the caller's, in ticks
// of 10 ns, to how long a block of a launch of both passes over dS waits for another's dS before it forms S and dP itself.  The
// counts behind the dS are, per slice, the waves that have stored dS, the dK/dV blocks that have started (of the last slices % 8
// only) and the dQ blocks that have done without, then 29 zeros.
int fmha_backward_waiting(const void* query_ptr, const void* key_ptr, const void* value_ptr, const void* output_ptr,
                          const void* d_output_ptr, const void* lse_ptr, void* workspace, size_t workspace_bytes,
                          void* d_query_ptr, void* d_key_ptr, void* d_value_ptr, int batch, int head, int n, int d, float scale,
                          int causal, unsigned ticks, void* stream);

}  // extern "C"
#endif  // FMHA_INTERNAL_H_
