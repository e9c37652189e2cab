// Launch interface of the matrix-core one-launch forward (onepass_mfma.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"

namespace cdssm {

// One inference forward of the readout form on scan-level bf16 inputs.
struct MfmaForward {
  const void *q, *k, *v, *beta, *sel_c, *dt, *r;
  const float *alpha, *omega;
  float c;
  const float* h0;
  void* y;
  float* h_final;
  float2* lookback;  // the look-back area of the workspace (FwdLayout::n_op float2s)
  int B, L, H, D, Q;
  bool cont;
  unsigned long long* stamps;  // or null
  int64_t stamps_len;
};

// Whether one round of resident workgroups takes every segment (each may wait on any earlier one).
bool mfma_forward_fits(int64_t B, int64_t L, int64_t H, int D, int Q);
// ev: five events recorded as by the other one-launch forwards, or null.
int launch_mfma_forward(const MfmaForward& p, hipStream_t stream, hipEvent_t* ev);
// Sticky look-back status word of this unit (bit kTimeoutFwd).
int mfma_forward_status(bool clear, unsigned* out);

}  // namespace cdssm
