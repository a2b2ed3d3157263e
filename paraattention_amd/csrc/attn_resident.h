// The attention kernel for keys that fit the LDS of one compute unit (attn_resident.hip).
#pragma once

#include "pa_common.h"

namespace pa {

struct ResidentCall {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  float* lse;  // may be null
  int B, H, Sq, Skv;
  int64_t qs_b, qs_h, qs_s;
  int64_t ks_b, ks_h, ks_s;
  int64_t vs_b, vs_h, vs_s;
  int64_t os_b, os_h, os_s;
  float scale_log2;
  const void* bias;  // additive, no query dimension; null: none
  int64_t ms_b, ms_h, ms_k;
  int bias_act;      // its elements have the activation type (else fp32)
  // the plan (plan_resident)
  int n_units;       // blocks of 32 query rows per (batch, head)
  int n_full;        // whole tiles of 64 keys
  int parts;         // workgroups per (batch, head)
  int xcd_chunk;     // workgroups per XCD, 0: plain order
};

// Whether the kernel takes the call.  want: -1 where it is expected to be the fastest, 1 wherever it can run.
bool resident_takes(ResidentCall& c, int D, int want);
// The same, and fills the plan's fields.
bool plan_resident(ResidentCall& c, int D, int want);
int launch_resident(const ResidentCall& c, int dtype, int D, hipStream_t stream);

}  // namespace pa
