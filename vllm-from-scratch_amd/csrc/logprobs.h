// Host/device interface of the speculative-logprobs kernel (logprobs.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mvsd {

struct LogprobParams {
  const void* target;          // verify rows, row stride tstride (elements)
  int64_t tstride;
  int64_t target_num_rows;     // rows of `target` that a row index is clamped to, or 0 (any)
  const int32_t* target_rows;  // [P] row of verify row v in `target`, or null (row v)
  const void* bonus;           // bonus rows, row stride bstride
  int64_t bstride;
  int64_t bonus_num_rows;      // as target_num_rows
  const int32_t* bonus_rows;   // [B] row of request q's bonus row in `bonus`, or null (row q)
  const int32_t* cu_sampled;   // [B] cumulative K_r + 1, no leading 0
  const void* tokens;          // [B, W] sampled ids (int32, or int64 with tokens64), -1 padded
  int64_t tok_stride;
  int B, P, V, W, k;
  int logits_mode;             // 1: report the values themselves, 0: their log-softmax
  int flat;                    // 1: position n reads row bonus + n * bstride, token tokens[n]
  int rank_raw;                // 1: top-k order and rank compare raw values, not log-softmax
  int tokens64, ids64;         // 64-bit token ids read / ids and ranks written
  void* ids;                   // [B * W, k + 1]
  float* lps;                  // [B * W, k + 1]
  void* ranks;                 // [B * W]
  // split path: per position and chunk, and per position and group of lanes (logprobs.hip)
  float4* stats;
  uint32_t* group_keys;
  int nchunks;
};

// One workgroup per position: fp32 rows, int32 ids, any 0 <= k <= V, no workspace.
hipError_t launch_spec_logprobs(const LogprobParams& p, hipStream_t stream);

// Rows split over workgroups (fp32 / bf16 / fp16 rows).  The workspace size is 0 where the
// split path does not apply.
int64_t split_logprobs_workspace_bytes(int64_t positions, int64_t V, int64_t k);
hipError_t launch_split_logprobs(LogprobParams p, int dtype, void* workspace, hipStream_t stream);

}  // namespace mvsd
