// Arguments of the gated delta rule's kernels (hybrid.hip, gdn_scan.hip).
#pragma once

#include "qsa_common.h"

namespace qsa {

constexpr int kGdnChunkMin = 16;  // sequences this long take a chunked kernel

struct GdnRecurArgs {
  const float* q;  // [tokens, key_heads, 128]
  const float* k;
  const uint16_t* v;  // [tokens, value_heads, 128]
  const float* g;     // [tokens, value_heads]
  const float* beta;
  float* state;  // [slots, value_heads, 128, 128]
  const int* seq_start;
  const int64_t* slots;
  int num_seqs, key_heads, value_heads, num_slots, tokens;
  uint16_t* o;  // [tokens, value_heads, 128]
  int chunk_min;  // sequences this long go to a chunked kernel, shorter ones to the per-token kernel
};

// The two-launch chunked form (gdn_scan.hip): workspace it needs, and its
// launches for the sequences of chunk_min tokens or more.
size_t gdn_scan_workspace_bytes(int tokens, int num_seqs, int key_heads, int value_heads);
int gdn_scan_launch(const GdnRecurArgs& a, int max_seq_tokens, void* workspace, hipStream_t stream);

}  // namespace qsa
