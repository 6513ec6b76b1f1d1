// The gated delta rule's arguments and per-token form, shared by its kernels
// (hybrid.hip, gdn_scan.hip).
#pragma once

#include "gdn_plan.h"
#include "qsa_common.h"

namespace qsa {

constexpr int kHeadDim = 128;

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

constexpr int kRecTokens = 16;  // tokens staged in LDS per block

struct GdnRecurLds {
  float sq[kRecTokens][kHeadDim];
  float sk[kRecTokens][kHeadDim];
  float sv[kRecTokens][kHeadDim];
  float sg[kRecTokens], sb[kRecTokens];
};

__device__ __forceinline__ void unpack8(const u32x4& v, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = bf16_lo(v[i]);
    f[2 * i + 1] = bf16_hi(v[i]);
  }
}

// The per-token rule for (sequence, value head) number `block`, 4 waves:
// sequences shorter than chunk_min.
__device__ __forceinline__ void gdn_recurrence_block(const GdnRecurArgs& a, int block, GdnRecurLds& L) {
  const int h = block % a.value_heads;
  const int seq = a.num_seqs - 1 - (int)(block / a.value_heads);  // longest (prefill) first
  const int m = h / (a.value_heads / a.key_heads);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = 32 * wave + (lane & 31);
  const int half = lane >> 5;
  const int start = a.seq_start[seq], len = a.seq_start[seq + 1] - start;
  if (len <= 0 || len >= a.chunk_min || start < 0 || start + len > a.tokens) return;
  const int64_t slot = a.slots[seq];
  const bool slot_ok = slot >= 0 && slot < a.num_slots;
  float* sp = a.state + ((slot_ok ? slot : 0) * a.value_heads + h) * (int64_t)(kHeadDim * kHeadDim) +
              (int64_t)(64 * half) * kHeadDim + j;
  float S[64];
#pragma unroll
  for (int i = 0; i < 64; ++i) S[i] = slot_ok ? sp[(int64_t)i * kHeadDim] : 0.0f;
  for (int b0 = 0; b0 < len; b0 += kRecTokens) {
    const int nb = min(kRecTokens, len - b0);
    // stage: thread -> (token tt = tid / 16, 8 dims at 8 (tid % 16))
    {
      const int tt = threadIdx.x >> 4, d0 = 8 * (threadIdx.x & 15);
      if (tt < nb) {
        const int64_t t = start + b0 + tt;
        const float* qp = a.q + (t * a.key_heads + m) * kHeadDim + d0;
        const float* kp = a.k + (t * a.key_heads + m) * kHeadDim + d0;
        *reinterpret_cast<f32x4*>(&L.sq[tt][d0]) = *reinterpret_cast<const f32x4*>(qp);
        *reinterpret_cast<f32x4*>(&L.sq[tt][d0 + 4]) = *reinterpret_cast<const f32x4*>(qp + 4);
        *reinterpret_cast<f32x4*>(&L.sk[tt][d0]) = *reinterpret_cast<const f32x4*>(kp);
        *reinterpret_cast<f32x4*>(&L.sk[tt][d0 + 4]) = *reinterpret_cast<const f32x4*>(kp + 4);
        float vv[8];
        unpack8(load_u32x4(a.v + (t * a.value_heads + h) * kHeadDim + d0), vv);
#pragma unroll
        for (int e = 0; e < 8; ++e) L.sv[tt][d0 + e] = vv[e];
        if ((threadIdx.x & 15) == 0) {
          L.sg[tt] = a.g[t * a.value_heads + h];
          L.sb[tt] = a.beta[t * a.value_heads + h];
        }
      }
    }
    __syncthreads();
    for (int tt = 0; tt < nb; ++tt) {
      const float* kr = &L.sk[tt][64 * half];
      float p0 = 0.0f, p1 = 0.0f, p2 = 0.0f, p3 = 0.0f;
#pragma unroll
      for (int i = 0; i < 64; i += 4) {
        const f32x4 kv = *reinterpret_cast<const f32x4*>(kr + i);
        p0 += kv[0] * S[i];
        p1 += kv[1] * S[i + 1];
        p2 += kv[2] * S[i + 2];
        p3 += kv[3] * S[i + 3];
      }
      const float ks = sum_wave_halves((p0 + p1) + (p2 + p3));
      const float decay = expf(L.sg[tt]);
      const float u = L.sb[tt] * (L.sv[tt][j] - decay * ks);
#pragma unroll
      for (int i = 0; i < 64; i += 4) {
        const f32x4 kv = *reinterpret_cast<const f32x4*>(kr + i);
        S[i] = S[i] * decay + kv[0] * u;
        S[i + 1] = S[i + 1] * decay + kv[1] * u;
        S[i + 2] = S[i + 2] * decay + kv[2] * u;
        S[i + 3] = S[i + 3] * decay + kv[3] * u;
      }
      const float* qr = &L.sq[tt][64 * half];
      p0 = p1 = p2 = p3 = 0.0f;
#pragma unroll
      for (int i = 0; i < 64; i += 4) {
        const f32x4 qv = *reinterpret_cast<const f32x4*>(qr + i);
        p0 += qv[0] * S[i];
        p1 += qv[1] * S[i + 1];
        p2 += qv[2] * S[i + 2];
        p3 += qv[3] * S[i + 3];
      }
      const float os = sum_wave_halves((p0 + p1) + (p2 + p3));
      if (half == 0) {
        const int64_t t = start + b0 + tt;
        const __bf16 ob = (__bf16)os;
        a.o[(t * a.value_heads + h) * kHeadDim + j] = __builtin_bit_cast(uint16_t, ob);
      }
    }
    __syncthreads();
  }
  if (slot_ok) {
#pragma unroll
    for (int i = 0; i < 64; ++i) sp[(int64_t)i * kHeadDim] = S[i];
  }
}

// The two-launch chunked form (gdn_scan.hip): workspace it needs, and its
// launches, which take every sequence (those below chunk_min with the per-token rule).
size_t gdn_scan_workspace_bytes(int tokens, int num_seqs, int key_heads, int value_heads);
int gdn_scan_launch(const GdnRecurArgs& a, int max_seq_tokens, void* workspace, hipStream_t stream);

}  // namespace qsa
