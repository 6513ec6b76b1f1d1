// Chunked gated delta rule in two launches, gfx950.
//
// Over a chunk of C = 64 tokens, with G the in-chunk cumulative log decay,
// gamma = e^G and S the state at the chunk's start:
//   A[t][s] = beta_t e^{G_t - G_s} k_t.k_s (s < t),  T = (I + A)^-1 diag(beta)
//   U = T (V - gamma (K S)),  O = gamma (Q S) + P U,  P[t][s] = e^{G_t - G_s} q_t.k_s (s <= t)
//   S <- gamma_C S + K^T (e^{G_C - G} U)
// Only S passes from chunk to chunk. gdn_chunk_operands_kernel computes what
// does not depend on it (T, P, the gates, and K, Q, K^T in bf16) for every
// chunk of the batch at once, one workgroup per (chunk, key head), and leaves
// it in the order in which the MFMA operands are held. gdn_scan_kernel then
// walks a sequence's chunks with the rest. Value columns never mix, so a
// (sequence, value head) is cut into 16 NL-column slices that run on
// different CUs.
//
// The one-launch kernel (gdn_chunk_kernel) does all of it chunk after chunk in
// one workgroup per (sequence, value head): ~14 us a chunk, and one prompt of
// 8192 tokens kept 16 workgroups busy for 1812 us. Here it takes 44 us for the
// operands (73 MB written, 67 MB of fp32 q and k read) and 117 us for the walk
// (0.9 us a chunk, bound by the state waves' chain of products).
//
// Bits: gdn_chunk_kernel solves for U in fp32. Here T is formed in fp32 (the
// diagonal blocks' inverses, their products) and R in fp32, but both enter the
// product U = T R as two bf16 halves, 16 significant bits, without the product
// of the lower halves. U goes on in bf16 in both kernels. K^T (e^{G_C - G} U)
// rounds the scaled U; the other kernel rounds the scaled K, which was rounded
// before, and U. Against 64 bits, over 26 batches of the serving ranges, a mixer's
// output is 0.988 to 1.000 times and its state 0.89 to 0.99 times as far off as
// with the one-launch kernel; with keys from orthogonal to all but parallel
// (k.k 0.99), beta up to 1 and decay from none to e^-0.5 a token 0.94 to 1.004
// and 0.78 to 1.001 times.
#include "gdn_device.h"
#include "../../include/qsa_hip.h"

namespace qsa {
namespace {

constexpr int kDim = 128;
constexpr int kC = kGdnChunk;  // tokens per chunk
// A fragment is one MFMA operand of a wave: 64 lanes x 8 bf16.
constexpr int kFrag = 512;  // bf16 elements
// Per (chunk, key head): K and Q, 16 fragments each.
constexpr int kQFrag = 16;
constexpr int kKeyElems = 32 * kFrag;
// Per (chunk, value head): T's upper and lower halves (6 fragments each), one
// fragment's room with gamma and e^{G_C - G} (64 fp32 each), then P (6).
constexpr int kGateFrag = 12, kPFrag = 13;
constexpr int kValElems = 19 * kFrag;

// Where a fragment of K keeps lane (m, g)'s operand. K is also read transposed
// (read_kt), 4 tokens x 16 dims by each 16 lanes; rotating the tokens by the
// lane group puts those 16 addresses in distinct LDS banks.
__device__ __forceinline__ constexpr int key_lane(int m, int g) { return 16 * g + ((m + 4 * g) & 15); }

// Lower-triangular 64 x 64 operands keep the fragments (ct, ks) of 16 rows x
// 32 columns that reach the diagonal: (0, 0) (1, 0) (2, 0) (2, 1) (3, 0) (3, 1).
__device__ __forceinline__ constexpr int tri(int ct, int ks) { return ct < 2 ? ct : 2 * ct - 2 + ks; }

__device__ __forceinline__ uint16_t to_bf16(float x) {
  const __bf16 b = (__bf16)x;
  return __builtin_bit_cast(uint16_t, b);
}

// Orders a wave's own LDS writes before its later reads of other lanes' data
// (the LDS serves one wave in issue order; this holds the compiler to it).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The sequences that take the chunked kernels (gdn_first_slot has their workspace slots).
__device__ __forceinline__ bool chunked_sequence(const GdnRecurArgs& a, int seq, int* start, int* len) {
  *start = a.seq_start[seq];
  *len = a.seq_start[seq + 1] - *start;
  return *len >= a.chunk_min && *start >= 0 && *start <= a.tokens - *len;
}

// The 32-deep slice ks of a token- or dim-indexed operand pairs 16-row tiles
// 2 ks and 2 ks + 1: element j of lane group g is row 16 (2 ks + (j >> 2)) +
// 4 g + (j & 3), the rows that an accumulator tile leaves in that lane group,
// so S, R and U go from accumulators to B operands without leaving the lane.
__device__ __forceinline__ int slice_row(int ks, int g, int j) {
  return 32 * ks + 16 * (j >> 2) + 4 * g + (j & 3);
}

// ---------------------------------------------------------------------------
// Operands of every chunk. 4 waves; wave w owns row tile w of K K^T and Q K^T,
// the diagonal block w of I + A (inverted by forward substitution, lane j <
// 16 its column j) and block column w of T (fp32 MFMA products of the blocks
// below the diagonal).
// ---------------------------------------------------------------------------
struct OperandLds {
  union {
    struct {
      uint16_t q[kC][136];
      uint16_t k[kC][136];
    };
    struct {
      float a[kC][68];     // strict lower triangle of A
      float t[kC][68];     // (I + A)^-1, blocks on and below the diagonal
      uint16_t p[kC][72];
    };
  };
  float G[kC], beta[kC];
};

__device__ __forceinline__ void chunk_operands(const GdnRecurArgs& a, uint16_t* __restrict__ ws,
                                               int ws_slots, int slot, int hk, OperandLds& L) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int m = lane & 15, g = lane >> 4;
  // The sequence whose chunks cover this slot (none: padding between sequences).
  int seq = -1, start = 0, len = 0;
  const bool mostly_short = gdn_mostly_short(a.tokens, a.num_seqs);
  for (int i0 = 0; i0 < a.num_seqs && seq < 0; i0 += 64) {
    const int i = min(i0 + lane, a.num_seqs - 1);
    int s0, n;
    const bool chunked = chunked_sequence(a, i, &s0, &n);
    const int at = slot - gdn_first_slot(s0, i, mostly_short);
    const uint64_t hit = __ballot(chunked && at >= 0 && at < (n + kC - 1) / kC);
    if (hit) {
      const int src = __builtin_ctzll(hit);
      seq = i0 + src;
      start = __builtin_amdgcn_readlane(s0, src);
      len = __builtin_amdgcn_readlane(n, src);
    }
  }
  if (seq < 0) return;
  const int c0 = (slot - gdn_first_slot(start, seq, mostly_short)) * kC;
  const int nc = min(kC, len - c0);
  const int r = a.value_heads / a.key_heads;

  {  // K and Q to bf16: thread -> row tid / 4, dims 32 (tid % 4) .. + 31; rows past the end are 0.
    const int row = tid >> 2, d0 = 32 * (tid & 3);
    const bool live = row < nc;
    const int64_t at = ((int64_t)(start + c0 + min(row, nc - 1)) * a.key_heads + hk) * kDim + d0;
    f32x4 qv[8], kv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      qv[e] = *reinterpret_cast<const f32x4*>(a.q + at + 4 * e);
      kv[e] = *reinterpret_cast<const f32x4*>(a.k + at + 4 * e);
    }
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const u32x4 qb = {pack_bf16x2(qv[e][0], qv[e][1]), pack_bf16x2(qv[e][2], qv[e][3]),
                        pack_bf16x2(qv[e + 1][0], qv[e + 1][1]), pack_bf16x2(qv[e + 1][2], qv[e + 1][3])};
      const u32x4 kb = {pack_bf16x2(kv[e][0], kv[e][1]), pack_bf16x2(kv[e][2], kv[e][3]),
                        pack_bf16x2(kv[e + 1][0], kv[e + 1][1]), pack_bf16x2(kv[e + 1][2], kv[e + 1][3])};
      const u32x4 zero = {0, 0, 0, 0};
      *reinterpret_cast<u32x4*>(&L.q[row][d0 + 4 * e]) = live ? qb : zero;
      *reinterpret_cast<u32x4*>(&L.k[row][d0 + 4 * e]) = live ? kb : zero;
    }
  }
  __syncthreads();
  uint16_t* key_ws = ws + ((int64_t)slot * a.key_heads + hk) * kKeyElems;
  // Fragments of K and Q, rows 16 w + m.
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const int lo = slice_row(ks, g, 0), hi = slice_row(ks, g, 4);
    const u32x2 k0 = load_u32x2(&L.k[16 * w + m][lo]), k1 = load_u32x2(&L.k[16 * w + m][hi]);
    const u32x2 q0 = load_u32x2(&L.q[16 * w + m][lo]), q1 = load_u32x2(&L.q[16 * w + m][hi]);
    *reinterpret_cast<u32x4*>(key_ws + (4 * w + ks) * kFrag + 8 * key_lane(m, g)) = u32x4{k0[0], k0[1], k1[0], k1[1]};
    *reinterpret_cast<u32x4*>(key_ws + (kQFrag + 4 * w + ks) * kFrag + 8 * lane) = u32x4{q0[0], q0[1], q1[0], q1[1]};
  }
  // Raw K K^T and Q K^T of row tile w: rows 16 w + 4 g + i, columns 16 ct + m.
  f32x4 kk[4], qk[4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    kk[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    qk[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (ct > w) continue;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const bf16x8 b = __builtin_bit_cast(bf16x8, load_u32x4(&L.k[16 * ct + m][32 * ks + 8 * g]));
      const bf16x8 ak = __builtin_bit_cast(bf16x8, load_u32x4(&L.k[16 * w + m][32 * ks + 8 * g]));
      const bf16x8 aq = __builtin_bit_cast(bf16x8, load_u32x4(&L.q[16 * w + m][32 * ks + 8 * g]));
      kk[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ak, b, kk[ct], 0, 0, 0);
      qk[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aq, b, qk[ct], 0, 0, 0);
    }
  }
  for (int hl = 0; hl < r; ++hl) {
    const int h = hk * r + hl;
    uint16_t* val_ws = ws + (int64_t)ws_slots * a.key_heads * kKeyElems +
                       ((int64_t)slot * a.value_heads + h) * kValElems;
    __syncthreads();  // K and Q (or the previous head's A, T, P) have been read
    if (w == 0) {     // gates of row `lane`, inclusive prefix sum of g
      const int64_t t = start + c0 + min(lane, nc - 1);
      float gv = lane < nc ? a.g[t * a.value_heads + h] : 0.0f;
      const float bv = lane < nc ? a.beta[t * a.value_heads + h] : 0.0f;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const float o = __shfl_up(gv, d, 64);
        if (lane >= d) gv += o;
      }
      L.G[lane] = gv;
      L.beta[lane] = bv;
      float* gates = reinterpret_cast<float*>(val_ws + kGateFrag * kFrag);
      const float total = __shfl(gv, 63, 64);
      gates[lane] = expf(gv);
      gates[kC + lane] = expf(total - gv);
    }
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      if (ct > w) continue;
      const int sc = 16 * ct + m;
      const float Gs = L.G[sc];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tr = 16 * w + 4 * g + i;
        const float e = sc <= tr ? expf(L.G[tr] - Gs) : 0.0f;
        L.a[tr][sc] = sc < tr ? L.beta[tr] * e * kk[ct][i] : 0.0f;
        L.p[tr][sc] = to_bf16(e * qk[ct][i]);
      }
    }
    // Wave w wrote rows 16 w .. 16 w + 15 of A, so it inverts the diagonal
    // block w without a barrier.
    wave_lds_order();
    if (lane < 16) {
      const int j = lane;
      float x[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float* arow = &L.a[16 * w + i][16 * w];
        float p0 = i == j ? 1.0f : 0.0f, p1 = 0.0f;
#pragma unroll
        for (int s2 = 0; s2 < i; ++s2) {
          if (s2 & 1) p1 -= arow[s2] * x[s2];
          else p0 -= arow[s2] * x[s2];
        }
        x[i] = p0 + p1;
        L.t[16 * w + i][16 * w + j] = x[i];
      }
    }
    __syncthreads();
    // Block column w below the diagonal: T_iw = -T_ii sum_{w <= k < i} A_ik T_kw.
    // v_mfma_f32_16x16x4f32: lane (m, g) holds A[m][g] and B[g][m]. The wave
    // reads back only its own block column and the diagonal blocks.
    for (int i = w + 1; i < 4; ++i) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      for (int k0 = 16 * w; k0 < 16 * i; k0 += 4)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(L.a[16 * i + m][k0 + g], L.t[k0 + g][16 * w + m],
                                                   acc, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) L.t[16 * i + 4 * g + e][16 * w + m] = acc[e];
      wave_lds_order();
      f32x4 out = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k0 = 0; k0 < 16; k0 += 4)
        out = __builtin_amdgcn_mfma_f32_16x16x4f32(-L.t[16 * i + m][16 * i + k0 + g],
                                                   L.t[16 * i + k0 + g][16 * w + m], out, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) L.t[16 * i + 4 * g + e][16 * w + m] = out[e];
      wave_lds_order();
    }
    __syncthreads();
    // Fragments of T diag(beta), split into two bf16 halves (16 significant
    // bits), and of P: rows 16 w + m.
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (32 * ks > 16 * w) continue;
      uint32_t hi[8], lo[8], pp[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int col = slice_row(ks, g, j);
        const bool in = (col >> 4) <= w;
        const float x = in ? L.t[16 * w + m][col] * L.beta[col] : 0.0f;
        hi[j] = to_bf16(x);
        lo[j] = to_bf16(x - __builtin_bit_cast(float, hi[j] << 16));
        pp[j] = in ? L.p[16 * w + m][col] : 0;
      }
      u32x4 vh, vl, vp;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        vh[j] = hi[2 * j] | (hi[2 * j + 1] << 16);
        vl[j] = lo[2 * j] | (lo[2 * j + 1] << 16);
        vp[j] = pp[2 * j] | (pp[2 * j + 1] << 16);
      }
      const int f = w < 2 ? w : 2 * w - 2 + ks;
      *reinterpret_cast<u32x4*>(val_ws + f * kFrag + 8 * lane) = vh;
      *reinterpret_cast<u32x4*>(val_ws + (6 + f) * kFrag + 8 * lane) = vl;
      *reinterpret_cast<u32x4*>(val_ws + (kPFrag + f) * kFrag + 8 * lane) = vp;
    }
  }
}

// One launch for the chunks' operands and the short sequences' per-token rule,
// alternating, so that neither leaves the chip half empty at its end (112
// decode requests beside 16 chunks of 512 tokens: 88 us against 48 + 42 as two
// launches and the gap between them; together they move 375 MB, 4.3 TB/s).
// Three waves a SIMD, as many as its LDS allows, need 157 registers.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void gdn_chunk_operands_kernel(const GdnRecurArgs a,
                                                                 uint16_t* __restrict__ ws,
                                                                 int ws_slots) {
  __shared__ __attribute__((aligned(16))) union {
    OperandLds operands;
    GdnRecurLds tokens;
  } L;
  const int chunk_blocks = ws_slots * a.key_heads, token_blocks = a.num_seqs * a.value_heads;
  const int both = 2 * min(chunk_blocks, token_blocks), b = blockIdx.x;
  const int i = b < both ? b / 2 : b - both / 2;
  if (b < both ? (b & 1) == 0 : chunk_blocks > token_blocks)
    chunk_operands(a, ws, ws_slots, i / a.key_heads, i % a.key_heads, L.operands);
  else
    gdn_recurrence_block(a, i, L.tokens);
}

// ---------------------------------------------------------------------------
// The walk over a sequence's chunks. A workgroup takes SW slices of 16 NL
// value columns of one (sequence, value head), lane (n, g) of a slice the
// columns NL n .. NL n + NL - 1, with SW + 2 waves:
//  * state wave i carries slice i of S: K S, the solve, the state update;
//  * wave SW follows one chunk behind with every slice's O, taking S and U as
//    bf16 operands from a double-buffered LDS slot;
//  * the last wave moves the state waves' operands (fragments, gates and V
//    rows) into LDS with global_load_lds, BUF - 1 chunks ahead.
// One barrier per chunk. A state wave is bound by its own instruction stream
// (it has a SIMD's issue port nearly to itself and every chunk depends on the
// last one), so it computes no address and waits for no load from memory.
// ---------------------------------------------------------------------------
template <int NL, int SW, int BUF>
struct ScanLds {
  static constexpr int kCols = 16 * NL * SW;
  struct {
    uint16_t key[16 * kFrag];              // K
    uint16_t val[13 * kFrag];              // T, gates
    uint16_t v[kC * kCols];                // rows of V
  } op[BUF];
  uint16_t s[2][SW][4 * NL][kFrag];
  uint16_t u[2][SW][2 * NL][kFrag];
};

__device__ __forceinline__ bf16x8 pack_tiles(const f32x4& a, const f32x4& b) {
  const u32x4 v = {pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]),
                   pack_bf16x2(b[2], b[3])};
  return __builtin_bit_cast(bf16x8, v);
}

// What pack_tiles rounded away, rounded in turn.
__device__ __forceinline__ bf16x8 pack_rest(const f32x4& a, const f32x4& b, const bf16x8& hi) {
  const u32x4 h = __builtin_bit_cast(u32x4, hi);
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4& x = i < 2 ? a : b;
    v[i] = pack_bf16x2(x[2 * (i & 1)] - bf16_lo(h[i]), x[2 * (i & 1) + 1] - bf16_hi(h[i]));
  }
  return __builtin_bit_cast(bf16x8, v);
}

__device__ __forceinline__ bf16x8 frag(const uint16_t* p, int lane) {
  return __builtin_bit_cast(bf16x8, load_u32x4(p + 8 * lane));
}

// K^T operand (dims 16 rt + m, token slice ks) from K's fragments. A transposing
// read takes 8 bytes from each of 16 lanes (lane l: dims 4 (l % 4) .. + 3 of
// token l / 4 of the four) and gives lane m dim m of the four tokens.
__device__ __forceinline__ bf16x8 read_kt(const uint16_t* key, int rt, int ks, int ktl) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  u32x2 half[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    half[i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_s16x4*)(key + (4 * (2 * ks + i) + (rt >> 1)) * kFrag + 4 * (rt & 1) + ktl)));
  const u32x4 v = {half[0][0], half[0][1], half[1][0], half[1][1]};
  return __builtin_bit_cast(bf16x8, v);
}

__device__ __forceinline__ void dma16(const void* src, void* dst) {  // 16 bytes a lane, dst wave-uniform
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// s_waitcnt immediate for the vector-memory counter alone (gfx9 encoding).
constexpr int vmcnt_only(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }

// Barrier of the loading wave: its loads into LDS are done but for the last N.
// (A fence before the barrier would wait for those too.)
template <int N>
__device__ __forceinline__ void loads_in_flight_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(vmcnt_only(N));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

template <int NL>
struct Columns;  // NL consecutive bf16 of a row
template <>
struct Columns<1> {
  typedef uint16_t bf;
  static __device__ __forceinline__ float get(bf x, int) { return __builtin_bit_cast(float, (uint32_t)x << 16); }
  static __device__ __forceinline__ bf pack(const float* f) { return to_bf16(f[0]); }
};
template <>
struct Columns<2> {
  typedef uint32_t bf;
  static __device__ __forceinline__ float get(bf x, int e) { return e ? bf16_hi(x) : bf16_lo(x); }
  static __device__ __forceinline__ bf pack(const float* f) { return pack_bf16x2(f[0], f[1]); }
};

template <int NL, int SW, int BUF>
__global__ __launch_bounds__(64 * (SW + 2)) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn_scan_kernel(const GdnRecurArgs a,
                                                                      const uint16_t* __restrict__ ws,
                                                                      int ws_slots) {
  typedef Columns<NL> Cols;
  typedef ScanLds<NL, SW, BUF> Lds;
  // Dynamic LDS: a static array of this size tells the compiler that one
  // wave fits a SIMD, and it then keeps accumulators in AGPRs, a move away from every use.
  extern __shared__ __attribute__((aligned(16))) unsigned char scan_lds[];
  Lds& L = *reinterpret_cast<Lds*>(scan_lds);
  constexpr int kCols = Lds::kCols;
  // Slices of one (sequence, head) are a multiple of the pair count apart, so
  // they share an XCD (and its L2) whenever that count is a multiple of 8.
  const int pairs = a.num_seqs * a.value_heads;
  const int pair = blockIdx.x % pairs, part = blockIdx.x / pairs;
  const int h = pair % a.value_heads;
  const int seq = a.num_seqs - 1 - pair / a.value_heads;
  int start, len;
  if (!chunked_sequence(a, seq, &start, &len)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int chunks = (len + kC - 1) / kC;
  const int64_t slot0 = gdn_first_slot(start, seq, gdn_mostly_short(a.tokens, a.num_seqs));
  const int hk = h / (a.value_heads / a.key_heads);
  const int64_t key_stride = (int64_t)a.key_heads * kKeyElems;
  const int64_t val_stride = (int64_t)a.value_heads * kValElems;
  const uint16_t* key = ws + slot0 * key_stride + (int64_t)hk * kKeyElems;
  const uint16_t* val = ws + (int64_t)ws_slots * key_stride + slot0 * val_stride + (int64_t)h * kValElems;

  if (wave < SW) {
    const int slice = wave;
    const int lcol = 16 * NL * slice + NL * n;  // this lane's first column of the workgroup's
    const int col = kCols * part + lcol;
    const int kl = 8 * key_lane(n, g), ktl = 8 * key_lane(4 * g + (n >> 2), n & 3);
    const int64_t state_slot = a.slots[seq];
    const bool slot_ok = state_slot >= 0 && state_slot < a.num_slots;
    float* state = a.state + ((slot_ok ? state_slot : 0) * a.value_heads + h) * (int64_t)(kDim * kDim) + col;
    f32x4 S[8][NL];
    if (slot_ok) {
#pragma unroll
      for (int rt = 0; rt < 8; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < NL; ++e) S[rt][e][i] = state[(16 * rt + 4 * g + i) * kDim + e];
    } else {
#pragma unroll
      for (int rt = 0; rt < 8; ++rt)
#pragma unroll
        for (int e = 0; e < NL; ++e) S[rt][e] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    int buf = 0;
    lds_barrier();
    for (int c = 0; c < chunks; ++c) {
      const auto& op = L.op[buf];
      const float* gates = reinterpret_cast<const float*>(op.val + kGateFrag * kFrag);
      // The LDS reads of a product are issued a step ahead of it, in the order
      // of use (the sched_barriers pin the steps).
      bf16x8 K[4][4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
          K[ct][ks] = __builtin_bit_cast(bf16x8, load_u32x4(op.key + (4 * ct + ks) * kFrag + kl));
      __builtin_amdgcn_sched_barrier(0);
      // K S, S as the B operand in bf16.
      bf16x8 sb[4][NL];
      f32x4 R[4][NL];
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int e = 0; e < NL; ++e) R[ct][e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
        for (int e = 0; e < NL; ++e) {
          sb[ks][e] = pack_tiles(S[2 * ks][e], S[2 * ks + 1][e]);
          *reinterpret_cast<u32x4*>(&L.s[c & 1][slice][ks * NL + e][8 * lane]) = __builtin_bit_cast(u32x4, sb[ks][e]);
        }
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
#pragma unroll
          for (int e = 0; e < NL; ++e)
            R[ct][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(K[ct][ks], sb[ks][e], R[ct][e], 0, 0, 0);
      }
      f32x4 gam[4];
      typename Cols::bf v[4][4];
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        gam[ct] = *reinterpret_cast<const f32x4*>(gates + 16 * ct + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          v[ct][i] = *reinterpret_cast<const typename Cols::bf*>(op.v + (16 * ct + 4 * g + i) * kCols + lcol);
      }
      __builtin_amdgcn_sched_barrier(0);
      bf16x8 Th[6], Tl[6];
#pragma unroll
      for (int f = 0; f < 6; ++f) {
        Tl[f] = frag(op.val + (6 + f) * kFrag, lane);
        Th[f] = frag(op.val + f * kFrag, lane);
      }
      const float gc = gates[kC - 1];
      __builtin_amdgcn_sched_barrier(0);
      // R = V - gamma K S, as two bf16 halves.
      bf16x8 rh[2][NL], rl[2][NL];
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < NL; ++e) R[ct][e][i] = Cols::get(v[ct][i], e) - gam[ct][i] * R[ct][e][i];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int e = 0; e < NL; ++e) {
          rh[ks][e] = pack_tiles(R[2 * ks][e], R[2 * ks + 1][e]);
          rl[ks][e] = pack_rest(R[2 * ks][e], R[2 * ks + 1][e], rh[ks][e]);
        }
      f32x4 dec[4];
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) dec[ct] = *reinterpret_cast<const f32x4*>(gates + kC + 16 * ct + 4 * g);
      bf16x8 KT[8];
#pragma unroll
      for (int rt = 0; rt < 8; ++rt) KT[rt] = read_kt(op.key, rt, 0, ktl);
      __builtin_amdgcn_sched_barrier(0);
      // U = T R to 16 significant bits: the product of the lower halves is below them.
      f32x4 U[4][NL];
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int e = 0; e < NL; ++e) U[ct][e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
          for (int ct = 2 * ks; ct < 4; ++ct)
#pragma unroll
            for (int e = 0; e < NL; ++e)
              U[ct][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  p == 0 ? Tl[tri(ct, ks)] : Th[tri(ct, ks)], p == 1 ? rl[ks][e] : rh[ks][e], U[ct][e], 0, 0, 0);
#pragma unroll
      for (int rt = 0; rt < 8; ++rt)
#pragma unroll
        for (int e = 0; e < NL; ++e) S[rt][e] = S[rt][e] * gc;
      __builtin_amdgcn_sched_barrier(0);
      // S <- gamma_C S + K^T (e^{G_C - G} U).
      bf16x8 KT1[8];
#pragma unroll
      for (int rt = 0; rt < 8; ++rt) KT1[rt] = read_kt(op.key, rt, 1, ktl);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int e = 0; e < NL; ++e) {
          const bf16x8 us = pack_tiles(U[2 * ks][e] * dec[2 * ks], U[2 * ks + 1][e] * dec[2 * ks + 1]);
          *reinterpret_cast<u32x4*>(&L.u[c & 1][slice][ks * NL + e][8 * lane]) =
              __builtin_bit_cast(u32x4, pack_tiles(U[2 * ks][e], U[2 * ks + 1][e]));
#pragma unroll
          for (int rt = 0; rt < 8; ++rt)
            S[rt][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ks ? KT1[rt] : KT[rt], us, S[rt][e], 0, 0, 0);
        }
      buf = buf + 1 == BUF ? 0 : buf + 1;
      lds_barrier();
    }
    if (slot_ok) {
#pragma unroll
      for (int rt = 0; rt < 8; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < NL; ++e) state[(16 * rt + 4 * g + i) * kDim + e] = S[rt][e][i];
    }
  } else if (wave == SW) {
    bf16x8 Q[4][4], P[6];
    f32x4 gam[4];
    auto load_q = [&](int c) {
      const uint16_t* p = key + c * key_stride + kQFrag * kFrag;
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) Q[ct][ks] = frag(p + (4 * ct + ks) * kFrag, lane);
    };
    auto load_p = [&](int c) {
      const uint16_t* p = val + c * val_stride;
      const float* gates = reinterpret_cast<const float*>(p + kGateFrag * kFrag);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) gam[ct] = *reinterpret_cast<const f32x4*>(gates + 16 * ct + 4 * g);
#pragma unroll
      for (int f = 0; f < 6; ++f) P[f] = frag(p + (kPFrag + f) * kFrag, lane);
    };
    load_q(0);
    load_p(0);
    lds_barrier();
    int c = 0;
    do {
      const int next = min(c + 1, chunks - 1);
      lds_barrier();
      f32x4 O[SW][4][NL];
#pragma unroll
      for (int sl = 0; sl < SW; ++sl)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
#pragma unroll
          for (int e = 0; e < NL; ++e) O[sl][ct][e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int sl = 0; sl < SW; ++sl)
#pragma unroll
          for (int e = 0; e < NL; ++e) {
            const bf16x8 b = frag(&L.s[c & 1][sl][ks * NL + e][0], lane);
#pragma unroll
            for (int ct = 0; ct < 4; ++ct)
              O[sl][ct][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Q[ct][ks], b, O[sl][ct][e], 0, 0, 0);
          }
      __builtin_amdgcn_sched_barrier(0);
      load_q(next);
#pragma unroll
      for (int sl = 0; sl < SW; ++sl)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
#pragma unroll
          for (int e = 0; e < NL; ++e) O[sl][ct][e] = O[sl][ct][e] * gam[ct];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int sl = 0; sl < SW; ++sl)
#pragma unroll
          for (int e = 0; e < NL; ++e) {
            const bf16x8 b = frag(&L.u[c & 1][sl][ks * NL + e][0], lane);
#pragma unroll
            for (int ct = 2 * ks; ct < 4; ++ct)
              O[sl][ct][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(P[tri(ct, ks)], b, O[sl][ct][e], 0, 0, 0);
          }
      __builtin_amdgcn_sched_barrier(0);
      load_p(next);
      uint16_t* o = a.o + ((int64_t)(start + c * kC + 4 * g) * a.value_heads + h) * kDim + kCols * part + NL * n;
      auto store = [&](bool whole_chunk) {
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            uint16_t* row = o + (16 * ct + i) * (int64_t)a.value_heads * kDim;
            if (whole_chunk || c * kC + 16 * ct + 4 * g + i < len) {
#pragma unroll
              for (int sl = 0; sl < SW; ++sl) {
                float f[NL];
#pragma unroll
                for (int e = 0; e < NL; ++e) f[e] = O[sl][ct][e][i];
                *reinterpret_cast<typename Cols::bf*>(row + 16 * NL * sl) = Cols::pack(f);
              }
            }
          }
      };
      if (c * kC + kC <= len) store(true);
      else store(false);
    } while (++c < chunks);
  } else {
    constexpr int kRowLanes = kCols / 8;               // lanes per V row, 16 bytes each
    constexpr int kRows = 64 / kRowLanes;              // V rows per instruction
    constexpr int kLoads = 16 + 13 + kC / kRows;       // instructions per chunk
    static_assert(kLoads <= 63, "the counter holds one chunk's loads");
    constexpr int kAhead = BUF > 2 ? kLoads : 0;       // in flight across a barrier
    const uint16_t* v = a.v + ((int64_t)start * a.value_heads + h) * kDim + kCols * part + 8 * (lane % kRowLanes);
    auto load = [&](int c, int to) {
      c = min(c, chunks - 1);  // past the end: the last chunk again, into a buffer that nothing reads
      auto& op = L.op[to];
      const uint16_t* kp = key + c * key_stride + 8 * lane;
      const uint16_t* vp = val + c * val_stride + 8 * lane;
#pragma unroll
      for (int f = 0; f < 16; ++f) dma16(kp + f * kFrag, op.key + f * kFrag);
#pragma unroll
      for (int f = 0; f < 13; ++f) dma16(vp + f * kFrag, op.val + f * kFrag);
#pragma unroll
      for (int i = 0; i < kC / kRows; ++i) {  // rows past the end: the last token, whose T column is 0
        const int row = min(c * kC + i * kRows + lane / kRowLanes, len - 1);
        dma16(v + row * (int64_t)a.value_heads * kDim, op.v + i * kFrag);
      }
    };
#pragma unroll
    for (int i = 0; i < BUF - 1; ++i) load(i, i);
    loads_in_flight_barrier<kAhead>();
    int to = BUF - 1;
    for (int c = 0; c < chunks; ++c) {
      load(c + BUF - 1, to);
      to = to + 1 == BUF ? 0 : to + 1;
      loads_in_flight_barrier<kAhead>();
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));  // no load into LDS outlives the wave
  }
}

template <int NL, int SW, int BUF>
void launch_scan(const GdnRecurArgs& a, const uint16_t* ws, int slots, hipStream_t stream) {
  const unsigned parts = kDim / ScanLds<NL, SW, BUF>::kCols;
  hipLaunchKernelGGL((gdn_scan_kernel<NL, SW, BUF>), dim3((unsigned)(a.num_seqs * a.value_heads) * parts),
                     dim3(64 * (SW + 2)), sizeof(ScanLds<NL, SW, BUF>), stream, a, ws, slots);
}

}  // namespace

size_t gdn_scan_workspace_bytes(int tokens, int num_seqs, int key_heads, int value_heads) {
  return (size_t)gdn_slots(tokens, num_seqs) * 2 *
         ((size_t)key_heads * kKeyElems + (size_t)value_heads * kValElems);
}

int gdn_scan_launch(const GdnRecurArgs& a, int max_seq_tokens, void* workspace, hipStream_t stream) {
  const int slots = (int)gdn_slots(a.tokens, a.num_seqs);
  uint16_t* ws = static_cast<uint16_t*>(workspace);
  hipLaunchKernelGGL(gdn_chunk_operands_kernel, 
                     dim3((unsigned)(slots * a.key_heads + a.num_seqs * a.value_heads)), dim3(256), 0, stream, a, ws, slots);
  const int st = check_launch("qsa_gdn_recurrence (chunk operands)");
  if (st != QSA_OK) return st;
  switch (gdn_scan_columns(a.tokens, a.num_seqs, a.value_heads, max_seq_tokens)) {
    case 16: launch_scan<1, 1, 3>(a, ws, slots, stream); break;
    case 32: launch_scan<1, 2, 2>(a, ws, slots, stream); break;
    default: launch_scan<2, 2, 2>(a, ws, slots, stream); break;
  }
  return check_launch("qsa_gdn_recurrence (scan)");
}

}  // namespace qsa
