// Host rules of the chunked gated delta rule (no HIP: the host tests compile this file alone).
#pragma once

#include <algorithm>
#include <cstdint>

namespace qsa {

constexpr int kGdnChunk = 64;     // tokens per chunk
constexpr int kGdnChunkMin = 16;  // sequences this long take a chunked kernel

// Whether a batch runs the two-launch chunked form (gdn_scan.hip) instead of
// gdn_chunk_kernel and gdn_recurrence_kernel. max_seq_tokens < 0: unknown.
//
// The one-launch kernel walks a (sequence, value head) pair's chunks in one
// workgroup, ~16 us a chunk, 256 pairs (one a CU) side by side; the two
// launches cost ~23 us and then ~1 us a chunk, with up to 128 pairs side by
// side where there are many. So they win with the length of the longest
// sequence. Times one-launch / two-launch, us, 16 value heads:
//  * up to one chunk there is nothing to walk: 16 sequences of 60 tokens 25 / 40;
//  * two chunks: two launches, unless the pairs end in the second half of the
//    one-launch kernel's first or second round (129-256, 385-512 pairs): 8 x 66
//    tokens 34 / 29, 9 x 66 35 / 39, 16 x 66 37 / 44, 16 x 128 41 / 49, 17 x 66
//    66 / 53, 24 x 96 70 / 59, 25 x 66 69 / 77, 32 x 96 75 / 82, 33 x 96 103 / 87,
//    48 x 96 109 / 107, 64 x 128 152 / 143. Single chunks beside a sequence of
//    two gain nothing: 24 x 33 and one of 66 42 / 52, 60 x 64 and one of 66 88 / 121;
//  * three chunks and more: 16 x 130 52 / 52, 16 x 256 71 / 58, 16 x 400 111 / 90,
//    one of 8192 1812 / 161;
//  * decode sequences run in the first of the two launches, but each puts empty
//    workgroups into the walk: 120 and one prompt of 100 77 / 61, 250 117 / 117,
//    500 223 / 228; of 200: 500 251 / 243, 1000 436 / 448; of 500: 1000 496 / 481.
//    32 and more of them hide what a half-empty round of two-chunk sequences
//    loses: 32 and 16 x 66 50 / 51, 112 and 16 x 66 83 / 73;
//  * unknown lengths: 100 decode requests 43 / 48, 200 x 3 tokens 91 / 95.
// Where many sequences of 16 to 64 tokens accompany a much longer one, the
// sizes known here do not tell them from decode requests beside several
// prompts: 128 x 64 and one of 512 190 / 260, but 112 decode requests and 16 x
// 512, of the same token count, 172 / 139. They are taken for the latter.
inline bool gdn_two_launches(int tokens, int num_seqs, int value_heads, int max_seq_tokens) {
  if (tokens <= kGdnChunk || num_seqs <= 0) return false;
  if (max_seq_tokens < 0) return tokens / 4 >= num_seqs;
  const int64_t longest = std::min(max_seq_tokens, tokens);
  if (longest <= kGdnChunk) return false;
  const int64_t chunks = (longest + kGdnChunk - 1) / kGdnChunk, n = num_seqs;
  const auto rounds_pay = [](int64_t pairs) {
    const int64_t halves = (pairs + 127) / 128;
    return halves != 2 && halves != 4;
  };
  const int64_t others = n > 1 ? (tokens - longest) / (n - 1) : longest;  // their mean length
  // The tokens past one per sequence, in sequences as long as the longest.
  const int64_t longs = std::min(n, std::max<int64_t>(tokens - n + longest - 2, 1) / (longest - 1));
  const int64_t pairs = n * value_heads, long_pairs = longs * value_heads;
  if (others < 32) {  // decode sequences, most likely, beside the long ones
    const int64_t short_pairs = pairs - long_pairs;
    if (short_pairs >= 5600 * chunks - 7700) return false;
    return chunks > 2 || short_pairs >= 512 || rounds_pay(long_pairs);
  }
  if (chunks > 2 || pairs <= 128) return true;
  if (others <= kGdnChunk) return long_pairs <= 128;  // single chunks, most likely
  return rounds_pay(pairs) || (long_pairs > 256 && rounds_pay(long_pairs));
}

// Workspace slots of the two-launch form, one per chunk: sequence `seq`'s chunks
// take consecutive ones from gdn_first_slot on. With floor(start / 64) + ceil(len
// / 64) - 1 <= floor((start + len) / 64), adding anything that grows by one from a
// chunked sequence to the next keeps their slots apart. The sequence's index
// does; in a batch of mostly decode sequences its minimum with start / 16 does too
// (a chunked sequence has 16 tokens) and is bounded by tokens / 16: 900 decode
// requests beside a prompt of 2000 tokens need 226 slots instead of 946. Unused
// slots cost next to nothing while there are few, and their workgroups, which
// end at once, leave room for the others': 7 and one of 1090, 32 value heads, 49 us
// with them, 52 without.
constexpr bool gdn_mostly_short(int tokens, int num_seqs) { return num_seqs > tokens / 4; }
constexpr int gdn_first_slot(int start, int seq, bool mostly_short) {
  return start / kGdnChunk + (mostly_short && start / kGdnChunkMin < seq ? start / kGdnChunkMin : seq);
}
constexpr int64_t gdn_slots(int tokens, int num_seqs) {
  return (int64_t)tokens / kGdnChunk + (gdn_mostly_short(tokens, num_seqs) ? tokens / kGdnChunkMin : num_seqs);
}

// Value columns per workgroup of the walk: the narrowest slices whose workgroups
// fit the chip's 256 CUs at once (LDS holds one workgroup a CU). A workgroup's
// time per chunk hardly depends on its width, so more of them only help while
// they run side by side. Long sequences of the batch: at least tokens /
// max_seq_tokens. Measured, both launches, 16 value heads, 8192 tokens (16 / 32 /
// 64 columns, us): one sequence 164 / 173 / 248, two 114 / 113 / 152, four
// 114 / 85 / 103, eight 128 / 95 / 84, sixteen 204 / 129 / 97.
inline int gdn_scan_columns(int tokens, int num_seqs, int value_heads, int max_seq_tokens) {
  const int64_t longest = std::min(max_seq_tokens, tokens);  // a bound may be any int
  const int64_t side = max_seq_tokens > 0 ? (tokens + longest - 1) / longest : num_seqs;
  const int64_t pairs = side * value_heads;
  return pairs * 8 <= 256 ? 16 : pairs * 4 <= 256 ? 32 : 64;
}

}  // namespace qsa
