// Rules that choose a decode plan from a call's sizes alone: host code with no HIP
// in it, so that a host test can sweep them.
#pragma once
#include "velokv.h"

#include <algorithm>
#include <array>
#include <cstdint>

namespace velokv {

constexpr int kBS = 16;   // tokens per tile, the kernels' block
constexpr int kMaxPartTokens = 4096;  // 256 blocks: four block-id windows of one wave
constexpr int kWgMaxWaves = 8;  // waves per workgroup of vk_decode_wg_* / vk_decode_pk_* at most (velokv_kernels.hip)

// Stream-K cost units charged to each segment ahead of its blocks, for what a
// worker spends starting a second piece (per-wave traces on config 3: ~5 us).
// Measured on configs 2 and 3 with 0, 4, 8, 12, 16, 24: 8 was fastest (config 3
// 110.7 -> 109.2 us per call, config 2 208 -> 206 us).
constexpr int kSkPenalty = 8;

inline int kv_esz(int kv) {
  switch (kv) {
    case VK_KV_F32: return 4;
    case VK_KV_F16: return 2;
    case VK_KV_I8_REF:
    case VK_KV_I8_BLK: return 1;
    default: return 0;
  }
}

// Small batches under VK_SCHED_AUTO take the workgroup split in one or a few
// partitions per sequence (small_plan) while their (sequence, KV head) pairs
// have at most this many blocks in all: ragged batches; uniform ones; uniform
// ones over fp16 pools or of at most kFewPairs pairs, where the alternative is
// split-K of one-wave units.
constexpr int64_t kSmallRagged = 16384;
constexpr int64_t kSmallUniform = 12288;
constexpr int64_t kSmallUniformWide = 65536;
constexpr int64_t kFewPairs = 64;
// K and V bytes of the least partition worth a workgroup, and of what a
// partition must take off the longest context's workgroup to pay for the merge
// launch it brings (3.4 us; a workgroup alone on its CU streams 43 KB per us).
constexpr int64_t kMinPartBytes = 65536;
constexpr int64_t kMergeBytes = 147456;
// Workgroups of a call in partitions at most: bounds the scratch (17 MB at 16
// query heads per KV head) and the workgroups past short contexts.
constexpr int64_t kMaxPartWgs = 2048;
// A ragged batch stays with stream-K when its longest context keeps one wave busy
// for longer than the small plan saves: bytes per us of a wave among eight of a
// workgroup, and among fewer; the merge launch of partitions; what stream-K costs
// beside its blocks, and for each partial that it leaves of the longest context
// (its merge reads them in turn). In ns. Fitted to 319 ragged batches of four KV types,
// skewed ones (16 to 200 sequences, one of 500 to 16,000 tokens and the others of 60 to
// 500) and evenly spread ones: 64 x 8 heads of 200 int8-block tokens, one of 1,000 15.4
// us against stream-K's 19.1, one of 2,000 22.1 against 20.2, one of 16,000 122 against
// 33.6; fp16 one of 500 16.3 against 19.8, one of 1,000 22.4 against 20.2.
constexpr int64_t kWaveRate8 = 5400, kWaveRate = 9000;
constexpr int64_t kMergeNs = 3400;
constexpr int64_t kTurnNs = 6000;  // each further turn of workgroups on a CU
constexpr int64_t kSkFixedNs = 9000, kSkPartialNs = 80;

// A uniform batch keeps the plan for uniform batches when its longest wave, of at
// least kLongWave bytes, streams past the even share for longer than that plan's
// merge of more and shorter pieces takes (the workgroups of 144 x 8-wave calls leave
// 112 of 256 CUs empty): 5 us, 18 us where it is the vector kernel with 4 or 8 query
// heads per KV head. 160 pairs of 4,861 fp16 tokens, 7 query heads per KV head, 78.3 us
// against 70.7; 170 of 1,114 24.6 against 25.8.
constexpr int64_t kLongWave = 60000;
constexpr int64_t kSplitNs = 5000, kVectorNs = 18000;

// Waves of a workgroup-split kernel on the device at once in workgroups of 1, 2, 4, 8.
using WgResident = std::array<int64_t, 4>;

inline bool uniform_batch(const vk_decode_args* a) {
  return a->sum_context_len > 0 &&
         (double)a->sum_context_len >= 0.97 * (double)a->n_seqs * (double)a->max_context_len;
}

// Workgroup split of a small batch (VK_SCHED_AUTO): *waves waves per (sequence,
// partition of *part_blocks blocks, KV head); false when the batch is too large
// for it, or a wave's share of its longest context is. tile: K bytes of one
// block and KV head. The lengths' sum only steers the choice: any lengths up to
// max_context_len are computed whatever it says.
inline bool small_plan(const vk_decode_args* a, const vk_pool_desc& d, const WgResident& resident, int64_t tile, int* waves,
                       int64_t* part_blocks) {
  const int64_t nb = ((int64_t)a->max_context_len + kBS - 1) / kBS;
  const int64_t pairs = (int64_t)a->n_seqs * d.n_kv_heads;
  const int64_t waves_total = resident[3];  // of kWgMaxWaves
  if (pairs <= 0 || nb <= 0 || pairs > waves_total) return false;
  // lengths the host does not know (any up to max_context_len) stay with stream-K,
  // which balances whatever they are
  if (a->sum_context_len <= 0 && a->n_seqs > 1) return false;
  // blocks of one KV head over all sequences (at most, when the lengths are not known)
  const int64_t most = (int64_t)a->n_seqs * nb;
  const int64_t sum = a->sum_context_len > 0 ? std::min(most, a->sum_context_len / kBS + a->n_seqs) : most;
  int64_t limit = kSmallRagged;
  if (uniform_batch(a)) limit = d.kv_type == VK_KV_F16 || pairs <= kFewPairs ? kSmallUniformWide : kSmallUniform;
  if (sum * d.n_kv_heads > limit) return false;
  // uniform contexts of up to four int8 blocks (one fp32 block) take one wave of
  // split-K, whose result needs no combining (5.6 us per call at two int8 blocks;
  // fp16 split-K runs the vector kernel, 13.0 us at 16 x 32 tokens against 5.6)
  if (uniform_batch(a) && d.kv_type != VK_KV_F16 && nb * kv_esz(d.kv_type) <= 4) return false;
  // uniform fp16 ones where the plan for uniform batches is not the vector kernel with 4
  // or 8 query heads per KV head (slow: 40 x 128 tokens 25.5 us against 11.7): one wave
  // per context needs no combining up to six blocks (47 x 8 heads of 48 tokens 10.2 us
  // against 12.4), with up to two query heads per KV head where it fills the SIMDs (41 x 8
  // heads of 23-207 tokens 7.4-12.3 against 9.0-13.1), and over 128-dim tiles past one
  // workgroup of eight waves a CU at any length (34 x 8 heads of 1,469 39.2 against 52.1).
  // One sequence has the append folded in instead (18 tokens 7.1 us against 8.5).
  const int G = a->n_heads / d.n_kv_heads;
  const bool vec = d.kv_type == VK_KV_F16 && a->q_dtype == VK_DT_F16 && d.head_dim == 128 &&
                   (G == 1 || G == 2 || G == 4 || G == 8);
  const bool slow = vec && G >= 4;
  if (uniform_batch(a) && d.kv_type == VK_KV_F16 && !slow) {
    const bool over = pairs * kWgMaxWaves > waves_total, wide = tile >= kBS * 128 * 2;
    if (wide && over) return false;
    if (!over && a->n_seqs > 1 && nb <= 6 && (!vec || pairs > 128)) return false;
  }
  int nw = nb <= kWgMaxWaves ? kWgMaxWaves / 2 : kWgMaxWaves, lg = nb <= kWgMaxWaves ? 2 : 3;
  while (nw > 1 && pairs * nw > waves_total) nw /= 2, --lg;
  // each workgroup takes the LDS of kWgMaxWaves waves whatever it has (64 KB with 7
  // query heads per KV head or 64-dim tiles, two on a CU), so those of few waves may
  // take turns: 116 x 8 heads of 105 fp16 tokens, 7 query heads per KV head, 24.9 us,
  // split-K 16.0
  const int64_t turns = (pairs * nw + resident[lg] - 1) / resident[lg];
  if (turns > 1 && uniform_batch(a)) return false;
  *waves = nw;
  *part_blocks = nb;
  if (nw == kWgMaxWaves) {
    // partitions whose workgroups fit one round: at most floor(slots / S) per
    // sequence, or sum / part + S in all (a partial one per sequence)
    const int64_t slots = waves_total / kWgMaxWaves / d.n_kv_heads;
    const int64_t per = std::max<int64_t>(1, slots / a->n_seqs);
    int64_t part = (nb + per - 1) / per;
    if (slots > a->n_seqs) part = std::min(part, (sum + slots - a->n_seqs - 1) / (slots - a->n_seqs));
    part = std::max(part, std::max<int64_t>(8, kMinPartBytes / (2 * tile)));
    if ((nb - part) * 2 * tile > kMergeBytes && (nb + part - 1) / part * pairs <= kMaxPartWgs) *part_blocks = part;
  }
  // bytes of the longest wave, of a wave if all had the same, and the time between them
  const int64_t even = sum * d.n_kv_heads * 2 * tile / waves_total;
  const int64_t wave = (*part_blocks + nw - 1) / nw * 2 * tile;
  int64_t late = std::max<int64_t>(0, turns * wave - even) * 1000 / (nw == kWgMaxWaves ? kWaveRate8 : kWaveRate);
  if (uniform_batch(a)) {
    if (wave >= kLongWave && late > (slow ? kVectorNs : kSplitNs)) return false;
  } else if (a->n_seqs > 1) {
    late += (turns - 1) * kTurnNs + (*part_blocks < nb ? kMergeNs : 0);
    const int64_t share = std::max<int64_t>(1, (sum * d.n_kv_heads + kSkPenalty * pairs) / waves_total);
    if (late > kSkFixedNs + kSkPartialNs * (nb / share)) return false;
  }
  // a wave holds the ids of 256 blocks (four windows): the longest context the call
  // allows must fit, whatever the sum says, as every other plan sees to
  return (*part_blocks + nw - 1) / nw <= kMaxPartTokens / kBS;
}

// Partition of a tree call of few units (`pairs` a partition), in tokens: of 64, 96, 128,
// 192 and 256 that whose longest walk and merge take least. A wave walks its blocks one
// after another (kTreeBlockNs, by row tiles of 16 per unit and KV type) and the merge
// reads a row's partials eight at a time (kTreePartialNs each): one sequence, 8 nodes,
// one KV head, int8 blocks, 64 / 256 tokens: 500 tokens 9.2 / 15.4 us, 4,000 14.2 / 16.4
// (128: 13.8), 16,000 39.6 / 21.6; fp32 8,000 25.2 / 35.8. Below 256 only while the units
// are at most `simds`: past one wave per SIMD the partials cost more than the walk saves
// (192 / 256: 512 units a partition, 4,000 int8 tokens, 99.8 / 95.3; 192 units, 1,500
// fp16 tokens, 44.0 / 32.1).
constexpr int64_t kTreePartialNs = 110;
inline int64_t tree_block_ns(int kv_type, int row_tiles) {
  const bool one = row_tiles == 1;
  switch (kv_type) {
    case VK_KV_F32: return one ? 1600 : 2750;
    case VK_KV_F16: return one ? 500 : 840;
    default: return one ? 520 : 760;
  }
}
inline int tree_short_part(int64_t tokens, int64_t pairs, int64_t simds, int row_tiles, int kv_type) {
  const auto ns = [&](int part) {
    return tree_block_ns(kv_type, row_tiles) * (part / kBS) + kTreePartialNs * ((tokens + part - 1) / part);
  };
  int best = 256;
  for (int part : {64, 96, 128, 192})
    if (pairs * ((tokens + part - 1) / part) <= simds && ns(part) < ns(best)) best = part;
  return best;
}

}  // namespace velokv
