// Sweep of the small-batch plan rule (velokv_plan.h small_plan) over batch shapes,
// length sums (true, unknown, too small) and kernels' resident waves; its choices and
// tree_short_part's at measured calls.
#include <cstdio>
#include <cstring>

#include "velokv_plan.h"

using namespace velokv;

static int bad = 0;

static void check(int n_seqs, int hkv, int64_t longest, int64_t sum, int kv, int dim, int64_t resident) {
  vk_decode_args a;
  vk_pool_desc d;
  memset(&a, 0, sizeof a);
  memset(&d, 0, sizeof d);
  a.n_seqs = n_seqs;
  a.max_context_len = (int32_t)longest;
  a.sum_context_len = sum;
  a.n_heads = hkv * 4;
  a.q_dtype = VK_DT_F16;
  d.n_kv_heads = hkv;
  d.head_dim = dim;
  d.kv_type = kv;
  int waves = 0;
  int64_t part = 0;
  const WgResident waves_at = {resident / 4, resident / 2, resident, resident};  // as with much LDS
  if (!small_plan(&a, d, waves_at, (int64_t)kBS * dim * kv_esz(kv), &waves, &part)) return;
  const int64_t nb = (longest + kBS - 1) / kBS;
  const bool range = waves >= 1 && waves <= kWgMaxWaves && part >= 1 && part <= nb;
  // a wave holds the ids of 256 blocks, whatever the lengths turn out to be
  if (range && (part + waves - 1) / waves <= kMaxPartTokens / kBS) return;
  if (bad++ < 10)
    printf("%d sequences x %d heads, longest %lld, sum %lld, kv %d dim %d, %lld waves: %d waves x %lld blocks\n", n_seqs, hkv,
           (long long)longest, (long long)sum, kv, dim, (long long)resident, waves, (long long)part);
}

// One sequence of `longest` tokens and n - 1 of `rest`, 2,048 resident waves (one_wave of them in
// workgroups of one): whether the rule takes the batch (measured both ways: us of the small plan,
// of stream-K or, for equal lengths, of the plan for uniform batches; 0: not measured).
struct Skewed { int kv, hkv, n, longest, rest; bool small; double us, sk_us; int one_wave = 2048, G = 4, dim = 128; };
static const Skewed kSkewed[] = {
    {VK_KV_I8_BLK, 8, 64, 500, 200, true, 12.3, 18.9},   {VK_KV_I8_BLK, 8, 64, 16000, 200, false, 122.3, 33.6},
    {VK_KV_I8_BLK, 8, 128, 4000, 100, false, 67.2, 23.4}, {VK_KV_I8_BLK, 8, 16, 8000, 500, true, 17.1, 29.6},
    {VK_KV_I8_BLK, 2, 100, 16000, 200, false, 100.3, 52.5}, {VK_KV_I8_BLK, 2, 40, 4000, 200, true, 13.6, 39.0},
    {VK_KV_F16, 8, 33, 2000, 200, false, 31.8, 20.1},    {VK_KV_F16, 4, 64, 4000, 200, false, 53.7, 24.0},
    {VK_KV_F16, 8, 24, 500, 300, true, 10.5, 16.0},      {VK_KV_F16, 2, 100, 8000, 200, true, 21.3, 36.0},
    {VK_KV_I8_REF, 8, 40, 8000, 200, false, 67.7, 30.4}, {VK_KV_I8_REF, 8, 24, 8000, 300, true, 24.8, 31.1},
    {VK_KV_F32, 8, 24, 16000, 300, false, 84.4, 65.2},   {VK_KV_F32, 8, 16, 16000, 500, true, 54.9, 65.3},
    {VK_KV_F32, 8, 200, 2000, 60, false, 211.2, 50.0},   {VK_KV_F32, 8, 24, 500, 300, true, 24.4, 32.3},
    {VK_KV_F16, 4, 199, 335, 180, true, 12.8, 16.9},     {VK_KV_I8_BLK, 8, 182, 160, 145, false, 36.9, 26.7, 512},
    {VK_KV_I8_BLK, 8, 182, 160, 145, true, 0, 0},         {VK_KV_I8_BLK, 8, 157, 79, 79, false, 24.0, 18.7, 512},
    {VK_KV_I8_REF, 8, 141, 68, 68, false, 31.5, 24.5, 1024}, {VK_KV_I8_REF, 8, 141, 68, 68, true, 0, 0},
    {VK_KV_I8_BLK, 8, 182, 160, 145, false, 37.1, 26.7, 512, 7, 64},
    // uniform fp16: seven, one and four query heads per KV head
    {VK_KV_F16, 8, 35, 37, 37, false, 11.2, 9.5, 2048, 7},   {VK_KV_F16, 8, 4, 41, 41, false, 9.9, 9.1, 2048, 7},
    {VK_KV_F16, 8, 23, 107, 107, true, 10.8, 11.1, 2048, 7}, {VK_KV_F16, 8, 20, 4861, 4861, false, 78.3, 70.7, 2048, 7},
    {VK_KV_F16, 8, 1, 18, 18, true, 7.3, 7.9, 2048, 7},      {VK_KV_F16, 8, 34, 1469, 1469, false, 52.1, 39.2, 2048, 1},
    {VK_KV_F16, 8, 54, 23, 23, false, 9.0, 7.4, 2048, 1},    {VK_KV_F16, 8, 6, 152, 152, true, 9.6, 9.5, 2048, 1},
    {VK_KV_F16, 8, 3, 288, 288, true, 11.0, 14.1, 2048, 1},  {VK_KV_F16, 8, 40, 128, 128, true, 11.7, 25.5, 2048, 4},
    {VK_KV_F16, 8, 18, 6985, 6985, false, 107.1, 91.5, 2048, 4}, {VK_KV_F16, 8, 29, 2070, 2070, true, 42.1, 58.3, 2048, 4},
    // and of other types, a few long contexts and many short ones
    {VK_KV_F32, 8, 6, 243, 243, true, 17.8, 33.5},           {VK_KV_I8_BLK, 8, 3, 771, 771, true, 18.5, 21.1},
};

static void check_skewed(const Skewed& c) {
  vk_decode_args a;
  vk_pool_desc d;
  memset(&a, 0, sizeof a);
  memset(&d, 0, sizeof d);
  a.n_seqs = c.n;
  a.max_context_len = c.longest;
  a.sum_context_len = c.longest + (int64_t)(c.n - 1) * c.rest;
  a.n_heads = c.G * c.hkv;
  a.q_dtype = VK_DT_F16;
  d.n_kv_heads = c.hkv;
  d.head_dim = c.dim;
  d.kv_type = c.kv;
  int waves = 0;
  int64_t part = 0;
  const WgResident waves_at = {c.one_wave, 2048, 2048, 2048};
  if (small_plan(&a, d, waves_at, (int64_t)kBS * c.dim * kv_esz(c.kv), &waves, &part) == c.small) return;
  if (bad++ < 10)
    printf("skewed: kv %d, %d x %d heads, longest %d, rest %d: small %d (%.1f us, else %.1f)\n", c.kv, c.n, c.hkv,
           c.longest, c.rest, !c.small, c.us, c.sk_us);
}

// Tree calls: `pairs` units a partition of row_tiles tiles, on 1,024 SIMDs; measured us of partitions
// of 64, 96, 128, 192 and 256 tokens. The rule's choice is within 7 % of the best, and of 256 at most 2 % above.
struct Tree { int kv; int64_t tokens, pairs; int row_tiles; double us[5]; };
static const Tree kTree[] = {
    {VK_KV_I8_BLK, 508, 1, 1, {9.2, 10.3, 11.5, 13.2, 15.4}},     {VK_KV_I8_BLK, 4008, 1, 1, {14.2, 14.2, 13.8, 15.0, 16.4}},
    {VK_KV_I8_BLK, 8008, 1, 1, {22.5, 18.6, 17.0, 17.4, 18.1}},   {VK_KV_I8_BLK, 16008, 1, 1, {39.6, 28.2, 24.5, 22.4, 21.6}},
    {VK_KV_I8_BLK, 8008, 8, 2, {24.5, 20.7, 19.6, 21.4, 22.7}},   {VK_KV_I8_REF, 6009, 8, 1, {19.0, 16.1, 15.5, 15.1, 16.4}},
    {VK_KV_F16, 6013, 10, 1, {21.9, 18.1, 17.1, 17.2, 17.6}},     {VK_KV_F16, 16009, 8, 1, {42.5, 34.0, 28.3, 24.9, 21.8}},
    {VK_KV_F16, 2008, 8, 2, {13.9, 15.0, 15.6, 19.3, 21.8}},      {VK_KV_F32, 4008, 8, 2, {28.0, 30.8, 34.6, 45.0, 55.4}},
    {VK_KV_F32, 16009, 8, 1, {59.5, 52.8, 40.1, 38.2, 40.7}},
};

static void check_tree(const Tree& c) {
  static const int parts[5] = {64, 96, 128, 192, 256};
  const int got = tree_short_part(c.tokens, c.pairs, 1024, c.row_tiles, c.kv);
  double us = 1e9, best = 1e9;
  for (int i = 0; i < 5; ++i) {
    if (parts[i] == got) us = c.us[i];
    if (c.us[i] < best) best = c.us[i];
  }
  if (us <= 1.07 * best && us <= 1.02 * c.us[4]) return;
  if (bad++ < 10) printf("tree: kv %d, %lld tokens: %d, %.1f us, best %.1f\n", c.kv, (long long)c.tokens, got, us, best);
}

int main() {
  for (const Tree& c : kTree) check_tree(c);
  for (const Skewed& c : kSkewed) check_skewed(c);
  for (int64_t resident : {1024, 2048, 4096, 8192})
    for (int kv : {VK_KV_F32, VK_KV_F16, VK_KV_I8_REF, VK_KV_I8_BLK})
      for (int dim : {64, 128})
        for (int hkv : {1, 2, 3, 8, 32})
          for (int n : {1, 2, 7, 16, 32, 40, 64, 70, 100, 128, 200, 256, 1000})
            for (int64_t longest : {1, 16, 129, 1000, 4096, 4097, 5000, 10000, 20000, 32768, 32769, 48000, 100000, 1000000})
              for (int64_t rest : {1, 20, 60, 150, 200, 1000, 100000}) {
                const int64_t sum = longest + (n - 1) * (rest < longest ? rest : longest);
                for (int64_t s : {sum, (int64_t)0, (int64_t)7}) check(n, hkv, longest, s, kv, dim, resident);
              }
  printf("%s\n", bad ? "failed" : "ok");
  return bad != 0;
}
