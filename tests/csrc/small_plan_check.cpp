// Sweep of the small-batch plan rule (velokv_plan.h small_plan) over batch shapes,
// length sums (true, unknown, too small) and kernels' resident waves.
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
  d.n_kv_heads = hkv;
  d.kv_type = kv;
  int waves = 0;
  int64_t part = 0;
  if (!small_plan(&a, d, resident, (int64_t)kBS * dim * kv_esz(kv), &waves, &part)) return;
  const int64_t nb = (longest + kBS - 1) / kBS;
  const bool range = waves >= 1 && waves <= kWgMaxWaves && part >= 1 && part <= nb;
  // a wave holds the ids of 256 blocks, whatever the lengths turn out to be
  if (range && (part + waves - 1) / waves <= kMaxPartTokens / kBS) return;
  if (bad++ < 10)
    printf("%d sequences x %d heads, longest %lld, sum %lld, kv %d dim %d, %lld waves: %d waves x %lld blocks\n", n_seqs, hkv,
           (long long)longest, (long long)sum, kv, dim, (long long)resident, waves, (long long)part);
}

int main() {
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
