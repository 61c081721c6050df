// Prints how sh_knn_pool cuts searches over the whole range of its arguments; host code only,
// built by test_knn_plan_host.py.
#include "sh_knn.hip"

#include <cstdio>

int main() {
  const int64_t nqs[] = {1, 7, 100, 500, 1000, 4096, 16384, 100000, 1000000, 20000000, 2147483647};
  const int64_t nrs[] = {1,      100,     511,       2048,       8192,       12000,      25000,
                         30000,  61440,   100000,    500000,     4000000,    400000000,  536870912,
                         536870913, 1100000000, 2200000000, 4294967294};
  const int dtypes[] = {SH_BF16, SH_FP8, SH_F32}, pools[] = {1, 20, 64, 100, 128, 200, 256};
  for (int dtype : dtypes)
    for (int D : {1, 50, 64, 100, 125})
      for (int pool : pools)
        for (int64_t nq : nqs)
          for (int64_t nr : nrs) {
            if (pool > 128 && dtype != SH_FP8) continue;
            const sh::PoolPlan p = sh::pool_plan(nq, nr, sh::pack_k(dtype, D), dtype, pool);
            printf("%d %d %d %lld %lld %d %d %d %d %d %d %lld %d %d %lld %zu\n", dtype, D, pool,
                   (long long)nq, (long long)nr, (int)p.bounded, (int)p.collect, p.rank, p.S1,
                   p.per, p.slots, (long long)p.m, p.S3, p.cap, (long long)p.len3, p.bytes);
          }
  printf("slots %d\n", sh::kTauSlots);
}
