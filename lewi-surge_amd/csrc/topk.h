// The order of the router's top-k, used by every selection kernel of router.hip (and compiled for the host by the
// tests): larger logit first, equal logits (-0 and +0 among them) by the lower expert index, NaN after -infinity.  That
// is argsort(-logits, stable), which sorts NaN last (modal/test_moe_permute.py:23-26 routes this way).
//
// It is a total order on (logit, expert), which the kernels rely on: lanes that reduce the same candidates in different
// orders must agree on one winner, or a token gets an expert twice, or none.  Float comparisons are not one (NaN), so the
// logits are compared through an integer key.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define LSURGE_HD __host__ __device__ __forceinline__
#else
#define LSURGE_HD inline
#endif

namespace lsurge {

// A place without a candidate: behind every logit, NaN included.
constexpr uint32_t TOPK_NO_KEY = 0;
constexpr int TOPK_NO_ID = 0x7fffffff;

// f32 -> key that grows with the logit (-0 as +0; -infinity is 0x007fffff, every NaN is 1)
LSURGE_HD uint32_t topk_key(float v) {
  uint32_t u = __builtin_bit_cast(uint32_t, v);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 1;
  if (u == 0x80000000u) u = 0;
  return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}
// the logit of a key (a NaN for a NaN's)
LSURGE_HD float topk_logit(uint32_t key) {
  return __builtin_bit_cast(float, key ^ ((uint32_t)((int32_t)~key >> 31) | 0x80000000u));
}
// candidate (ka, ia) comes before (kb, ib)
LSURGE_HD bool topk_before(uint32_t ka, int ia, uint32_t kb, int ib) { return ka > kb || (ka == kb && ia < ib); }

// The K best candidates, in order, of those inserted in ascending expert index: a new one moves ahead only of strictly
// smaller keys, and those it passes shift down by one.
template <int K>
struct TopkList {
  uint32_t key[K];
  int id[K];
  LSURGE_HD void clear() {
#pragma unroll
    for (int j = 0; j < K; ++j) {
      key[j] = TOPK_NO_KEY;
      id[j] = TOPK_NO_ID;
    }
  }
  LSURGE_HD void insert(uint32_t ck, int ci) {
    bool placed = false;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const bool g = placed || ck > key[j];
      const uint32_t ok = key[j];
      const int oi = id[j];
      key[j] = g ? ck : ok;
      id[j] = g ? ci : oi;
      ck = g ? ok : ck;
      ci = g ? oi : ci;
      placed = g;
    }
  }
  // candidate j, or none past the list's end
  LSURGE_HD void get(int j, uint32_t* k, int* i) const {
    *k = TOPK_NO_KEY;
    *i = TOPK_NO_ID;
#pragma unroll
    for (int q = 0; q < K; ++q)
      if (q == j) {
        *k = key[q];
        *i = id[q];
      }
  }
};

}  // namespace lsurge
