"""The router's top-k order (csrc/topk.h, the header that the selection kernels use) compiled for the host: the lists of
a token's L lanes and the merge over them give argsort(-logits)[:, :k], ids distinct and in range, whatever the logits
are -- NaN (last, by index), infinities and signed zeros among them."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import c_oracle as co
from oracle import moe_oracle as mo

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# router_fused_kernel's selection with its lanes as a loop: the shuffles of a merge round read the round's values
HOST = r"""
#include "topk.h"
#include <stddef.h>
using namespace lsurge;
template <int KL> static void route(const float* l, int E, int L, int k, int32_t* sel) {
  TopkList<KL> list[32];
  int head[32] = {};
  for (int p = 0; p < L; ++p) {
    list[p].clear();
    for (int e = p; e < E; e += L) list[p].insert(topk_key(l[e]), e);
  }
  for (int j = 0; j < k; ++j) {
    uint32_t bk[32], nk[32];
    int bi[32], ni[32], hi[32];
    for (int p = 0; p < L; ++p) {
      list[p].get(head[p], &bk[p], &hi[p]);
      bi[p] = hi[p];
    }
    for (int o = 1; o < L; o <<= 1) {
      for (int p = 0; p < L; ++p) {
        const bool g = topk_before(bk[p ^ o], bi[p ^ o], bk[p], bi[p]);
        nk[p] = g ? bk[p ^ o] : bk[p];
        ni[p] = g ? bi[p ^ o] : bi[p];
      }
      for (int p = 0; p < L; ++p) bk[p] = nk[p], bi[p] = ni[p];
    }
    for (int p = 0; p < L; ++p) {
      if (bi[p] != bi[0]) { sel[j] = -2; return; }  // the lanes disagree
      if (hi[p] == bi[p]) ++head[p];
    }
    sel[j] = bi[0];
  }
}
extern "C" void host_route(const float* l, int64_t T, int E, int L, int k, int32_t* sel) {
  for (int64_t t = 0; t < T; ++t) {
    if (E / L < 8) route<4>(l + t * E, E, L, k, sel + t * k);
    else route<8>(l + t * E, E, L, k, sel + t * k);
  }
}
extern "C" void host_round_trip(const float* l, int64_t n, float* out) {
  for (int64_t i = 0; i < n; ++i) out[i] = topk_logit(topk_key(l[i]));
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("topk")
    (d / "host.cpp").write_text(HOST)
    so = str(d / "host.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wno-unknown-pragmas", "-I",
                    os.path.join(ROOT, "lewi-surge_amd", "csrc"), str(d / "host.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def _logits(E, seed):
    rng = np.random.default_rng(seed)
    l = rng.standard_normal((400, E)).astype(np.float32)
    l[0] = np.nan                                            # a NaN in the token's row of x
    l[1:200][rng.random((199, E)) < 0.5] = np.nan
    l[2, 1:] = np.nan                                        # fewer numbers than k
    l[200:300] = rng.integers(-1, 2, size=(100, E))          # ties
    l[250:300][l[250:300] == 0] = -0.0
    l[250:300, ::3] = 0.0
    special = np.array([np.inf, -np.inf, np.nan, -np.nan, 0.0, -0.0, 1e-45, -1e-45, 3e38, -3e38], np.float32)
    l[300:] = special[rng.integers(0, special.size, size=(100, E))]
    return l


@pytest.mark.parametrize("E,L", [(32, 2), (32, 4), (32, 8), (64, 2), (64, 4), (64, 8), (64, 16), (128, 4), (128, 8), (128, 16),
                                 (256, 8), (256, 16), (256, 32)])
def test_lists_and_merge_are_a_stable_descending_sort(E, L, host):
    l = _logits(E, E + L)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    for k in (1, 4, 6, 8):
        sel = np.empty((l.shape[0], k), np.int32)
        host.host_route(ptr(l), ctypes.c_int64(l.shape[0]), E, L, k, ptr(sel))
        want = mo.topk_lower_index(l, k)
        assert np.array_equal(co.topk(l, k), want)
        assert np.array_equal(sel, want)
    back = np.empty_like(l)
    host.host_round_trip(ptr(l), ctypes.c_int64(l.size), ptr(back))
    assert np.array_equal(back, l, equal_nan=True)  # -0 comes back as the equal +0
