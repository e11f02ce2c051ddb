"""The fused router's launch rule (csrc/router_tiles.h) compiled for the host: the shapes of the GPU tests that compare the
kernel with the split router reach every instantiation that the launcher can pick."""
import ctypes
import itertools
import os
import subprocess

from test_layer_gpu import FUSED_ROUTER, FUSED_ROUTER_EDGES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = r"""
#include "router_tiles.h"
extern "C" void host_tiles(int64_t t, int64_t d, int64_t e, int* out) {
  const lsurge::RouterTiles r = lsurge::router_tiles(t, d, e);
  out[0] = r.tt, out[1] = r.ht, out[2] = r.dc;
}
"""


def test_shapes_reach_every_fused_router(tmp_path):
    (tmp_path / "host.cpp").write_text(HOST)
    so = str(tmp_path / "host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "lewi-surge_amd", "csrc"),
                    str(tmp_path / "host.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)

    def tiles(t, d, e):
        out = (ctypes.c_int * 3)()
        lib.host_tiles(ctypes.c_int64(t), ctypes.c_int64(d), ctypes.c_int64(e), out)
        return (e, *out)

    # token counts over the whole range by their logarithm, and around every one at which a whole number of chunks ends
    counts = sorted({max(1, t + o) for b in range(21) for t in (1 << b, 3 << b >> 1) for o in (-64, -1, 0, 1, 64)})
    picked = {tiles(t, d, e) for t, d, e in itertools.product(counts, (64, 128), (32, 64, 128, 256))}
    assert len(picked) == 2 * (4 * 3 + 2)  # three tile counts everywhere, one expert tile at 32 and 64 experts
    assert {tiles(t, d, e) for t, d, e, _ in FUSED_ROUTER + FUSED_ROUTER_EDGES} == picked
