"""The two grouped-GEMM kernel families give bitwise identical results.

LSURGE_GEMM_CLASSIC (128 x 256 tiles over 128-row blocks; the 8-wave ping-pong kernel over 256-row tiles) and
LSURGE_GEMM_G256 (the persistent 256 x 256 x 64 kernel, the default) compute every output element with the same
ascending sequence of 16-deep MFMA steps, so every output of ragged_dot (modal/padded_gmm.py:45-69) and of the whole
MoE layer must match bit for bit.  The oracle tests check each family against the reference semantics; this file
checks the identity itself, on shapes that exercise what differs between the two: row, column and K tails (partial
tiles, zero stages past K), empty groups, gathered rows, both B layouts and every epilogue.
"""
import contextlib

import numpy as np
import pytest
import torch

import _lib
import padded_gmm as pg
from moe_layer import MoELayer, MoEShape
from oracle import moe_oracle as mo

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def variant(v):
    L = _lib.lib()
    old = L.lsurge_get_gemm_variant()
    _lib.check(L.lsurge_set_gemm_variant(v), "set_gemm_variant")
    try:
        yield
    finally:
        L.lsurge_set_gemm_variant(old)


def test_variant_switch_rejects_unknown():
    L = _lib.lib()
    assert L.lsurge_get_gemm_variant() == 1  # the persistent kernel is the default
    assert L.lsurge_set_gemm_variant(7) != 0
    assert L.lsurge_get_gemm_variant() == 1


def _ragged(gs, M, K, N, dt, out_dtype, dev, seed):
    rng = np.random.default_rng(seed)
    E = len(gs)
    a = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(dev).to(dt)
    b = torch.from_numpy(rng.standard_normal((E, K, N)).astype(np.float32)).to(dev).to(dt)
    g = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).to(dev).to(out_dtype or dt)
    gst = torch.tensor(gs, dtype=torch.int32, device=dev)
    res = {}
    for v in (0, 1):
        with variant(v):
            at = a.clone().requires_grad_(True)
            bt = b.clone().requires_grad_(True)
            out = pg.padded_ragged_dot(at, bt, gst, preferred_element_type=out_dtype)
            out.backward(g)
            torch.cuda.synchronize()
            res[v] = (out.detach().clone(), at.grad.clone(), bt.grad.clone())
    return res


@pytest.mark.parametrize("gs,M,K,N,dt,out_dtype", [
    ([5, 0, 9, 3, 7, 1, 6, 4], 38, 64, 48, torch.bfloat16, None),       # modal/te_run.py:72-79; one stage + a zero stage
    ([5, 0, 9, 3, 7, 1, 6, 4], 38, 64, 48, torch.bfloat16, torch.float32),
    ([300, 0, 517, 1, 255, 256, 257], 1700, 192, 200, torch.bfloat16, None),  # K of 3 stages, N tail inside a tile
    ([700, 0, 1300, 20, 5000], 7100, 512, 1024, torch.bfloat16, None),
    ([700, 0, 1300, 20, 5000], 7100, 512, 1024, torch.float16, None),
    ([1536] * 16, 24576, 1024, 512, torch.float16, torch.float32),
    ([1000, 3000, 0, 2000], 6001, 1024, 768, torch.bfloat16, torch.float32),
])
def test_ragged_dot_bitwise(gs, M, K, N, dt, out_dtype, dev):
    res = _ragged(gs, M, K, N, dt, out_dtype, dev, seed=M + K)
    for name, x0, x1 in zip(("out", "dlhs", "drhs"), res[0], res[1]):
        assert torch.equal(x0, x1), f"{name}: max |diff| {(x0.float() - x1.float()).abs().max().item()}"


def _layer(p, shape, dev):
    tp = {n: torch.from_numpy(np.ascontiguousarray(p[n])).to(dev).to(torch.bfloat16)
          for n in ("x", "w_r", "w_gate", "w_up", "w_down", "ws_gate", "ws_up", "ws_down") if p.get(n) is not None}
    tp["bias"] = None if p.get("bias") is None else torch.from_numpy(p["bias"]).to(dev)
    dy = torch.from_numpy(np.ascontiguousarray(p["dy"])).to(dev).to(torch.bfloat16)
    res = {}
    for v in (0, 1):
        with variant(v):
            layer = MoELayer(shape, dev)
            out = layer.forward(tp).clone()
            g = layer.backward(tp, dy)
            torch.cuda.synchronize()
            res[v] = {"out": out, **{k: t.clone() for k, t in g.items()}}
    return res


@pytest.mark.parametrize("T,d,E,k,f,fs,zipf", [
    (1000, 512, 64, 6, 256, 256, False),   # shared expert merged as expert E
    (1000, 512, 16, 4, 256, 512, False),   # shared expert on dense GEMMs of its own
    (777, 256, 8, 2, 128, 0, False),       # no shared expert, row tails
    (4096, 1024, 64, 6, 512, 512, False),  # C1's shape, forward and backward
    (4096, 1024, 128, 6, 512, 512, True),  # Zipf loads: empty experts, one hot expert
    (2048, 2048, 256, 8, 512, 2048, False),  # C5's d, E, k and shared width on a token slice
    (1500, 1024, 32, 4, 1024, 1024, False),  # gathered dY rows in the down GEMMs, merged shared expert
])
def test_layer_bitwise(T, d, E, k, f, fs, zipf, dev):
    p = mo.make_inputs(T=T, d=d, E=E, k=k, f=f, fs=fs, seed=T + E, zipf=zipf)
    res = _layer(p, MoEShape(T, d, E, k, f, fs), dev)
    for name in res[0]:
        x0, x1 = res[0][name], res[1][name]
        assert torch.equal(x0, x1), f"{name}: max |diff| {(x0.float() - x1.float()).abs().max().item()}"


@pytest.mark.parametrize("m,e,hot", [(256, 4, False), (257, 4, False), (512, 8, True), (513, 8, True), (64, 1, False)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_ragged_dot_few_rows_rule(m, e, hot, dt, dev):
    """Both sides of the few-rows rule (m = 64 e rows and one more), all rows in one group included: the bits of the
    classic kernels, forward and backward."""
    gs = [0] * e
    if hot:
        gs[-1] = m
    else:
        gs = [m // e] * e
        gs[0] += m % e
    res = _ragged(gs, m, 72, 264, dt, None, dev, seed=m)
    for x0, x1 in zip(res[0], res[1]):
        assert torch.equal(x0, x1)


@pytest.mark.parametrize("T", [512, 513])
@pytest.mark.parametrize("fs", [0, 128, 256])
@pytest.mark.parametrize("zipf", [False, True])
def test_layer_few_rows_rule(T, fs, zipf, dev):
    """Both sides of the layer's few-rows rule (T k = 128 E slots and k more), with the shared expert merged, of its own
    width and absent: the bits of the classic kernels."""
    p = mo.make_inputs(T=T, d=256, E=16, k=4, f=128, fs=fs, seed=T + fs, zipf=zipf)
    res = _layer(p, MoEShape(T, 256, 16, 4, 128, fs), dev)
    for name in res[0]:
        assert torch.equal(res[0][name], res[1][name]), name


def test_layer_few_rows_rule_full_gpu(dev):
    """Both sides of the rule's line at T k = 96 E, where the gate/up tiles take both slots of every CU: the classic bits."""
    p = mo.make_inputs(T=2049, d=1024, E=128, k=6, f=512, fs=512, seed=7)
    for T in (2048, 2049):
        q = dict(p, x=p["x"][:T], dy=p["dy"][:T])
        res = _layer(q, MoEShape(T, 1024, 128, 6, 512, 512), dev)
        for name in res[0]:
            assert torch.equal(res[0][name], res[1][name]), (T, name)


@pytest.mark.parametrize("M,K,N,E,hot,dtype", [(1000, 64, 72, 8, 0, torch.bfloat16), (3000, 512, 520, 4, 2600, torch.bfloat16),
                                               (2304, 1024, 1024, 8, 0, torch.bfloat16), (700, 136, 256, 300, 0, torch.bfloat16),
                                               (9000, 256, 264, 2, 8900, torch.float16), (640, 128, 128, 8, 0, torch.float16)])
def test_ragged_dot_bwd_16bit_drhs(M, K, N, E, hot, dtype, dev):
    """drhs in the operands' dtype is the f32 drhs rounded once, bit for bit: both kernel families, single chunks, split
    hot groups (partials summed in f32 first), the unchunked path (300 groups), column remainders, empty groups."""
    gen = torch.Generator(device=dev).manual_seed(M + N)
    lhs = torch.randn((M, K), device=dev, generator=gen).to(dtype)
    rhs = torch.randn((E, K, N), device=dev, generator=gen).to(dtype)
    g = torch.randn((M, N), device=dev, generator=gen).to(dtype)
    gs = torch.zeros(E, dtype=torch.int32)
    gs[0] = hot
    rest = M - hot - 5  # five rows past the groups
    gs[1:-1 if E > 2 else E] += rest // (E - 2 if E > 2 else 1)
    gs = gs.to(dev)
    lib = _lib.lib()
    ws = _lib.workspace(lib.lsurge_ragged_dot_bwd_workspace_bytes(M, K, N, E), dev)
    for variant in (0, 1):
        lib.lsurge_set_gemm_variant(variant)
        try:
            out = {}
            for dt in (torch.float32, dtype):
                dl = torch.empty((M, K), dtype=dtype, device=dev)
                dr = torch.full((E, K, N), float("nan"), dtype=dt, device=dev)
                _lib.check(lib.lsurge_ragged_dot_bwd_as(_lib.ptr(lhs), _lib.ptr(rhs), _lib.ptr(gs), _lib.ptr(g), M, K, N, E, _lib.dt(lhs),
                                                     _lib.ptr(dl), _lib.ptr(dr), _lib.dt(dr), _lib.ptr(ws), ws.numel(),
                                                     _lib.stream(dev)), "ragged_dot_bwd_as")
                out[dt] = dr
            assert torch.equal(out[torch.float32].to(dtype).view(torch.int16), out[dtype].view(torch.int16))
        finally:
            lib.lsurge_set_gemm_variant(1)
    rc = lib.lsurge_ragged_dot_bwd_as(_lib.ptr(lhs), _lib.ptr(rhs), _lib.ptr(gs), _lib.ptr(g), M, K, N, E, _lib.dt(lhs), _lib.ptr(dl),
                                      _lib.ptr(dr), _lib.F16 if dtype == torch.bfloat16 else _lib.BF16, _lib.ptr(ws), ws.numel(),
                                      _lib.stream(dev))
    assert rc == -2  # a 16-bit dtype other than the operands'


@pytest.mark.parametrize("T,d,E,k,f,fs", [(1000, 256, 16, 4, 128, 128), (700, 512, 32, 6, 256, 1024), (900, 1024, 8, 2, 1024, 0)])
def test_layer_backward_bf16_weight_gradients(T, d, E, k, f, fs, dev):
    """Layer weight gradients written in bf16 are the f32 ones rounded once; dx and dweights do not change."""
    p = mo.make_inputs(T=T, d=d, E=E, k=k, f=f, fs=fs, seed=3)
    tp = {n: torch.from_numpy(p[n]).to(dev).to(torch.bfloat16) for n in
          ("x", "w_r", "w_gate", "w_up", "w_down") + (("ws_gate", "ws_up", "ws_down") if fs else ())}
    dy = torch.from_numpy(p["dy"]).to(dev).to(torch.bfloat16)
    layer = MoELayer(MoEShape(T, d, E, k, f, fs), dev)
    layer.forward(tp)
    g32 = layer.backward(tp, dy)
    g16 = layer.backward(tp, dy, layer.alloc_grads(torch.bfloat16))
    for n, t in g32.items():
        same = g16[n] if n in ("dx", "dweights") else g16[n].view(torch.int16)
        want = t if n in ("dx", "dweights") else t.to(torch.bfloat16).view(torch.int16)
        assert torch.equal(same, want), n
    mixed = dict(layer.alloc_grads(), dw_down=g16["dw_down"])
    with pytest.raises(ValueError, match="one dtype"):
        layer.backward(tp, dy, mixed)
