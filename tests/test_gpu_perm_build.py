"""The permutation with the tile list in one launch (batches of at most 8192 routing pairs on the
LDS-tiled GEMMs), and the token counts per expert where those GEMMs begin, against the CPU oracle."""
import ctypes

import numpy as np
import pytest
import torch

from layerbatch_amd import _lib
from layerbatch_amd.synth import MoEShape, make_layer, make_x
from oracle import moe as om
from tests import gpu_checks as gc
from tests.helpers import layer_np, to_np
from tests.test_gpu_fp8 import _run_fp8
from tests.test_gpu_parity import _block, _run_and_check

pytestmark = pytest.mark.gpu


# 2 / 4 / 8 entries per thread and one entry past each, the last size of all (8192) and the chunked
# permutation after it; 2 to 1000 experts (4 to 16 per workgroup); ids outside [0, E)
@pytest.mark.parametrize("T,k,E,dt", [
    (1024, 2, 8, torch.int64), (683, 3, 20, torch.int32), (2048, 2, 48, torch.int32),
    (4097, 1, 3, torch.int64), (1024, 8, 128, torch.int64), (1639, 5, 256, torch.int32),
    (800, 10, 300, torch.int64), (1000, 8, 1000, torch.int32), (57, 2, 2, torch.int32)])
def test_experts_perm_build(gpu, T, k, E, dt):
    shape = MoEShape(256, E, k, 256 if E >= 300 else 128, 0)
    w, g = make_layer(shape, seed=T)
    x = make_x(g, T, 256)
    blk = _block(shape, {n: v.to(gpu) for n, v in w.items()}, gpu)
    rng = np.random.default_rng(T)
    idx = np.argsort(rng.random((T, E)), axis=1)[:, :k].astype(np.int64)
    idx[3, 0], idx[T - 1, k - 1] = E, -1                   # dropped pairs
    tw = (torch.rand((T, k), generator=g) + 0.1).to(torch.bfloat16)
    d_idx, d_tw, xd = torch.from_numpy(idx).to(gpu, dt), tw.to(gpu), x.to(gpu)
    L = _lib.LbmoeLayer()
    blk.experts.fill_layer(L)
    L.top_k = k
    y = torch.empty_like(xd)
    ws = torch.empty(_lib.workspace_size(L, T), dtype=torch.uint8, device=gpu)
    _lib.check(_lib.lib().lbmoe_experts(
        ctypes.byref(L), _lib.ptr(xd), _lib.ptr(d_idx), d_idx.element_size(), _lib.ptr(d_tw), T,
        _lib.ptr(y), _lib.ptr(ws), ws.numel(), _lib.stream_of(gpu)), "lbmoe_experts")
    torch.cuda.synchronize()

    def region(name, n):
        off, _ = _lib.workspace_region(L, T, name)
        return ws[off:off + 4 * n].view(torch.int32).cpu().numpy()

    # the oracle's order of the kept pairs: expert, then slot, then token
    key = [(idx[t, s], s, t) for s in range(k) for t in range(T) if 0 <= idx[t, s] < E]
    key.sort(key=lambda v: v[0])                            # stable: (slot, token) within an expert
    n = len(key)
    np.testing.assert_array_equal(region("counts", E), np.bincount([v[0] for v in key], minlength=E))
    np.testing.assert_array_equal(region("perm_slot", n), [v[1] for v in key])
    np.testing.assert_array_equal(region("perm_tok", n), [v[2] for v in key])
    inv = np.full((T, k), -1)
    for r, (_, s, t) in enumerate(key):
        inv[t, s] = r
    np.testing.assert_array_equal(region("inv", T * k).reshape(T, k), inv)
    ok = (idx >= 0) & (idx < E)
    wn = layer_np(w)
    rows = rng.choice(T, 24, replace=False) if T > 24 else np.arange(T)
    ref = om.experts(to_np(x)[rows], np.where(ok, idx, 0)[rows], np.where(ok, to_np(tw), 0.0)[rows],
                     wn["gate_up"], wn["down"])
    gc.check_output(to_np(y)[rows], ref, gc.TOL_BF16)


# (shape, T, fp8): T is the first batch on the LDS-tiled GEMMs (test_dispatch_rules checks that): whole
# and partly filled rounds of the CUs, less than one, the shared expert's items past a whole round
SWITCH = [(MoEShape(256, 512, 2, 512, 128), 2048, False), (MoEShape(256, 256, 4, 256, 0), 640, False),
          (MoEShape(256, 96, 2, 512, 128), 860, False), (MoEShape(1024, 128, 4, 512, 512), 434, False),
          (MoEShape(256, 128, 4, 256, 0), 320, True), (MoEShape(512, 64, 4, 512, 256), 160, True),
          (MoEShape(1024, 48, 4, 768, 0), 120, True), (MoEShape(768, 100, 3, 512, 256), 334, True)]


@pytest.mark.parametrize("shape,T", [
    (MoEShape(256, 256, 4, 256, 0), 831), (MoEShape(256, 256, 4, 256, 0), 832),
    (MoEShape(256, 96, 2, 512, 128), 815), (MoEShape(256, 96, 2, 512, 128), 816)]
    + [(s, t - d) for s, t, fp8 in SWITCH if not fp8 for d in (1, 0)])
def test_block_at_the_switch(gpu, shape, T):
    _run_and_check(shape, T, gpu, seed=T, sample=48)


@pytest.mark.parametrize("shape,T", [(s, t - d) for s, t, fp8 in SWITCH if fp8 for d in (1, 0)])
def test_fp8_block_at_the_switch(gpu, shape, T):
    _run_fp8(shape, T, gpu, seed=T, sample=48)


def _at(t, off):
    """t's values in a tensor that starts off bytes past a 16-byte boundary."""
    n = t.numel() * t.element_size()
    v = torch.empty(n + 32, dtype=torch.uint8, device=t.device)[off:off + n].view(t.dtype).view(t.shape)
    v.copy_(t)
    assert v.data_ptr() % 16 == off
    return v


def test_unaligned_rows_at_the_switch(gpu):
    """Token rows between 16-byte boundaries: the same result."""
    shape, T = MoEShape(256, 256, 4, 256, 0), 1024
    w, g = make_layer(shape, seed=4)
    blk = _block(shape, {n: v.to(gpu) for n, v in w.items()}, gpu)
    xd = make_x(g, T, 256).to(gpu)
    view = torch.empty(T * 256 + 1, dtype=torch.bfloat16, device=gpu)[1:].view(T, 256)
    view.copy_(xd)
    a, b = to_np(blk(xd)).astype("float64"), to_np(blk(view)).astype("float64")
    # a router logit summed in another order may move a token to another expert: all but a few rows
    close = np.abs(a - b).max(axis=1) <= gc.TOL_BF16 * np.abs(a).max()
    assert close.mean() >= 0.99


# T = 1100: 17 tokens per expert, where weights between 16-byte boundaries stay on the streaming
# kernels; 3000: 47, copies from any address. Wide, narrow and tiny tiles. The same indices on both sides, so
# that one kernel's results do not depend on the addresses by a bit
@pytest.mark.parametrize("T", [1100, 3000])
@pytest.mark.parametrize("what,fp8", [("x", False), ("workspace", False), ("weights", False),
                                      ("packed", False), ("x", True), ("workspace", True),
                                      ("weights", True)])
def test_operands_between_boundaries(gpu, T, what, fp8):
    shape, k = MoEShape(512, 256, 4, 256, 256), 4
    w, g = make_layer(shape, seed=6)
    x = make_x(g, T, 512).to(gpu)
    blk = _block(shape, {n: v.to(gpu) for n, v in w.items()}, gpu)
    if fp8:
        blk.quantize_fp8_()
    elif what == "packed":
        blk.pack_tiled_()
    ex = blk.experts
    idx = 2 + torch.rand((T, 254), generator=g).argsort(dim=1)[:, :k]
    idx[:T // 2, 0], idx[T // 2:T // 2 + 100, 0] = 0, 1       # experts of T / 2 and of 100 tokens
    idx = idx.to(gpu, torch.int32).contiguous()
    tw = torch.rand((T, k), generator=g).to(gpu, torch.bfloat16)

    def run(off):
        L = _lib.LbmoeLayer()
        ex.fill_layer(L)
        L.top_k = k
        n = _lib.workspace_size(L, T)
        ws = torch.empty(n + 32, dtype=torch.uint8, device=gpu)[(off if what == "workspace" else 0):][:n]
        y = torch.empty_like(x)
        xv = _at(x, off) if what == "x" else x
        _lib.check(_lib.lib().lbmoe_experts(
            ctypes.byref(L), _lib.ptr(xv), _lib.ptr(idx), 4, _lib.ptr(tw), T, _lib.ptr(y), _lib.ptr(ws),
            ws.numel(), _lib.stream_of(gpu)), "lbmoe_experts")
        torch.cuda.synchronize()
        return y

    want = run(0)
    for off in (2, 4, 8) if what in ("x", "packed") else (4, 12) if what == "workspace" else (8, 2):
        if what == "weights" and fp8:
            ex.gate_up_q, ex.down_q = _at(ex.gate_up_q, off - 1), _at(ex.down_q, off - 1)
        elif what == "weights":
            ex.gate_up_proj.data, ex.down_proj.data = _at(ex.gate_up_proj.data, off), _at(ex.down_proj.data, off)
        elif what == "packed":
            ex.gate_up_tiled, ex.down_tiled = _at(ex.gate_up_tiled, off), _at(ex.down_tiled, off)
        got = run(off)
        if T < 28 * 256 // k and what in ("weights", "packed") and not fp8:
            gc.check_output(to_np(got), to_np(want).astype("float64"), gc.TOL_BF16)   # other kernels
        else:
            assert torch.equal(got, want)
