"""The host extension against the general Python path: the plain calls it takes give the same bits,
and everything else is left to the general path (None), on the CPU and under torch's modes."""
import os
import sys
import types

import pytest
import torch

import layerbatch_amd
from layerbatch_amd import _lib, build, moe
from layerbatch_amd.synth import MoEShape, make_layer, make_x


def _block(device, cls=moe.Qwen3_5SparseMoeBlock, Is=256):
    w, _ = make_layer(MoEShape(512, 16, 4, 256, Is), seed=2)
    b = cls(512, 16, 4, 256, Is).to(device=device, dtype=torch.bfloat16)
    with torch.no_grad():
        b.gate.weight.copy_(w["gate"])
        b.experts.gate_up_proj.copy_(w["gate_up"])
        b.experts.down_proj.copy_(w["down"])
        if Is:
            b.shared_expert.gate_proj.weight.copy_(w["sh_gate"])
            b.shared_expert.up_proj.weight.copy_(w["sh_up"])
            b.shared_expert.down_proj.weight.copy_(w["sh_down"])
            b.shared_expert_gate.weight.copy_(w["sh_gate_w"])
    return b


def test_left_to_the_general_path_on_cpu(lbmoe):
    h, b = moe._host(), _block("cpu")
    x = torch.zeros((3, 512), dtype=torch.bfloat16)
    idx, tw = torch.zeros((3, 4), dtype=torch.int64), torch.zeros((3, 4), dtype=torch.bfloat16)
    assert h.block(b, x, None) is None and h.block(b, "x", None) is None
    assert h.block(None, x, None) is None and h.block(b, None, None) is None
    assert h.block_norm(b, x, x, object(), None) is None
    assert h.router(b.gate, x) is None and h.router(b, x) is None
    assert h.experts(b.experts, x, idx, tw) is None and h.mlp(b.shared_expert, x) is None
    assert h.mlp(b.shared_expert) is None                 # a wrong argument count


def test_a_default_device_is_no_mode_to_decline(lbmoe):
    """torch.set_default_device leaves a DeviceContext on the mode stack for good: it changes no call
    that names its devices, so it must not send every call to the general path."""
    h = moe._host()
    assert h.plain()
    with torch.device("cpu"):
        assert h.plain()
        with _Mode():
            assert not h.plain()
    torch.set_default_device("cpu")
    try:
        assert torch._C._len_torch_function_stack() == 1 and h.plain()
    finally:
        torch.set_default_device(None)
    with _Mode(), torch.device("meta"):
        assert not h.plain()


@pytest.mark.parametrize("ext,why", [
    (None, "_host"), (types.SimpleNamespace(torch_version="1.0"), "built against torch 1.0")])
def test_the_general_path_runs_without_the_extension(lbmoe, monkeypatch, ext, why):
    """An extension that is missing, or was built against another torch, is left out with one
    warning; the calls (refused ones here, on the CPU) reach the general path."""
    monkeypatch.setattr(_lib, "_host", None)
    if ext is None:
        monkeypatch.delattr(layerbatch_amd, "_host", raising=False)
        monkeypatch.setitem(sys.modules, "layerbatch_amd._host", None)
    else:
        monkeypatch.setattr(layerbatch_amd, "_host", ext, raising=False)
        monkeypatch.setitem(sys.modules, "layerbatch_amd._host", ext)
    b, x = _block("cpu"), torch.zeros((3, 512), dtype=torch.bfloat16)
    with pytest.warns(RuntimeWarning, match=why) as caught:
        for call in (b, b.gate, b.shared_expert, lambda v: b.forward_norm(v, v, None),
                     lambda v: b.experts(v, None, None)):
            with pytest.raises(RuntimeError, match="is on cpu"):
                call(x)
    assert len(caught) == 1
    assert _lib.host(()).block(b, x, None) is None


def test_build_without_a_host_compiler(monkeypatch, tmp_path):
    """Any C++ compiler will do, hipcc's own too; with none the library is still built and no stale
    extension stays behind."""
    stale = tmp_path / "_host.so"
    stale.write_bytes(b"")
    monkeypatch.setattr(build, "HOST", str(stale))
    monkeypatch.delenv("CXX", raising=False)
    rocm = tmp_path / "bin"
    rocm.mkdir()
    hipcc = rocm / "hipcc"
    monkeypatch.setenv("PATH", str(tmp_path / "empty"))
    assert build._host_cxx(str(hipcc)) is None
    with pytest.warns(RuntimeWarning, match="no host C\\+\\+ compiler"):
        build._build_host(str(hipcc))
    assert not stale.exists()
    clang = rocm / "amdclang++"
    clang.write_text("#!/bin/sh\n")
    os.chmod(clang, 0o755)
    assert build._host_cxx(str(hipcc)) == str(clang)


class _Norm(torch.nn.Module):
    eps = 1e-6

    def __init__(self, device):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.linspace(-0.2, 0.2, 512).to(device, torch.bfloat16))


def _calls(b, x, res, norm, idx, tw):
    """The five module calls of one block, outputs flattened."""
    out = [b(x), *b.forward_norm(x, res, norm), *b.gate(x), b.experts(x, idx, tw)]
    return out + ([b.shared_expert(x)] if b.shared_expert is not None else [])


@pytest.mark.gpu
@pytest.mark.parametrize("Is,fp8,bias,T", [(256, False, False, 1), (256, True, False, 70),
                                           (0, False, True, 5), (0, True, True, 1),
                                           (256, False, True, 600), (256, False, False, 0)])
def test_same_results_as_the_general_path(gpu, monkeypatch, Is, fp8, bias, T):
    b, h = _block(gpu, Is=Is), moe._host()
    if fp8:
        b.quantize_fp8_()
    g = torch.Generator().manual_seed(T)
    if bias:
        b.gate.logit_bias = torch.randn(16, generator=g).to(gpu)
    x, res = make_x(g, T, 512).to(gpu), make_x(g, T, 512).to(gpu)
    idx = torch.randint(0, 16, (T, 4), generator=g).to(gpu)
    tw = torch.rand((T, 4), generator=g).to(gpu, torch.bfloat16)
    norm = _Norm(gpu)
    args = (b, x, res, norm, idx, tw)
    assert h.block(b, x, None) is not None and h.block_norm(b, x, res, norm, None) is not None
    assert h.router(b.gate, x) is not None and h.experts(b.experts, x, idx, tw) is not None
    assert Is == 0 or h.mlp(b.shared_expert, x) is not None
    ws = torch.empty(b.workspace_size(T), dtype=torch.uint8, device=gpu)
    assert h.block(b, x, ws) is not None
    fast = _calls(*args)

    class _Declines:
        def __getattr__(self, name):
            return lambda *a: None

    monkeypatch.setattr(moe, "_host", lambda: _Declines())
    for a, c in zip(fast, _calls(*args)):
        assert a.dtype == c.dtype and torch.equal(a, c)


@pytest.mark.gpu
@pytest.mark.parametrize("default", ["cpu", "cuda"])
def test_taken_under_a_default_device(gpu, default):
    b, h, norm = _block(gpu), moe._host(), _Norm(gpu)
    g = torch.Generator().manual_seed(3)
    x, res = make_x(g, 3, 512).to(gpu), make_x(g, 3, 512).to(gpu)
    tw, idx = b.gate(x)
    want = _calls(b, x, res, norm, idx, tw)
    torch.set_default_device(default)
    try:
        got = [h.block(b, x, None), *h.block_norm(b, x, res, norm, None), *h.router(b.gate, x),
               h.experts(b.experts, x, idx, tw), h.mlp(b.shared_expert, x)]
    finally:
        torch.set_default_device(None)
    for a, c in zip(got, want, strict=True):
        assert a.device == gpu and torch.equal(a, c)


@pytest.mark.gpu
def test_left_to_the_general_path(gpu):
    b, h = _block(gpu), moe._host()
    x = torch.zeros((3, 512), dtype=torch.bfloat16, device=gpu)

    class Sub(moe.Qwen3_5SparseMoeBlock):
        pass

    assert h.block(_block(gpu, Sub), x, None) is None            # another class
    assert h.block(b, x[:, ::2], None) is None                   # strides, widths, types, ranks
    assert h.block(b, x.float(), None) is None and h.block(b, x[0], None) is None
    assert h.block(b, x[:, :256].contiguous(), None) is None
    assert h.block(b, x, torch.empty(4, device=gpu)) is None
    assert h.experts(b.experts, x, torch.zeros((3, 4), device=gpu), x[:, :4].contiguous()) is None
    with _Mode():
        assert h.block(b, x, None) is None
    assert torch.func.vmap(lambda v: torch.tensor(h.router(b.gate, v) is None))(x[None]).all()
    b.pack_tiled_()
    assert h.block(b, x, None) is None and h.mlp(b.shared_expert, x) is None
    y = _block(gpu)
    y.gate.register_parameter("extra", torch.nn.Parameter(torch.zeros(1)))   # on the CPU
    assert h.block(y, x, None) is None
    with pytest.raises(RuntimeError, match="device"):
        y(x)
    with pytest.raises(RuntimeError, match="workspace too small"):
        _block(gpu)(x, workspace=torch.empty(16, dtype=torch.uint8, device=gpu))


class _Mode(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))
