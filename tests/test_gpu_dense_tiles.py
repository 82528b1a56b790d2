"""The dense MLP and the router logits on their LDS-tiled kernels, at the sizes where a tile shape or
a k split begins or ends, against the CPU oracle (gpu_checks' tolerances)."""
import pytest
import torch

from layerbatch_amd.moe import Qwen3_5SharedExpertMLP, Qwen3_5SparseMoeBlock, Qwen3_5TopKRouter
from layerbatch_amd.synth import MoEShape, make_layer, make_x
from oracle import moe as om
from tests import gpu_checks as gc
from tests.helpers import bf16_bits_of, layer_np, to_np

pytestmark = pytest.mark.gpu


def _mlp(H, Is, T, gpu, seed):
    w, g = make_layer(MoEShape(H, 1, 1, 128, Is), seed=seed)
    m = Qwen3_5SharedExpertMLP(H, Is).to(device=gpu, dtype=torch.bfloat16)
    with torch.no_grad():
        m.gate_proj.weight.copy_(w["sh_gate"])
        m.up_proj.weight.copy_(w["sh_up"])
        m.down_proj.weight.copy_(w["sh_down"])
    return m, layer_np(w), make_x(g, T, H)


# 28 / 29: streaming / tiles; K = 384 and 128 (two k groups, one k-tile each at K = 128), K = 256 and
# 2048 (four); 64 x 64, 128 x 64, 128 x 128, 256 x 128 and 256 x 256 tiles of each GEMM with ragged
# last token tiles (160 workgroups of (gate_up, down) tiles at the sizes named)
@pytest.mark.parametrize("H,Is,T", [
    (384, 128, 28), (384, 128, 29), (128, 128, 65), (2048, 512, 64), (2048, 512, 129),
    (512, 256, 1283),       # 64 x 64 in two k groups, 64 x 64
    (1024, 512, 1217),      # 128 x 64 gate_up and down
    (1024, 512, 2477),      # 128 x 128
    (384, 256, 6001),       # 128 x 128 gate_up; 384 output rows: no 256-row tiles
    (256, 256, 10369),      # 256 x 128 gate_up
    (256, 256, 20993),      # 256 x 256 gate_up, 256 x 128 down
    (256, 128, 41001),      # 256 x 256 down and gate_up
])
def test_dense_mlp_tiles(gpu, H, Is, T):
    m, w, x = _mlp(H, Is, T, gpu, seed=T)
    out = m(x.to(gpu))
    gc.check_output(to_np(out), om.shared_expert(to_np(x), w["sh_gate"], w["sh_up"], w["sh_down"]),
                    gc.TOL_BF16)


@pytest.mark.parametrize("H,Is,T", [
    (512, 256, 28), (512, 256, 29), (256, 256, 65), (1024, 512, 777),     # 256 x 64
    (512, 512, 5121 + 7),                                                  # 256 x 128 gate_up
    (512, 512, 10241 + 6),                                                 # 256 x 256 gate_up
])
def test_dense_mlp_tiles_fp8(gpu, H, Is, T):
    w, g = make_layer(MoEShape(H, 2, 1, 256, Is), seed=T)
    blk = Qwen3_5SparseMoeBlock(H, 2, 1, 256, Is).to(device=gpu, dtype=torch.bfloat16)
    with torch.no_grad():
        blk.experts.gate_up_proj.zero_()
        blk.experts.down_proj.zero_()
        blk.shared_expert.gate_proj.weight.copy_(w["sh_gate"])
        blk.shared_expert.up_proj.weight.copy_(w["sh_up"])
        blk.shared_expert.down_proj.weight.copy_(w["sh_down"])
    blk.quantize_fp8_()
    se = blk.shared_expert
    x = make_x(g, T, H)
    out = se(x.to(gpu))
    qq = {n: (se.q[n][0].cpu().numpy(), se.q[n][1].cpu().numpy()) for n in ("gate", "up", "down")}
    ref = om.shared_expert_fp8(to_np(x), *qq["gate"], *qq["up"], *qq["down"])
    gc.check_output(to_np(out), ref, gc.TOL_FP8)


@pytest.mark.parametrize("T", [64, 2048])
def test_dense_mlp_unaligned_rows(gpu, T):
    """Tensors that start between 16-byte boundaries (views of a larger buffer): the same result."""
    m, _, x = _mlp(512, 256, T, gpu, seed=3)
    xd = x.to(gpu)
    buf = torch.empty(T * 512 + 1, dtype=torch.bfloat16, device=gpu)
    view = buf[1:].view(T, 512)
    view.copy_(xd)
    a, b = to_np(m(xd)).astype("float64"), to_np(m(view)).astype("float64")
    assert abs(a - b).max() <= gc.TOL_BF16 * abs(a).max()


# more than 384 blocks of 16 experts x 16 tokens and at most 256 of 64 x 64; E = 1000 rows of 8-entry
# chunks past the last whole tile, E = 66 no whole chunks, H = 384 (two k groups), 640, 2048
@pytest.mark.parametrize("T,E,H", [(193, 512, 2048), (200, 500, 384), (100, 1000, 640), (1023, 66, 512),
                                   (1500, 66, 2048), (2048, 512, 384), (4096, 256, 1024),
                                   (16384, 4, 512)])
def test_router_small_tiles(gpu, T, E, H):
    w, g = make_layer(MoEShape(H, E, 1, 128, 0), seed=T)
    r = Qwen3_5TopKRouter(E, H, min(E, 4)).to(device=gpu, dtype=torch.bfloat16)
    with torch.no_grad():
        r.weight.copy_(w["gate"])
    x = make_x(g, T, H)
    gc.check_logits(bf16_bits_of(r.logits(x.to(gpu))), to_np(x), to_np(w["gate"]))
