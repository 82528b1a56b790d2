"""Routing inside the decode gate_up kernel (at most 8 tokens and 64 routing pairs, while a CU runs few of
its workgroups) and the permutation
inside it for batches of at most 16 tokens with at least as many pairs as experts: every stage against
the CPU oracle at the sizes where the path changes."""
import pytest

from layerbatch_amd.synth import MoEShape
from tests.test_gpu_parity import _run_and_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,T", [
    (MoEShape(512, 128, 8, 256, 0), 8),        # 64 pairs: the last size routed in gate_up
    (MoEShape(512, 128, 13, 256, 256), 5),     # 65 pairs: not
    (MoEShape(512, 128, 8, 768, 0), 5),        # more than 3.5 workgroups per CU: four per CU
    (MoEShape(512, 512, 8, 256, 0), 8),        # 4 workgroups per CU, 8 experts per lane: the last of them
    (MoEShape(512, 512, 8, 768, 128), 5),      # 7.7: a launch of its own
    (MoEShape(256, 1000, 4, 256, 0), 8),       # 16 experts per lane
    (MoEShape(256, 1000, 10, 256, 0), 6),      # 3.75 workgroups per CU: a launch of its own
    (MoEShape(256, 256, 8, 512, 128), 8),      # 8.1: a launch of its own
    (MoEShape(512, 48, 7, 128, 384), 9),       # 63 pairs, 9 tokens: in gate_up as T * k >= E
    (MoEShape(1024, 16, 2, 256, 0), 8),        # both apply: routed in gate_up
    (MoEShape(1024, 32, 3, 256, 0), 10),       # T * k < E
    (MoEShape(1024, 32, 2, 256, 128), 16),     # T * k = E
    (MoEShape(256, 2, 2, 65536, 0), 8),        # the largest width
    (MoEShape(256, 2, 2, 32768, 65536), 8),    # 8 tokens per expert on the tiled GEMMs: not routed inside
])
def test_small_batches(gpu, shape, T):
    _run_and_check(shape, T, gpu, seed=T + shape.num_experts)
