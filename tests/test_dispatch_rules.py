"""csrc/rules.hpp, compiled by a host compiler: the line between two kernels of one job takes the side
that was measured faster (GPU us of the whole call on an MI355X, both sides in one process)."""
import math
import os
import subprocess

import pytest

RULES = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                     "layerbatch_amd", "csrc", "rules.hpp")


def _evaluate(tmp_path, exprs):
    src, exe = tmp_path / "rules_probe.cpp", tmp_path / "rules_probe"
    body = "".join(f'  std::printf("%.17g\\n", static_cast<double>({e}));\n' for e in exprs)
    src.write_text(f'#include <cstdio>\n#include "{RULES}"\nusing namespace lbmoe;\n'
                   f"int main() {{\n{body}  return 0;\n}}\n")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    return [float(v) for v in out.split()]


# H, E, I, Is, T (8 experts per token), fp8, us streaming and tiled with uniform routing, the same under a
# Zipf bias. Whole rounds of the CUs with and without the shared expert's items past them, partly filled
# rounds, less than one round, a shared expert wider than the routed ones, many and few experts
MEASURED = [
    (512, 64, 512, 512, 105, False, 40.5, 47.9, 47.0, 40.0),
    (512, 32, 768, 0, 69, False, 34.7, 38.0, 43.6, 42.0),
    (512, 48, 512, 512, 103, False, 36.8, 40.9, 45.1, 40.0),
    (2048, 160, 512, 0, 261, False, 191.7, 187.2, 212.8, 105.6),
    (1024, 160, 256, 0, 341, False, 74.6, 76.7, 115.0, 58.1),
    (512, 96, 256, 512, 157, False, 49.1, 48.4, 54.3, 45.1),
    (512, 128, 384, 512, 209, False, 64.2, 55.1, 75.0, 45.8),
    (2048, 96, 384, 512, 205, False, 121.8, 115.0, 163.8, 85.1),
    (512, 256, 512, 0, 417, False, 98.5, 92.0, 122.2, 53.8),
    (512, 512, 512, 512, 641, False, 175.8, 171.2, 182.7, 61.0),
    (2048, 96, 768, 256, 205, False, 190.1, 186.8, 237.2, 136.2),
    (2048, 512, 128, 0, 1089, False, 213.7, 192.9, 397.7, 108.2),
    (512, 96, 512, 512, 205, False, 55.7, 53.7, 70.1, 46.5),
    (512, 48, 768, 0, 79, False, 42.2, 49.0, 49.4, 43.1),
    (512, 48, 512, 0, 79, False, 33.0, 35.7, 38.4, 38.5),
    (512, 96, 256, 256, 157, False, 36.5, 41.0, 45.1, 41.1),
    (512, 512, 768, 0, 641, True, 158.3, 166.1, 263.4, 64.4),
    (2048, 96, 768, 0, 121, True, 113.9, 112.8, 158.4, 88.9),
    (2048, 48, 768, 256, 133, True, 88.7, 80.5, 137.9, 85.6),
    (1024, 160, 512, 256, 441, True, 99.2, 84.1, 172.6, 63.3),
    (2048, 128, 512, 256, 161, True, 107.8, 116.0, 162.5, 76.6),
]


def test_tiled_line_takes_the_faster_side_of_the_mix(tmp_path):
    """Three uniform calls to one under a bias, by the expected logarithm of the time."""
    got = _evaluate(tmp_path, [
        f"tiled_min_tokens(CallSizes{{{E}, {H}, {I}, {Is}, {T}, {str(fp8).lower()}, 256}})"
        for H, E, I, Is, T, fp8, *_ in MEASURED])
    for (H, E, I, Is, T, fp8, us, ut, zs, zt), line in zip(MEASURED, got):
        gain = 0.75 * math.log(us / ut) + 0.25 * math.log(zs / zt)
        assert (T * 8 / E >= line) == (gain > 0), (H, E, I, Is, T, fp8, line)


# H, E, k, I, Is, T, us with a routing launch, us routed inside gate_up
MEASURED_ROUTE = [
    (1024, 20, 3, 512, 0, 8, 25.3, 23.6), (1024, 256, 10, 256, 256, 6, 36.9, 33.7),
    (1536, 64, 10, 384, 0, 5, 41.9, 39.9), (2048, 160, 9, 512, 256, 7, 81.7, 79.7),
    (1024, 256, 8, 512, 256, 8, 55.5, 57.2), (512, 160, 8, 768, 0, 6, 35.7, 38.0),
    (512, 100, 12, 768, 0, 5, 37.8, 41.8), (1024, 512, 4, 512, 0, 8, 36.4, 34.2),
    (2048, 512, 8, 256, 0, 8, 55.8, 53.4), (1536, 512, 7, 384, 0, 6, 45.2, 42.8),
    (1536, 512, 7, 384, 0, 7, 51.7, 56.1), (512, 512, 8, 512, 0, 5, 30.2, 31.2),
    (1024, 1000, 8, 256, 0, 6, 36.5, 34.8), (1024, 1000, 8, 256, 0, 7, 38.9, 42.2),
    (2048, 1000, 3, 512, 0, 8, 48.6, 46.9), (1024, 1000, 6, 256, 256, 8, 37.7, 41.3),
    (2048, 1024, 8, 512, 0, 8, 86.1, 91.8),
]


def test_routing_inside_gate_up_takes_the_measured_side(tmp_path):
    got = _evaluate(tmp_path, [
        f"route_in_gate_up_pays(CallSizes{{{E}, {H}, {I}, {Is}, {T}, false, 256}}, {k})"
        for H, E, k, I, Is, T, _, _ in MEASURED_ROUTE])
    for case, inside in zip(MEASURED_ROUTE, got):
        assert bool(inside) == (case[-1] < case[-2]), case


# H, E, k, Is, T (I = 256), us with the plain router behind the norm, us with the selecting one
MEASURED_NORM = [
    (2048, 96, 1, 512, 4096, 145.5, 155.4), (1024, 64, 1, 512, 3000, 80.4, 86.1),
    (512, 64, 1, 512, 2048, 57.9, 62.8), (512, 16, 2, 0, 1024, 46.2, 48.5),
    (2048, 128, 2, 512, 2048, 137.5, 144.1), (2048, 48, 4, 0, 1500, 103.5, 98.7),
    (2048, 16, 2, 0, 1500, 84.4, 81.0), (2048, 128, 8, 0, 1024, 127.5, 122.9),
]


def test_norm_path_takes_the_measured_router(tmp_path):
    got = _evaluate(tmp_path, [
        f"norm_takes_selecting_router(CallSizes{{{E}, {H}, 256, {Is}, {T}, false, 256}})"
        for H, E, _, Is, T, _, _ in MEASURED_NORM])
    for case, selecting in zip(MEASURED_NORM, got):
        assert bool(selecting) == (case[-1] < case[-2]), case


@pytest.mark.parametrize("E,I", [(16, 512), (4, 768), (1, 256)])
def test_few_items_stay_on_the_streaming_kernels(tmp_path, E, I):
    sizes = [f"CallSizes{{{E}, 2048, {I}, {Is}, 50, {fp8}, 256}}" for Is in (0, 512)
             for fp8 in ("true", "false")]
    assert _evaluate(tmp_path, [f"tiled_min_tokens({s})" for s in sizes]) == [28.0] * 4


def test_the_gpu_tests_lie_on_both_sides_of_the_line(tmp_path):
    from tests.test_gpu_perm_build import SWITCH
    at = [(s, t - d, fp8) for s, t, fp8 in SWITCH for d in (1, 0)]
    got = _evaluate(tmp_path, [
        f"tiled_min_tokens(CallSizes{{{s.num_experts}, {s.hidden_size}, {s.moe_intermediate_size}, "
        f"{s.shared_expert_intermediate_size}, {t}, {str(fp8).lower()}, 256}})" for s, t, fp8 in at])
    tiled = [t * s.top_k / s.num_experts >= line for (s, t, _), line in zip(at, got)]
    assert tiled == [False, True] * len(SWITCH)
