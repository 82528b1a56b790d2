"""csrc/rules.hpp, compiled by a host compiler: the line between two kernels of one job takes the side
that was measured faster (GPU us of the whole call on an MI355X, both sides in one process)."""
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


# H, E, I, Is, T (8 experts per token), fp8, us streaming, us tiled. Whole rounds of the CUs with and
# without the shared expert's items past them, partly filled rounds, less than one round, a shared
# expert wider than the routed ones, short k ranges
MEASURED = [
    (1024, 64, 512, 256, 137, False, 61.8, 70.4),
    (512, 128, 384, 0, 241, False, 54.7, 49.8),
    (512, 128, 256, 256, 209, False, 42.9, 50.1),
    (512, 48, 512, 512, 103, False, 36.8, 40.9),
    (512, 160, 256, 512, 341, False, 69.2, 63.9),
    (512, 100, 512, 0, 188, False, 54.9, 50.3),
    (512, 96, 512, 256, 181, False, 57.2, 50.1),
    (512, 128, 384, 512, 241, False, 66.7, 55.5),
    (512, 100, 768, 256, 188, False, 76.0, 66.3),
    (512, 160, 768, 0, 481, False, 111.6, 95.2),
    (1024, 512, 256, 512, 1281, False, 267.4, 193.7),
    (512, 256, 512, 512, 865, False, 132.3, 112.5),
    (2048, 100, 384, 0, 163, False, 100.4, 118.8),
    (2048, 100, 768, 0, 301, False, 211.7, 197.4),
    (2048, 128, 256, 256, 161, True, 72.9, 82.6),
    (512, 96, 512, 512, 121, True, 42.4, 45.5),
    (512, 100, 256, 256, 188, True, 37.0, 40.9),
    (2048, 64, 512, 256, 81, True, 70.3, 77.9),
    (2048, 64, 512, 512, 81, True, 70.5, 79.9),
    (2048, 96, 768, 256, 121, True, 112.8, 123.6),
    (512, 128, 512, 256, 161, True, 48.6, 53.9),
    (1024, 100, 256, 512, 126, True, 51.3, 57.5),
    (512, 48, 512, 512, 73, True, 33.3, 36.7),
    (512, 100, 768, 256, 276, True, 64.7, 54.4),
    (2048, 128, 256, 0, 161, True, 74.0, 68.3),
    (2048, 100, 768, 0, 326, True, 161.7, 128.9),
    (2048, 100, 512, 256, 226, True, 101.9, 94.6),
    (512, 256, 768, 0, 833, True, 119.9, 104.2),
]


def test_tiled_line_takes_the_measured_side(tmp_path):
    got = _evaluate(tmp_path, [
        f"tiled_min_tokens(CallSizes{{{E}, {H}, {I}, {Is}, {T}, {str(fp8).lower()}, 256}})"
        for H, E, I, Is, T, fp8, _, _ in MEASURED])
    for (H, E, I, Is, T, fp8, stream, tiled), line in zip(MEASURED, got):
        assert (T * 8 / E >= line) == (tiled < stream), (H, E, I, Is, T, fp8, line)


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
