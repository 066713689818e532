"""Which kernels a grouped call runs on (csrc/grouped_plan.h), without a GPU:
the header is plain C++, compiled here and asked."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MAIN = """
#include <cstdio>
#include "grouped_plan.h"
int main() {
  int T, k, E, H, F, s;
  while (scanf("%d %d %d %d %d %d", &T, &k, &E, &H, &F, &s) == 6) {
    const grouped_plan p = plan_grouped(T, k, E, H, F, s != 0);
    printf("%s %d\\n", !p.octets ? "pairs" : !p.stacked ? (p.octet_f64 ? "octets_f64" : "octets") : p.in_order ? "stacked_f32" : "stacked_f64", p.item_rows);
  }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    exe = d / "plan"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(REPO, "llama-sandbox_amd", "csrc"),
                    "-o", str(exe), str(d / "main.cpp")], check=True)

    def ask(calls):  # calls: (T, k, E, H, F, shared) -> (kernels, rows of an item)
        text = "".join(" ".join(str(int(v)) for v in c) + "\n" for c in calls)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.split("\n")
        return [(o.split()[0], int(o.split()[1])) for o in out if o]

    return ask


# Calls that leave the chip unfilled, which the stacked kernels run slower than
# the octets (us per layer with cold weights, octets / stacked).
SLOWER_STACKED = [
    (8, 2, 8, 5120, 1536, False),      # 33 / 46
    (64, 2, 8, 5120, 1536, False),     # 49 / 61
    (16, 2, 8, 6400, 2560, False),     # 60 / 66
    (128, 2, 8, 2048, 768, False),     # 28 / 38
    (24, 4, 32, 2048, 768, True),      # 31 / 36
    (16, 2, 8, 1152, 512, False),
    (128, 2, 8, 4096, 640, False),
    (16, 2, 8, 7168, 2048, False),     # 46 / 65
    (32, 2, 8, 2048, 1024, False),     # 22 / 30
]

# and calls that gain from them: enough workgroups (octets / stacked)
FASTER_STACKED = [
    (300, 6, 160, 5120, 1536, True, "stacked_f64"),
    (128, 2, 8, 5120, 1536, False, "stacked_f64"),     # 70 / 65
    (32, 8, 128, 5120, 1536, True, "stacked_f64"),     # 261 / 251
    (64, 4, 32, 6400, 2560, True, "stacked_f64"),      # 217 / 185
    (256, 8, 128, 6400, 2560, True, "stacked_f64"),    # 1095 / 719
    (512, 4, 32, 1152, 512, True, "stacked_f64"),
    (64, 8, 256, 7168, 2048, True, "stacked_f32"),
    (32, 2, 8, 7168, 2048, False, "stacked_f32"),      # 62 / 59
    (128, 8, 128, 7168, 2048, True, "stacked_f32"),    # 628 / 525
    (512, 8, 256, 7168, 2048, True, "stacked_f32"),
    (509, 6, 384, 7168, 3072, True, "stacked_f32"),
    (512, 4, 32, 2048, 1024, True, "stacked_f32"),     # 146 / 74
]


def test_small_calls_run_on_octets(plan):
    f32 = [(7168, 2048), (2048, 1024)]
    assert plan(SLOWER_STACKED) == [("octets" if c[3:5] in f32 else "octets_f64", 8) for c in SLOWER_STACKED]


def test_full_calls_run_stacked(plan):
    assert [p[0] for p in plan([c[:6] for c in FASTER_STACKED])] == [c[6] for c in FASTER_STACKED]


def test_items_of_64_rows_only_where_the_chip_stays_full(plan):
    """Two token tiles halve the workgroups: us per layer, 32-row / 64-row items."""
    slower = [(128, 2, 8, 7168, 2048, False),    # 78 / 92
              (128, 4, 32, 7168, 2048, True),    # 170 / 175
              (512, 4, 32, 7168, 2048, True),    # 323 / 340
              (256, 2, 8, 2048, 1024, False),    # 35 / 48
              (256, 4, 32, 2048, 1024, True),    # 54 / 65
              (64, 4, 32, 2048, 1024, True)]     # 45 / 54: the shared expert's item of 64 rows
    faster = [(512, 8, 128, 7168, 2048, True),   # 748 / 718
              (256, 4, 32, 7168, 2048, True),    # 230 / 209: an expert is one item
              (913, 3, 63, 7168, 1536, True),    # 466 / 371: the same
              (1024, 8, 128, 4096, 1536, True),
              (512, 8, 256, 7168, 2048, True),   # Zipf 682 / 658
              (509, 6, 384, 7168, 3072, True),   # Zipf 768 / 746
              (2048, 8, 256, 7168, 2048, True)]  # 2298 / 2115
    assert plan(slower) == [("stacked_f32", 32)] * len(slower)
    assert plan(faster) == [("stacked_f32", 64)] * len(faster)


def test_plan_limits(plan):
    """Pairs up to 4 tokens; never stacked below 2 pairs per expert; the f32
    loops only where K of both kernels is whole groups of 4 quads (they have no
    code for a partial one)."""
    calls = [(T, k, E, 128 * h, 128 * f, s) for T in (2, 4, 5, 9, 64, 700, 8191) for k in (1, 3, 8)
             for E in (8, 33, 384, 1024) for h in (1, 5, 16, 31, 32, 48, 56, 80) for f in (1, 4, 6, 8, 12, 13, 16, 24, 28)
             for s in (0, 1)]
    seen = set()
    for (T, k, E, H, F, _), (kind, rows) in zip(calls, plan(calls)):
        assert (kind == "pairs") == (T <= 4)
        if T * k < 2 * E:
            assert kind in ("pairs", "octets")
        if kind == "stacked_f32":
            assert H % 512 == 0 and F % 512 == 0
        assert rows in {"pairs": (4,), "octets": (8,), "octets_f64": (8,), "stacked_f64": (32,), "stacked_f32": (32, 64)}[kind]
        seen.add((kind, rows))
    assert len(seen) == 6


def test_gpu_tests_reach_the_kernels_they_name(plan):
    import test_gpu_block as gpu

    for H, F, E, first, rest in gpu.STACKED_EDGES:
        T = sum(first) + rest * (E - len(first))
        kinds = plan([(T, 1, E, H, F, s) for s in (False, True)])
        assert kinds == [("stacked_f32", 64 if E == 128 else 32) if H == 2048 else ("stacked_f64", 32)] * 2, (H, F)
    # the layers of test_out_of_range_ids_contribute_nothing
    dropped = plan([(12, 4, 32, 2048, 768, False), (16, 8, 256, 7168, 2048, True), (64, 8, 256, 7168, 2048, True),
                    (160, 4, 16, 1152, 512, True), (160, 4, 16, 1152, 512, False), (192, 4, 128, 2048, 1024, True)])
    assert dropped[:2] == [("octets", 8), ("octets", 8)]
    assert dropped[2:] == [("stacked_f32", 32), ("stacked_f64", 32), ("stacked_f64", 32),
                       ("stacked_f32", 64)]
    for H, F, E, T, few in gpu.F64_LAYERS:
        assert plan([(T, 1, E, H, F, False), (few, 1, E, H, F, False)]) == [("stacked_f64", 32), ("octets_f64", 8)]
    sweep = [c for c in gpu.SWEEP if c[4] > 1]
    kinds = [k for k, _ in plan([(T, k, E, H, F, sh) for H, F, E, k, T, sh, _, _ in sweep])]
    assert {"pairs", "octets", "octets_f64", "stacked_f32", "stacked_f64"} <= set(kinds)
    octets = {c[1] // 128 for c, k in zip(sweep, kinds) if k == "octets"}  # F / 128: the down kernel's instance
    assert {6, 8, 16, 28} <= octets and octets - {6, 8, 16, 28}  # k_down_ol<6, 8, 16, 28> and k_down_o
