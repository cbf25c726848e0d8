"""The launch rules of ``csrc/dispatch.h``, evaluated on the CPU.

A small program prints, for one problem a line, what the rules choose:
forward shape, the splits, the projection tiles and the backward GEMM plan.
"""

from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FIELDS = ("fwd", "bwd_split", "soft_fwd_split", "soft_bwd_split", "fvals_lanes", "fvals_grid", "pbm", "pbn", "pgw", "pcpt", "pvpt",
          "nr", "bt", "g", "n_a", "p", "tiles_w", "kw", "kx")
PROGRAM = r'''
#include <cstdio>
#include "dispatch.h"
using namespace morpho;
int main() {
  long long B, N, H, M, DV, causal, det;
  while (scanf("%lld %lld %lld %lld %lld %lld %lld", &B, &N, &H, &M, &DV, &causal, &det) == 7) {
    Dims d{};
    d.causal = (int)causal;
    d.det = (int)det;
    fill_sizes(d, B, N, H * DV, H, M);
    choose_proj_tiles(d);
    const BwdGemmPlan P = bwd_gemm_plan(d);
    printf("%d %d %d %d %d %u %d %d %d %d %d %d %d %d %d %d %d %d %d\n", attn_fwd_shape(d), attn_bwd_split(d),
           soft_fwd_split(d), soft_bwd_split(d), soft_fvals_lanes(d), soft_fvals_grid(d), d.PBM, d.PBN, d.PGW, d.PCPT, d.PVPT, d.NR, P.bt,
           P.g, P.n_a, P.p, P.tiles_w, P.kw, P.kx);
  }
}
'''
REGULAR, SMALL, SPLIT = 0, 1, 2

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    """rules([(B, N, H, m, dv, causal), ...]) -> one dict of FIELDS per problem."""
    d = tmp_path_factory.mktemp("dispatch")
    (d / "rules.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{ROOT}/morphottention_amd/csrc",
                    str(d / "rules.cpp"), "-o", str(d / "rules")], check=True)

    def evaluate(problems):
        text = "".join(" ".join(str(int(v)) for v in (*p, *([0] * (7 - len(p))))) + "\n" for p in problems)
        out = subprocess.run([str(d / "rules")], input=text, capture_output=True, text=True, check=True).stdout
        rows = [dict(zip(FIELDS, map(int, line.split()))) for line in out.splitlines()]
        assert len(rows) == len(problems)
        return rows

    return evaluate


def test_rules_at_measured_points(rules):
    """The shapes at the configurations whose figures stand beside the rules."""
    c2, c3, c4, c5, image = rules([(8, 1024, 8, 16, 64, False), (4, 4096, 16, 16, 64, True),
                                   (1, 16384, 16, 32, 64, True), (16, 2048, 32, 64, 64, False),
                                   (64, 197, 12, 64, 64, False)])
    assert [r["fwd"] for r in (c2, c3, c4, c5, image)] == [SMALL, REGULAR, REGULAR, REGULAR, REGULAR]
    assert not any(r[k] for r in (c2, c3, c4, c5, image) for k in ("bwd_split", "soft_fwd_split", "soft_bwd_split"))
    assert [(r["pbm"], r["pbn"]) for r in (c2, c3, c4, c5, image)] == [
        (128, 160), (256, 320), (128, 256), (256, 256), (128, 256)]
    few, = rules([(1, 3001, 16, 16, 64, True)])
    assert few["fwd"] == SPLIT and few["bwd_split"] and few["soft_fwd_split"] and few["soft_bwd_split"]
    det, = rules([(1, 3001, 16, 16, 64, True, True)])
    assert not det["bwd_split"]


def test_projection_tiles_hold_whole_heads(rules):
    """Every projection tile holds whole heads (a head's row sums are formed
    within one tile), and rows are whole groups of 8 tokens."""
    problems = [(B, N, H, m, dv, False) for B in (1, 9, 300) for N in (1, 5, 100, 197, 2048)
                for H in (1, 2, 3, 5, 6, 7, 8, 12, 16, 20, 24, 32) for m in (16, 32, 64) for dv in (32, 64, 128)]
    for (B, N, H, m, dv, _), r in zip(problems, rules(problems)):
        assert r["nr"] == (N + 7) // 8 * 8
        if r["pcpt"]:
            groups = r["pbn"] // r["pgw"]
            assert r["pcpt"] * groups % m == 0 and r["pcpt"] % 16 == 0 and r["pvpt"] % 16 == 0
            assert (r["pcpt"] + r["pvpt"]) == r["pgw"]
        else:
            assert r["pbn"] % m == 0


def test_soft_fvals_grid_at_the_limits(rules):
    """The launch covers every column and stays below 2^31 work-items at every
    accepted size (one 256-lane workgroup per column had passed 2^32 from B D =
    2^24 on; B8192 N513 D2048 fits an MI355X)."""
    problems = [(8192, 513, 32, 16, 64, False), (1 << 25, 1, 1, 16, 32, False), (1 << 17, 600, 2, 16, 64, True),
                (1 << 20, 64, 16, 16, 64, False), (4, 4096, 16, 16, 64, True), (2, 1001, 8, 32, 64, False),
                (1, 1, 1, 16, 32, False), (3, 65, 5, 64, 128, True), (7, 200, 3, 16, 32, False)]
    for (B, N, H, m, dv, _), r in zip(problems, rules(problems)):
        cols = 256 // r["fvals_lanes"]
        assert 0 < r["fvals_grid"] * 256 < 2 ** 31
        assert r["fvals_grid"] * cols >= B * H * dv or r["fvals_grid"] == 1 << 20
        assert r["fvals_grid"] * cols - cols < B * H * dv


def test_gpu_parity_cases_run_the_shapes_they_name(rules):
    from test_gpu_parity import LAUNCH_SHAPES
    for case, r in zip(LAUNCH_SHAPES, rules([c[:6] for c in LAUNCH_SHAPES])):
        assert (("regular", "small", "split")[r["fwd"]], "split" if r["bwd_split"] else "regular") == case[6:], case


    from test_gpu_parity import EIGHT_WAVE_BWD, VARIANT_SHAPES
    for case, r in zip(VARIANT_SHAPES, rules([c[:6] for c in VARIANT_SHAPES])):
        assert (("regular", "small", "split")[r["fwd"]], "split" if r["bwd_split"] else "regular") == case[8:], case
    B, N, H = EIGHT_WAVE_BWD
    assert not any(r["bwd_split"] for r in rules([(B, N, H, m, dv, c) for m, dv in ((32, 64), (64, 32), (64, 64))
                                                  for c in (False, True)]))


def test_gpu_soft_cases_run_the_shapes_they_name(rules):
    from test_gpu_soft import BENCHMARKED_HEADS, SOFT_SHAPES
    for case, r in zip(SOFT_SHAPES, rules([c[:6] for c in SOFT_SHAPES])):
        assert (bool(r["soft_fwd_split"]), bool(r["soft_bwd_split"])) == case[8:], case
    few, many = rules([(1, 4096, H, 16, 64, True) for H in BENCHMARKED_HEADS])
    assert few["soft_fwd_split"] and few["soft_bwd_split"]
    assert not many["soft_fwd_split"] and not many["soft_bwd_split"]


def test_only_the_regular_forward_sees_long_rows(rules):
    """The small and split forwards address V^T from the head's base with 32-bit
    lane offsets, 2 dv bytes a token; their rows stay below 2^18 tokens (a
    static_assert has the offsets of 2^18 tokens fit), the regular shape takes
    every accepted length (a wrapped offset reads another token's values)."""
    cases = [(1, N, 1, m, dv, c) for N in (1 << 17, (1 << 17) + 1, 1 << 18, 16_900_000, 34_000_000, 1 << 28)
             for m in (16, 32, 64) for dv in (32, 64, 128) for c in (False, True)]
    assert all(r["fwd"] == REGULAR or case[1] < 1 << 18 for case, r in zip(cases, rules(cases)))


def test_split_shapes_stay_where_they_gain(rules):
    """No split forward for the few key tiles where one group is as fast, and no
    second round of one-per-CU workgroups for short causal chains (measured up
    to 1.2 and 1.6 times the time without)."""
    def workgroups(case):
        return case[0] * case[2] * ((case[1] + 127) // 128)

    short = [(1, N, H, m, dv, c) for N in (1, 33, 64, 100, 128, 192) for H in (1, 8) for m in (16, 32, 64)
             for dv in (32, 64, 128) for c in (False, True)]
    for case, r in zip(short, rules(short)):
        assert r["fwd"] != SPLIT and not r["bwd_split"] and not r["soft_bwd_split"], case
        assert r["soft_fwd_split"] == (case[1] > 64 and case[4] <= 64), case
    rounds = [(B, N, 8, m, dv, True) for N in (193, 256, 300, 384, 512, 640, 768) for B in range(5, 23)
              for m in (16, 32, 64) for dv in (32, 64, 128)]
    for case, r in zip(rounds, rules(rounds)):
        if workgroups(case) > 256:
            assert r["fwd"] != SPLIT and not r["soft_fwd_split"] and not r["soft_bwd_split"], case
            assert not r["bwd_split"] or (case[3] >= 32 and case[4] <= 64), case
    long = [(1, N, H, m, dv, c) for N in (1000, 3000) for H in (8, 10) for m in (16, 32, 64) for dv in (32, 64)
            for c in (False, True)]
    assert all(r["fwd"] == SPLIT and r["bwd_split"] and r["soft_fwd_split"] and r["soft_bwd_split"]
               for r in rules(long))


def test_wide_heads_keep_one_round_of_regular_workgroups(rules):
    """dv = 128 without the causal mask: the small shape takes up to 1.12 times
    the regular one's time where one regular round covers the problem."""
    cases = [(B, N, H, m, 128, c) for m in (16, 32) for N in (300, 512, 640, 1000, 1500, 3000) for B in (3, 6, 12, 24)
             for H in (8, 16) for c in (False, True)]
    for (B, N, H, m, dv, c), r in zip(cases, rules(cases)):
        regular = (N + 255) // 256 * B * H
        if r["fwd"] != SPLIT:
            assert r["fwd"] == (REGULAR if regular >= 512 or (not c and regular <= 256 and N > 512) else SMALL)
