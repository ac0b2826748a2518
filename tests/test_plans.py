"""The dispatch rules of the batched attention and products (csrc/plans.h), CPU only.

The header is compiled for the host, so these tests ask the code itself which
form a call takes: that the GPU tests' case lists reach every form, and that
the forms chosen at measured sizes are those measured as the faster ones."""

from __future__ import annotations

import json
import shutil
import subprocess
from pathlib import Path

import pytest

import test_gpu_attention_any as attention_any
import test_gpu_decode as decode
import test_gpu_gemm as gemm
import test_gpu_long_context as long_context
import test_gpu_prefill_ops as prefill_ops

NATIVE = Path(__file__).resolve().parent / "native"


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    """plan(line, ...) -> what plans.h says of each call (plan_dump.cpp)."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path_factory.mktemp("plans") / "plan_dump"
    subprocess.run(["g++", "-O1", "-std=c++17", str(NATIVE / "plan_dump.cpp"), "-o", str(exe)], check=True)

    def run(lines):
        out = subprocess.run([str(exe)], input="\n".join(lines), check=True, capture_output=True, text=True).stdout
        plans = [json.loads(line) for line in out.splitlines()]
        assert len(plans) == len(lines)
        return plans

    return run


def attn_line(nh, nkv, hd, kf, vf, cap, sw, start, batch):
    wlimit = sw if sw is not None and 0 < sw < cap else cap
    return f"attn {start} {batch} {nh} {nkv} {hd} {kf} {vf} {cap} {wlimit}"


def prefill_cases():
    """Every attention_prefill call whose rows the GPU tests compare with the oracle."""
    yield from attention_any.MANY_ROWS
    for start, batch, sw, cap, nh, nkv, _ in prefill_ops.PREFILL_CASES:
        rows = max(1, (64 << 20) // (4 * nh * cap))  # a launch's scores stay within 64 MiB
        for r0 in range(0, batch, rows):
            yield nh, nkv, 256, 0, 0, cap, sw, start + r0, min(rows, batch - r0)


def test_score_blocks_dispatch_their_windows(plan):
    """A row block's tiles hold every position its rows see, and under a sliding
    window few beyond them (the tiles of the whole launch left most workgroups without work)."""
    cases = [(nh, nkv, 256, kf, 0, 4096, sw, start, batch)
             for nh, nkv in ((8, 8), (8, 4), (12, 4), (8, 1)) for kf in (0, 1)
             for sw in (None, 1, 20, 63, 64, 65, 130, 1000)
             for start, batch in ((0, 1), (0, 200), (37, 64), (1000, 1), (1000, 500), (3000, 129))]
    for (nh, nkv, _, kf, _, cap, sw, start, batch), p in zip(cases, plan([attn_line(*c) for c in cases])):
        g, limit = nh // nkv, sw or cap
        chains, per = batch * g, 4 * p["score_m"] * p["score_reps"]
        t_lo = max(0, start + 1 - limit)
        assert p["score_blocks"] * per >= chains > (p["score_blocks"] - 1) * per
        for c0 in range(0, chains, per):
            first, last = start + c0 // g, start + (min(c0 + per, chains) - 1) // g
            tile0 = t_lo + (max(0, first + 1 - limit) - t_lo) // 64 * 64
            assert tile0 <= max(0, first + 1 - limit) and tile0 + 64 * p["tiles"] > last
        assert 4 * 64 * p["tiles"] <= 5 * (limit + per // g + 1 + 3 * 64)


# (heads, kv heads, dims, K format, start, batch): where the decode kernels' scores measured
# faster, and where not
ONE_ROW = [(8, 4, 256, 0, 100, 16), (8, 8, 256, 0, 0, 64), (4, 4, 256, 0, 700, 8), (16, 4, 256, 0, 40, 8),
           (8, 8, 64, 0, 0, 8), (2, 2, 32, 0, 700, 3), (32, 8, 64, 0, 100, 3)]
NOT_ONE_ROW = [(8, 4, 256, 0, 700, 32), (8, 8, 256, 0, 100, 64), (16, 4, 256, 0, 0, 4), (8, 1, 256, 0, 0, 8),
               (8, 1, 512, 0, 0, 3), (8, 4, 256, 1, 0, 3), (8, 8, 64, 0, 2500, 16)]


def test_few_rows_take_the_decode_scores(plan):
    for cases, want in ((ONE_ROW, 1), (NOT_ONE_ROW, 0)):
        lines = [attn_line(nh, nkv, hd, kf, 0, 4096, None, start, batch) for nh, nkv, hd, kf, start, batch in cases]
        assert [p["one_row_scores"] for p in plan(lines)] == [want] * len(cases)
    windows = [attn_line(8, 8, 256, 0, 0, 4096, w, 1000, 20) for w in (64, 65, 72, 73, 200, 208)]
    assert [p["one_row_scores"] for p in plan(windows)] == [1, 0, 0, 1, 0, 1]
    assert plan([attn_line(8, 8, 64, 0, 0, 4096, 200, 1000, 10)])[0]["one_row_scores"] == 1


# (V format, workgroups of the decode form, widest window) -> the rows form measured the faster
LINE = {(0, 256, 10): 0, (0, 512, 60): 1, (0, 512, 200): 0, (0, 768, 500): 1, (0, 768, 1000): 0, (0, 1024, 2000): 1,
        (1, 256, 10): 0, (1, 512, 20): 1, (1, 512, 60): 0, (1, 768, 120): 1, (1, 768, 500): 0, (1, 1024, 350): 1,
        (1, 1024, 1000): 0, (2, 1280, 700): 1, (2, 1280, 2000): 0, (2, 1536, 1000): 1}


def test_line_between_decode_and_rows_form(plan):
    got = plan([attn_line(8, 4, 256, vf, vf, 4096, None, span - wgs // 64, wgs // 64) for vf, wgs, span in LINE])
    assert [p["rows_form"] for p in got] == list(LINE.values())


# (heads = kv heads, window, start, batch) -> whether softmax and sum in one launch measured the faster
SHORT = {(8, None, 0, 1): 1, (8, None, 60, 1): 0, (8, None, 0, 64): 1, (8, None, 60, 16): 1, (8, None, 60, 50): 0,
         (8, None, 200, 9): 0, (8, 20, 1000, 200): 1, (8, 60, 1000, 64): 1, (16, 60, 1000, 100): 0}


def test_short_windows_of_single_heads_in_one_launch(plan):
    got = plan([attn_line(h, h, 256, 0, 0, 4096, sw, start, batch) for h, sw, start, batch in SHORT])
    assert [p["short_form"] for p in got] == list(SHORT.values())
    others = [attn_line(8, 4, 256, 0, 0, 4096, 20, 1000, 64), attn_line(8, 8, 128, 0, 0, 4096, 20, 1000, 64),
              attn_line(8, 8, 256, 0, 1, 4096, 20, 1000, 64)]
    assert [p["short_form"] for p in plan(others)] == [0, 0, 0]


# (heads, kv heads, dims, V format, window, start, batch) -> chain rows a wave x dims a lane of the weighted sum,
# measured the fastest of the four there
PV = {(8, 4, 256, 0, None, 2500, 40): [2, 1], (8, 4, 256, 0, None, 2500, 80): [2, 1],
      (8, 4, 256, 0, None, 2500, 150): [4, 1], (4, 4, 256, 0, None, 950, 64): [1, 1],
      (8, 1, 512, 0, None, 2500, 300): [4, 2], (8, 8, 64, 0, None, 300, 500): [2, 1],
      (8, 4, 256, 0, 20, 1000, 200): [2, 1], (8, 4, 256, 1, None, 2500, 40): [2, 1],
      (8, 4, 256, 1, None, 2500, 150): [4, 2], (8, 2, 128, 1, None, 2500, 80): [2, 1],
      (8, 4, 256, 2, None, 2500, 40): [2, 1], (8, 4, 256, 2, None, 2500, 80): [4, 1],
      (8, 4, 256, 2, None, 2500, 300): [4, 2], (16, 4, 128, 2, None, 2500, 300): [4, 1],
      (8, 8, 64, 2, None, 2500, 80): [1, 1], (8, 8, 64, 2, None, 2500, 300): [4, 1]}


def test_weighted_sum_form(plan):
    got = plan([attn_line(nh, nkv, hd, vf, vf, 4096, sw, start, batch) for nh, nkv, hd, vf, sw, start, batch in PV])
    assert [p["pv"] for p in got] == list(PV.values())


def test_prefill_cases_reach_every_form(plan):
    cases = list(prefill_cases())
    plans = plan([attn_line(*c) for c in cases])
    scores, softmax, weighted = set(), set(), set()
    for (nh, nkv, hd, kf, vf, *_), p in zip(cases, plans):
        if p["one_row_scores"]:
            scores.add("tuned" if hd == 256 else "any")
        else:
            scores.add((kf, p["score_m"], min(p["score_reps"], 2)))
        if p["short_form"]:
            weighted.add("short")
        elif p["rows_form"]:
            chunks = p["span"] > 4 * p["softmax_threads"]
            softmax.add((p["softmax_threads"], chunks))
            weighted.add((vf, *p["pv"]))
        else:
            weighted.add((vf, "long" if p["long"] else "decode"))
    assert scores >= {"tuned", "any"}
    assert scores >= {(0, 1, 1), (0, 2, 1), (0, 4, 1), (0, 4, 2), (1, 4, 1), (1, 4, 2), (2, 4, 1), (2, 4, 2)}
    assert softmax >= {(64, False), (256, False), (256, True), (512, False), (1024, False), (1024, True)}
    forms = [(4, 2), (4, 1), (2, 1), (1, 1)]
    assert weighted >= {(vf, *f) for vf in range(3) for f in forms if (vf, f) != (1, (4, 1))}  # (not built)
    assert weighted >= {(vf, f) for vf in range(3) for f in ("decode", "long")} | {"short"}


def gemm_plans(plan, cases):
    return plan([f"gemm {rows} {cols} {batch}" for rows, cols, batch in cases])


def test_gemm_cases_are_on_their_side_of_the_line(plan):
    few = [p["few"] for p in gemm_plans(plan, gemm.FEW_CASES)]
    assert few == [1] * (len(few) - 1) + [0]
    cases = gemm.TILE_CASES
    plans = gemm_plans(plan, cases)
    assert not any(p["few"] for p in plans)
    full = [(c, p) for c, p in zip(cases, plans) if p["full_tiles"] == p["tiles"]]
    half = [(c, p) for c, p in zip(cases, plans) if p["full_tiles"] < p["tiles"]]
    assert {c[1] // 32 % 8 for c, _ in full if c[1] // 32 > 8} == set(range(8))  # every tail after a whole chunk
    assert {c[1] // 32 for c, _ in full if c[1] // 32 < 8} == set(range(1, 8))   # and before any
    for kind in (full, half):
        assert any(c[0] % 32 and c[0] % 4 for c, _ in kind) and any(c[0] % 4 == 0 for c, _ in kind)


# (rows, cols, batch) -> few-token kernel in EXACT, in FAST, measured as the faster one
GEMM_LINE = {(4608, 512, 128): (0, 0), (18432, 512, 32): (1, 1), (4096, 512, 128): (1, 1), (4608, 2304, 128): (1, 0),
             (2304, 2304, 256): (1, 0), (18432, 2304, 32): (1, 1), (5120, 2304, 128): (0, 0), (4608, 4096, 128): (1, 1),
             (4608, 9216, 128): (1, 1), (9216, 2304, 80): (0, 0)}


def test_few_token_line(plan):
    got = [(p["few"], p["few_fast"]) for p in gemm_plans(plan, GEMM_LINE)]
    assert got == list(GEMM_LINE.values())


def test_fast_prefill_test_has_both_folds(plan):
    layer = decode.FAST_LAYER.values()
    got = gemm_plans(plan, [(rows, cols, 150) for rows, cols, _ in layer])
    assert [not p["few_fast"] for p in got] == [relaxed for _, _, relaxed in layer]


def test_long_cases_are_long(plan):
    """The windows of the long-context tests that are meant for the long softmax, on both sides of its chunks."""
    windows = [min(n_past + 1, cap) for n_past, cap in long_context.LONG_CASES]
    long = {w for w, p in zip(windows, plan([f"span {w}" for w in windows])) if p["long"]}
    assert long >= {10241, 16381, 16382, 16383, 16384, 24573}
    assert {6144, 8191, 8192, 10240} <= set(windows) - long
    assert plan(["span 12288"])[0]["long"]  # test_attention_long_form_short_windows
