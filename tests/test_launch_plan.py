"""What a batch's launches tell their kernels, from the library's own host code
over recording launchers (tests/cpp/launch_plan.cpp; no GPU).

A greedy row has no uniform: its place in the uniforms, or the index its entry
holds, may lie outside them. Every kernel that would read a row's uniform
before its record must therefore be told of greedy rows."""
import json
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
BIN = os.path.join(HERE, "cpp", "_build", "launch_plan")
LEAN_GREEDY = 0x80000000


def plan(*batches):
    assert os.path.exists(BIN), "build first: python tests/cpp/build.py"
    res = subprocess.run([BIN, *batches], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stderr
    out = [json.loads(line) for line in res.stdout.splitlines()]
    for b in out:
        assert b["rc"] == 0, b
        assert b["launches"], b
    return out


@pytest.mark.parametrize("batch,launch", [
    ("kkkg", "merge_small"), ("gk", "merge_small"), ("gug", "uncut"), ("ng", "cut"),
    ("nkug", "cut"), ("dugd", "residual"), ("gd", "residual")])
def test_launches_know_of_greedy_rows(batch, launch):
    (b,) = plan(batch)
    names = [l["launch"] for l in b["launches"]]
    assert launch in names, names
    for l in b["launches"]:
        # A sampled row, whose uniform stands for those a greedy row lacks.
        assert l["uniform_row"] == next(r for r, k in enumerate(batch) if k != "g")
        if l["launch"] == "merge_small":
            assert l["late_uniform"] == 1 and l["chunks"] == 3
        if l["launch"] == "residual":
            # The lean (drafted) rows lead; each greedy row is marked.
            marked = {v & ~LEAN_GREEDY: bool(v & LEAN_GREEDY) for v in l["row_of"]}
            assert marked == {r: k == "g" for r, k in enumerate(batch)}


@pytest.mark.parametrize("batch", ["kkk", "uuu", "nku", "dud"])
def test_sampled_launches_read_uniforms_early(batch):
    (b,) = plan(batch)
    for l in b["launches"]:
        assert l["uniform_row"] == 0xffffffff
        assert l.get("late_uniform", 0) == 0
        assert all(v < LEAN_GREEDY for v in l.get("row_of", []))


@pytest.mark.parametrize("rows", [1, 64, 32767, 32768, 32769, 65535, 65536, 65600, 300001])
def test_cut_slices_of_any_row_count(rows):
    """The cut passes' launches hold every row once, each in a grid a launch
    may have (65,535 blocks in y), and the slice numbers fit their argument."""
    (b,) = plan(f"n:{rows}")
    (cut,) = [l for l in b["launches"] if l["launch"] == "cut"]
    assert sum(cut["slices"]) == rows
    assert all(n == 32768 for n in cut["slices"][:-1]) and 0 < cut["slices"][-1] <= 32768
    assert 4194304 // 32768 <= 1 << 16
