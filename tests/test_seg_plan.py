"""The segment plans (theorem_amd/csrc/seg_plan.h) on the host: what every plan
promises the kernels, the plans behind the GPU tests, and shapes that measured
slower or faster in segments."""
from __future__ import annotations

import itertools
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    exe = tmp_path_factory.mktemp("plan") / "seg_plan_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{ROOT / 'theorem_amd' / 'csrc'}",
                    str(ROOT / "tests" / "csrc" / "seg_plan_check.cpp"), "-o", str(exe)], check=True)

    def run(calls):
        r = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, c)) for c in calls), capture_output=True,
                           text=True, check=True)
        return [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    return run


def test_every_chunk_in_one_segment(plans):
    calls = [(f, BH, NT, K, V) for f, BH, NT, K, V in itertools.product(
        ("fwd", "hbf16", "hf32"), (1, 2, 3, 7, 12, 16, 33, 64, 100), (0, 1, 2, 3, 5, 17, 37, 64, 100, 122, 128),
        (64, 128), (64, 128))]
    for (f, BH, NT, K, V), (out, per, ln, ws) in zip(calls, plans(calls), strict=True):
        what = f"{f} {BH} {NT} {K} {V}: {out} x {per} x {ln}"
        if out == 1:
            assert (per, ln, ws) == (1, max(NT, 1), 0), what
            continue
        nt = -(-NT // ln)
        assert out >= 3 and per >= 1 and (nt - 1) * ln < NT <= nt * ln, what  # no empty transition segment
        assert (out - 1) * per < nt <= out * per, what                        # nor output segment
        assert ws == ((nt - 2) * BH * K * K + (nt - 1) * BH * K * V + BH * V // 16) * 4, what


def test_plans_of_the_gpu_tests(plans):
    """test_gpu_segment_per.py is about plans of several transition segments per
    output segment: its shapes have them, some with a remainder in each count."""
    from tests.test_gpu_segment_per import FWD, H_BF16, H_F32

    calls = [(f, B * H, NT, K, V) for f, shapes in (("fwd", FWD), ("hbf16", H_BF16), ("hf32", H_F32))
             for B, H, NT, K, V in shapes]
    got = plans(calls)
    for c, (out, per, ln, _) in zip(calls, got, strict=True):
        assert out >= 3 and per >= 2, c
    assert sum(-(-c[2] // p[2]) % p[1] != 0 for c, p in zip(calls, got)) >= 4
    assert sum(c[2] % p[2] != 0 for c, p in zip(calls, got)) >= 2


@pytest.mark.parametrize("call", [
    # us, in one piece and in segments: 83 / 90, 43 / 45, 70 / 74
    ("fwd", 40, 32, 128, 128), ("fwd", 12, 16, 128, 128), ("fwd", 63, 24, 128, 64),
    # with inputs in the memory-side cache 70 / 85, 26 / 31, 72 / 84, 22 / 26
    ("hbf16", 32, 96, 64, 128), ("hbf16", 12, 32, 64, 128), ("hbf16", 21, 64, 128, 128), ("hbf16", 6, 28, 64, 128)])
def test_one_piece_where_segments_measured_slower(plans, call):
    assert plans([call])[0][0] == 1


@pytest.mark.parametrize("call", [
    ("fwd", 16, 128, 128, 128), ("fwd", 4, 64, 128, 128), ("fwd", 16, 12, 64, 64), ("hbf16", 16, 128, 128, 128),
    ("hbf16", 4, 128, 128, 128), ("hbf16", 32, 128, 64, 128), ("hf32", 16, 32, 128, 128)])
def test_segments_where_they_measured_faster(plans, call):
    assert plans([call])[0][0] > 1
