"""Counts of the device walk past 32 bits.  On the host: the bounds themselves
(tests/cpp/visit_counts_check.cpp; a round of 2^32 and one children used to be
taken for a round of one).  On the GPU: a walk with a round of more than 2^25
pairs, whose children are added up in 64 bits: the host's lists."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_counts_past_an_int(tmp_path):
    exe = str(tmp_path / "visit_counts_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "exafmm-beta_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "visit_counts_check.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout


@pytest.mark.gpu
def test_round_counted_in_64_bits():
    """25579 cells, the last round 34080262 pairs (64 times that passes an int)."""
    import exafmm_amd as F
    x, q = F.make_bodies(60000, "cube1", 5)
    kw = dict(ncrit=8, theta=0.15, nspawn=1)
    h = F.Plan(x, **kw)
    with F.FMM(P=2, m2l_mode=F.M2L_TARGET, **kw) as f:
        f.set_bodies(x, q)
        for k in ("m2l_pairs", "p2p_pairs", "p2p_body_pairs"):
            assert f.stats()[k] == h.stats()[k], k
        for a, b in zip(f.lists(), h.lists()):
            assert np.array_equal(a, b)
