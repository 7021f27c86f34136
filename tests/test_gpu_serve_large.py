"""Batches and request size: on target tiles requests of more than 2^14 bodies run
alone unless batch_delay_ms holds batches open; smaller ones that are ready
together are fused past them.  Results are the same either way (1e-12: the order
of additions)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("device", [0, 1])
def test_large_requests_run_alone(precision, device):
    import exafmm_amd as F
    sizes = [120000, 900, 16385, 16384, 20000, 5000, 40, 1200]  # the first keeps the slot busy
    systems = [F.make_bodies(n, "plummer1" if i % 2 else "cube1", 60 + i) for i, n in enumerate(sizes)]
    got = []
    for delay in (0.0, 1000.0):
        s = F.Server(P=6, precision=precision, slots=1, batch_requests=64, batch_delay_ms=delay, plan_on_device=device)
        ids = [s.submit(x, q) for x, q in systems]
        got.append([s.wait(i) for i in ids])
        s.close()
    for (a, ia), (b, ib), n in zip(got[0], got[1], sizes):
        assert ia["n"] == ib["n"] == n
        if n > 16384:
            assert ia["batch_requests"] == 1
        assert np.linalg.norm(a[:, 0] - b[:, 0]) <= 1e-12 * np.linalg.norm(b[:, 0])
        assert np.linalg.norm(a[:, 1:] - b[:, 1:]) <= 1e-12 * np.linalg.norm(b[:, 1:])
    assert max(i["batch_requests"] for _, i in got[1]) > 2
    assert any(i["batch_requests"] > 1 for (_, i), n in zip(got[1], sizes) if n > 16384)
