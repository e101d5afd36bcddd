"""A matrix with one NaN or infinite entry among finite ones in a batch of the
eigensolver: every eigenvalue word of it is written, some of them not finite, and
the other problems' results are those they have alone.  The orders run the leaves
alone, both resident layouts and the panels with word exchanges."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,batch", [(1, 3), (12, 3), (40, 3), (300, 3), (700, 3), (1028, 12)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_one_problem_not_finite(cuda, prec, n, batch, bad):
    import torch
    from gammcor_amd import _lib
    dt = torch.float64 if prec == "f64" else torch.float32
    g = torch.Generator(device=cuda)
    g.manual_seed(n)
    a = torch.randn(batch, n, n, generator=g, device=cuda, dtype=torch.float64)
    a = (a + a.transpose(1, 2)).contiguous().to(dt)

    def solve(x):
        v, w = x.clone(), torch.full((batch, n), 7.5e8, device=cuda, dtype=dt)
        print(f"not finite: {prec} n={n} batch={batch} {bad}", flush=True)
        _lib.call("gmc_syevd_dev", 0 if prec == "f64" else 1, n, batch, v.data_ptr(), w.data_ptr(), None)
        return v, w

    # (the deterministic mode: the finite problems' results bit for bit)
    _lib.call("gmc_set_deterministic", 1)
    try:
        v0, w0 = solve(a)
        b = a.clone()
        i, j = (3 * n) // 4, n // 3
        b[1, i, j] = b[1, j, i] = bad
        v1, w1 = solve(b)
    finally:
        _lib.call("gmc_set_deterministic", 0)
    assert not bool((w1 == 7.5e8).any())
    assert not bool(torch.isfinite(w1[1]).all())
    for p in range(batch):
        if p != 1:
            assert torch.equal(w0[p], w1[p]) and torch.equal(v0[p], v1[p])
