"""Tridiagonal matrices with equal diagonal entries and couplings whose squares
underflow (1e-20 is 0 squared in FP32, 1e-170 in FP64), from rounding level
down: the leaves of the divide & conquer must give orthonormal vectors for
them, alone (orders up to 16) and under merges.  Such a matrix passes the
reduction unchanged, so its couplings arrive in the leaves as they are.

Bounds as in the eigensolver's other tests: computed values and vectors are
those of A + E, |E| <= c n eps |A|, c = 200 (eigenvalues c sqrt(n))."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [2, 5, 16, 33, 300])
def test_couplings_below_rounding(cuda, prec, n):
    import torch
    from gammcor_amd import _lib
    dt, eps = (torch.float64, 2.2e-16) if prec == "f64" else (torch.float32, 1.2e-7)
    g = [10.0 ** -x for x in (range(14, 34, 2) if prec == "f32" else range(146, 166, 2))]
    g += [np.finfo(np.float32).tiny if prec == "f32" else np.finfo(np.float64).tiny, eps, 1e-3]
    a = np.zeros((2 * len(g), n, n))
    i = np.arange(n - 1)
    for b, x in enumerate(g):
        # every coupling, and every third one with equal pairs between
        a[b, range(n), range(n)] = 1.0
        a[b, i, i + 1] = a[b, i + 1, i] = x
        c = len(g) + b
        a[c, range(n), range(n)] = 1.0 + np.arange(n) // 3
        a[c, i, i + 1] = a[c, i + 1, i] = np.where(i % 3 == 0, x, 0.0)
    at = torch.from_numpy(a).to(cuda).to(dt)
    v, w = at.clone(), torch.zeros(len(a), n, device=cuda, dtype=dt)
    print(f"leaf couplings {prec} n={n}", flush=True)
    _lib.call("gmc_syevd_dev", 0 if prec == "f64" else 1, n, len(a), v.data_ptr(), w.data_ptr(), None)
    eye = torch.eye(n, device=cuda, dtype=torch.float64)
    for b in range(len(a)):
        ab = at[b].double()
        ref = np.linalg.eigvalsh(ab.cpu().numpy())
        scale = np.max(np.abs(ref))
        wb, z = w[b].double(), v[b].double().T.contiguous()
        what = f"coupling {g[b % len(g)]:.1e}"
        assert float(torch.linalg.norm(z.T.contiguous() @ z - eye)) < 200 * n * eps, what
        assert float(torch.linalg.norm(ab @ z - z * wb[None, :])) / scale < 200 * n * eps, what
        assert np.max(np.abs(wb.cpu().numpy() - ref)) < 200 * n ** 0.5 * eps * scale, what
