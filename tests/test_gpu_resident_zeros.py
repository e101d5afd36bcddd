"""The register-resident tridiagonalisation on matrices full of exact zeros
(its exchange marks a word that is not there yet by zero and sends a zero as
-0), at the edges of its two layouts: 64-column chunks, 4 and 8 of them, the
last order of the layout by whole rows and the first of the other.

Bounds: the computed values are those of A + E, |E| <= c n eps |A|, c = 200 as
in the eigensolver's other tests (eigenvalues c sqrt(n))."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(kind, n, rng):
    a = np.zeros((n, n))
    if kind == "diagonal":
        a[np.arange(n), np.arange(n)] = rng.standard_normal(n)
    elif kind == "tridiagonal":
        e = rng.standard_normal(n - 1)
        a[np.arange(n - 1), np.arange(1, n)] = a[np.arange(1, n), np.arange(n - 1)] = e
    elif kind == "corner":
        a[0, n - 1] = a[n - 1, 0] = 1.0
    elif kind == "blocks":
        h = n // 2
        b = rng.standard_normal((h, h))
        a[:h, :h] = b + b.T
    return a


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [2, 9, 63, 65, 256, 257, 512, 513, 1030])
def test_resident_zeros(cuda, prec, n):
    import torch
    from gammcor_amd import _lib
    dt = torch.float64 if prec == "f64" else torch.float32
    kinds = ["zero", "diagonal", "tridiagonal", "corner", "blocks"]
    rng = np.random.default_rng(n)
    a = torch.from_numpy(np.stack([_matrix(k, n, rng) for k in kinds])).to(cuda).to(dt)
    v, w = a.clone(), torch.zeros(len(kinds), n, device=cuda, dtype=dt)
    print(f"resident zeros {prec} n={n}", flush=True)
    _lib.call("gmc_syevd_dev", 0 if prec == "f64" else 1, n, len(kinds), v.data_ptr(), w.data_ptr(), None)
    eps = 2.2e-16 if prec == "f64" else 1.2e-7
    for b, kind in enumerate(kinds):
        ab = a[b].double()
        ref = np.linalg.eigvalsh(ab.cpu().numpy())
        scale = max(1.0, np.max(np.abs(ref)))
        wb, z = w[b].double(), v[b].double().T.contiguous()
        assert np.max(np.abs(wb.cpu().numpy() - ref)) < 200 * n ** 0.5 * eps * scale, kind
        assert float(torch.linalg.norm(ab @ z - z * wb[None, :])) / scale < 200 * n * eps, kind
        eye = torch.eye(n, device=cuda, dtype=torch.float64)
        assert float(torch.linalg.norm(z.T.contiguous() @ z - eye)) < 200 * n * eps, kind
