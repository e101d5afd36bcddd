"""Symmetric matrices times a large power of two, the squares of their entries
in range but not the cubes: the eigensolver's reductions (both layouts of the
resident one, the panels before it) must give the vectors of the unscaled
matrix and its values times the same power.

Bounds as in the eigensolver's other tests: computed values and vectors are
those of A + E, |E| <= c n eps |A|, c = 200 (eigenvalues c sqrt(n))."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,batch", [(12, 2), (300, 2), (512, 2), (514, 2), (1030, 2), (1030, 12), (1537, 1), (2048, 1)])
def test_scaled_matrices(cuda, prec, n, batch):
    import torch
    from gammcor_amd import _lib
    dt, eps = (torch.float64, 2.2e-16) if prec == "f64" else (torch.float32, 1.2e-7)
    g = torch.Generator(device=cuda)
    g.manual_seed(n + batch)
    a = torch.randn(batch, n, n, generator=g, device=cuda, dtype=torch.float64)
    a = (a + a.transpose(1, 2)).contiguous().to(dt)
    ref = [np.linalg.eigvalsh(a[b].double().cpu().numpy()) for b in (0, batch - 1)]
    eye = torch.eye(n, device=cuda, dtype=torch.float64)
    for k in ((360, 400) if prec == "f64" else (44, 48)):
        f = 2.0 ** k
        v, w = a * f, torch.zeros(batch, n, device=cuda, dtype=dt)
        print(f"scale 2^{k} {prec} n={n} batch={batch}", flush=True)
        _lib.call("gmc_syevd_dev", 0 if prec == "f64" else 1, n, batch, v.data_ptr(), w.data_ptr(), None)
        for b, r in zip((0, batch - 1), ref):
            ab, wb, z = a[b].double(), w[b].double() / f, v[b].double().T.contiguous()
            scale = np.max(np.abs(r))
            assert np.max(np.abs(wb.cpu().numpy() - r)) < 200 * n ** 0.5 * eps * scale
            assert float(torch.linalg.norm(ab @ z - z * wb[None, :])) / scale < 200 * n * eps
            assert float(torch.linalg.norm(z.T.contiguous() @ z - eye)) < 200 * n * eps
