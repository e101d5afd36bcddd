"""The panels whose exchanges travel in epoch-tagged words, over several panels
of a reduction: one to many workgroups per problem, row counts around the
rows-per-thread steps (1024, 2048), padded orders, FP64 and FP32, and the
deterministic mode (bit-equal repeats).

Bounds as for any backward-stable solver of this kind: the computed
eigenvalues and vectors are those of A + E, |E| <= c n eps |A|, with the
same c = 200 that the eigensolver's other tests use (eigenvalues c sqrt(n))."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,batch", [(400, 128), (700, 64), (701, 33), (860, 24), (1024, 24), (1028, 12), (1359, 5),
                                     (2052, 3), (2400, 1)])
def test_panels_with_word_exchanges(cuda, prec, n, batch):
    import torch
    from gammcor_amd import _lib
    dt = torch.float64 if prec == "f64" else torch.float32
    g = torch.Generator(device=cuda)
    g.manual_seed(1000 * n + batch)
    a = torch.randn(batch, n, n, generator=g, device=cuda, dtype=torch.float64)
    a = (a + a.transpose(1, 2)).contiguous().to(dt)
    print(f"panel exchange {prec} n={n} batch={batch}", flush=True)

    def solve():
        v = a.clone()
        w = torch.zeros(batch, n, device=cuda, dtype=dt)
        _lib.call("gmc_syevd_dev", 0 if prec == "f64" else 1, n, batch, v.data_ptr(), w.data_ptr(), None)
        return v, w

    v, w = solve()
    eps = 2.2e-16 if prec == "f64" else 1.2e-7
    for b in (0, batch - 1):
        ref = np.linalg.eigvalsh(a[b].double().cpu().numpy())
        scale = max(1.0, np.max(np.abs(ref)))
        wb, z = w[b].double(), v[b].double().T.contiguous()          # columns: eigenvectors
        ab = a[b].double()
        assert np.max(np.abs(wb.cpu().numpy() - ref)) < 200 * n ** 0.5 * eps * scale
        assert float(torch.linalg.norm(ab @ z - z * wb[None, :])) / scale < 200 * n * eps
        assert float(torch.linalg.norm(z.T.contiguous() @ z - torch.eye(n, device=cuda, dtype=torch.float64))) < \
            200 * n * eps
    _lib.call("gmc_set_deterministic", 1)
    try:
        (v1, w1), (v2, w2) = solve(), solve()
    finally:
        _lib.call("gmc_set_deterministic", 0)
    assert torch.equal(w1, w2) and torch.equal(v1, v2)
