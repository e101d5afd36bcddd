"""The panels with word exchanges where a workgroup owns too many rows to keep
their panel columns in LDS (they are read back from memory instead): one, two and
four workgroups per problem, FP64 and FP32, and the deterministic mode
(bit-equal repeats).  The LDS of a workgroup with its panel columns, 32 of V and of
W', is (2 n + 65 rows + 2 rows' + 2148) elements, rows' = max(rows, 1024): beyond
160 KB at these sizes.

Bounds as in the eigensolver's other tests: computed values and vectors are
those of A + E, |E| <= c n eps |A|, c = 200 (eigenvalues c sqrt(n))."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,n,batch", [("f64", 700, 200), ("f64", 1000, 100), ("f64", 1400, 64), ("f32", 700, 200),
                                          ("f32", 1200, 100)])
def test_panel_columns_in_memory(cuda, prec, n, batch):
    import torch
    from gammcor_amd import _lib
    es, workgroups = (8, 256 // batch) if prec == "f64" else (4, 256 // batch)
    rows = 8 * -(-(-(-n // 8)) // workgroups)
    assert (2 * n + 65 * rows + 2 * max(rows, 1024) + 2148) * es > 160 * 1024
    dt, eps = (torch.float64, 2.2e-16) if prec == "f64" else (torch.float32, 1.2e-7)
    g = torch.Generator(device=cuda)
    g.manual_seed(n + batch)
    a = torch.randn(batch, n, n, generator=g, device=cuda, dtype=dt)
    a = (a + a.transpose(1, 2)).contiguous()
    print(f"panel columns in memory: {prec} n={n} batch={batch}", flush=True)

    def solve():
        v, w = a.clone(), torch.zeros(batch, n, device=cuda, dtype=dt)
        _lib.call("gmc_syevd_dev", 0 if prec == "f64" else 1, n, batch, v.data_ptr(), w.data_ptr(), None)
        return v, w

    v, w = solve()
    eye = torch.eye(n, device=cuda, dtype=torch.float64)
    for b in (0, batch // 2, batch - 1):
        ab, wb, z = a[b].double(), w[b].double(), v[b].double().T.contiguous()
        ref = np.linalg.eigvalsh(ab.cpu().numpy())
        scale = np.max(np.abs(ref))
        assert np.max(np.abs(wb.cpu().numpy() - ref)) < 200 * n ** 0.5 * eps * scale
        assert float(torch.linalg.norm(ab @ z - z * wb[None, :])) / scale < 200 * n * eps
        assert float(torch.linalg.norm(z.T.contiguous() @ z - eye)) < 200 * n * eps
    _lib.call("gmc_set_deterministic", 1)
    try:
        (v1, w1), (v2, w2) = solve(), solve()
    finally:
        _lib.call("gmc_set_deterministic", 0)
    assert torch.equal(w1, w2) and torch.equal(v1, v2)
