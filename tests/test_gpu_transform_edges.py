"""The half-transform kernel at the edges of its blocks: one block of 16
orbitals and the first past it, the change from 16 to 32 rows per wave (64 ->
65), a last panel of one block of rows, uneven rounds of column blocks.

Bound: each quarter transformation is a sum of N products, |error| <= N eps
|U|^T |V| |U|... entry by entry; with an orthogonal U (row sums at most
sqrt(N)) that is 4 N eps N^2 max |V|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 47, 64, 65, 81, 97, 130])
def test_transform_edges(cuda, n):
    import torch
    from gammcor_amd import _lib
    g = torch.Generator(device=cuda)
    g.manual_seed(n)
    r = 4
    f = torch.randn(r, n, n, generator=g, device=cuda, dtype=torch.float64)
    f = f + f.transpose(1, 2)
    u = torch.linalg.qr(torch.randn(n, n, generator=g, device=cuda, dtype=torch.float64))[0].contiguous()   # U[no, ao]
    i, j = torch.tril_indices(n, n, device=cuda)

    def packed(x):
        c = x[:, i, j].contiguous()
        v = c.T.contiguous() @ c
        k, m = torch.tril_indices(c.shape[1], c.shape[1], device=cuda)
        return v[k, m].contiguous()

    tno = packed(f)
    top = float(tno.abs().max())
    ref = packed(torch.matmul(torch.matmul(u, f), u.T.contiguous()))
    ure = u.T.contiguous().reshape(-1)
    print(f"transform n={n}", flush=True)
    _lib.call("gmc_twono1_dev", tno.data_ptr(), ure.data_ptr(), n, tno.numel(), None)
    assert float((tno - ref).abs().max()) < 4 * n ** 3 * 2.2e-16 * max(top, float(ref.abs().max()))
