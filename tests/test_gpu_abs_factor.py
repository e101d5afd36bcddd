"""The Cholesky factor of |A+| from the eigenpairs below zero alone, which
orders from 2048 up take in place of A+'s eigensolve.

- On a system whose A+ is indefinite at every alpha point (N=144, NDimX about
  2 150, odd), FP64 and mixed, one alpha point per call and several: W(alpha),
  the omegas and the count of negative eigenvalues against numpy's eigensolves
  of the same A+-B (the host AB_CAS gives the matrices).  The integrand is a
  sum over n^2 products of FP64 values: 1e-9 Eh as everywhere in these tests,
  the mixed path 1e-6.
- Without integrals A+ is diagonal with a few dozen distinct values, so the
  Krylov space is exhausted within a few blocks and the eigensolve must take
  over: omega = |h_pp - h_qq| in closed form, to 1e-10."""
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))


def _device_system(cuda):
    import torch
    from gammcor_amd import host, synth, _lib
    s = synth.make_system(144, 11, 7, 6, 432, 0.1, 21, with_integrals=False)
    ao = synth.ao_integrals_device(s.chol, cuda)
    ure = torch.from_numpy(np.asfortranarray(s.uaomo).ravel(order="F")).to(cuda)
    _lib.call("gmc_twono1_dev", ao.data_ptr(), ure.data_ptr(), s.nbasis, ao.numel(), None)
    d = host.DeviceSystem(ao, s.occ, s.xone, s.gamma_act, s.nbasis, s.ninact, s.nact, s.nele, device=cuda)
    return s, d


def test_factor_route_matches_numpy(cuda):
    import accas_oracle as O
    from gammcor_amd import host
    s, d = _device_system(cuda)
    print(f"abs factor: NDimX {d.ndimx}", flush=True)
    assert d.ndimx >= 2048
    alphas, weights = np.array([0.1, 0.6]), np.array([0.4, 0.6])
    r = host.ACECORR(d, alphas, weights, prec=host.GMC_FP64, return_eig=True)
    one = host.ACECORR(d, alphas, weights, prec=host.GMC_FP64, alpha_batch=1)
    mix = host.ACECORR(d, alphas, weights, prec=host.GMC_MIXED)
    tw = d.twono.cpu().numpy()
    indn, igem = host.ACCAS_pairs(s.occ, s.nele), host.geminals(s.nbasis, s.ninact, s.nact)
    rdm = host.pack_rdm2act(s.gamma_act)
    for k, al in enumerate(alphas):
        ap, am, _, ci = host.AB_CAS(tw, None, s.occ, s.xone, indn, s.nbasis, s.ninact, s.nact, igem, rdm, float(al))
        y, eig, nneg = O.erpasymm1(ap, am)
        w, _ = O.aceneerpa(y, eig, tw, s.occ, ci, igem, indn)
        assert nneg > 0
        assert r["nneg"][k] == nneg and one["nneg"][k] == nneg and mix["nneg"][k] == nneg
        assert abs(r["walpha"][k] - w) < 1e-9 and abs(one["walpha"][k] - w) < 1e-9
        assert abs(mix["walpha"][k] - w) < 1e-6
        got = r["eig"][k].cpu().numpy()
        keep = eig > 1e-3
        assert np.max(np.abs(got[keep] - eig[keep])) < 1e-10 * np.max(eig)


def test_exhausted_krylov_space_takes_the_eigensolve(cuda):
    import torch
    from gammcor_amd import host
    n, ni, na = 140, 10, 8
    t = n * (n + 1) // 2
    tw = torch.zeros(t * (t + 1) // 2, dtype=torch.float64, device=cuda)
    eps = np.concatenate([np.full(ni, -10.0), np.linspace(-1.0, 1.0, na), np.full(n - ni - na, 10.0)])
    occ = np.concatenate([np.ones(ni), np.linspace(0.93, 0.07, na), np.zeros(n - ni - na)])
    h = np.diag(eps)
    i, j = np.tril_indices(n)
    d = host.DeviceSystem(tw, occ, h[i, j], np.zeros((na,) * 4), n, ni, na, ni + na // 2, device=cuda)
    assert d.ndimx >= 2048
    r = host.ACECORR(d, np.array([0.5]), np.array([1.0]), prec=host.GMC_FP64, return_eig=True)
    p, q = d.indn_host[:, 0] - 1, d.indn_host[:, 1] - 1
    want = np.sort(np.abs(eps[p] - eps[q]))
    assert np.max(np.abs(np.sort(r["eig"][0].cpu().numpy()) - want)) < 1e-10
    assert r["nneg"][0] == 0 and abs(r["ecorr"]) < 1e-12
