"""Which way the factor of |A+| goes at orders from 2048, as the library's own
report (GMC_OA_STATS) tells it, and the results on that way.

- N=150, NDimX=2236 (and 148, 2170), weakly coupled: A+ has few eigenvalues
  below zero, the Krylov basis converges and |A+| is factored: FP64, mixed, one
  alpha point per call and in the batching form with padded modes.  W(alpha)
  against numpy's eigensolves of the same A+-B, 1e-9 Eh in FP64 and 1e-6 mixed
  as everywhere in these tests.
- The stronger coupling (residual 1e-3 at the first Ritz problem, a basis limit
  of 992): the eigensolve takes over after that one, no second one is tried.
- Without integrals A+ is diagonal with a few dozen distinct values: the Krylov
  space is exhausted, goes on with rounding noise and breaks down before the basis
  of the first Ritz problem (832) is full: the eigensolve takes over there.
- With a NaN among the integrals the basis breaks down at once, the eigensolve
  takes over and no eigenvalue word is left as it was."""
import os
import re
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))

FACTORED = "abs_factor: |A| factored"
RITZ = re.compile(r"restricted step on a basis of (\d+)")
TAKEN_OVER = re.compile(r"abs_factor: (.*) in a basis of (\d+), the eigensolve takes over")


def _device_system(cuda, *cfg):
    import torch
    from gammcor_amd import host, synth, _lib
    s = synth.make_system(*cfg, with_integrals=False)
    ao = synth.ao_integrals_device(s.chol, cuda)
    ure = torch.from_numpy(np.asfortranarray(s.uaomo).ravel(order="F")).to(cuda)
    _lib.call("gmc_twono1_dev", ao.data_ptr(), ure.data_ptr(), s.nbasis, ao.numel(), None)
    d = host.DeviceSystem(ao, s.occ, s.xone, s.gamma_act, s.nbasis, s.ninact, s.nact, s.nele, device=cuda)
    return s, d


def _report(capfd, call):
    capfd.readouterr()
    r = call()
    err = capfd.readouterr().err
    print(err, flush=True)
    return r, err


def test_converged_basis_gives_the_factor(cuda, monkeypatch, capfd):
    import accas_oracle as O
    from gammcor_amd import host
    monkeypatch.setenv("GMC_OA_STATS", "1")
    s, d = _device_system(cuda, 150, 8, 8, 8, 450, 0.05, 3)
    _, d2 = _device_system(cuda, 148, 8, 7, 6, 444, 0.05, 4)
    print(f"factor route: NDimX {d.ndimx}, {d2.ndimx}", flush=True)
    assert d2.ndimx >= 2048 and d2.ndimx < d.ndimx
    alphas, weights = np.array([0.1, 0.9]), np.array([0.4, 0.6])

    def factored(call, calls):
        r, err = _report(capfd, call)
        assert err.count(FACTORED) == calls and not TAKEN_OVER.search(err)
        assert [int(m) for m in RITZ.findall(err)] == [832] * calls
        return r

    two = factored(lambda: host.ACECORR(d, alphas, weights, prec=host.GMC_FP64, return_eig=True), 1)
    one = factored(lambda: host.ACECORR(d, alphas, weights, prec=host.GMC_FP64, alpha_batch=1), 2)
    mix = factored(lambda: host.ACECORR(d, alphas, weights, prec=host.GMC_MIXED), 1)
    alone = factored(lambda: host.ACECORR(d2, alphas, weights, prec=host.GMC_FP64), 1)
    # one group of both systems (a cost per batch alone), d2 padded to d's order
    cost = (1.0, 0.0, 0.0, 0.0)
    pad = factored(lambda: host.ACECORR_BATCH([d2, d], alphas, weights, prec=host.GMC_FP64, cost=cost), 1)
    assert np.max(np.abs(pad["walpha"][0] - alone["walpha"])) < 1e-9
    assert np.max(np.abs(pad["walpha"][1] - two["walpha"])) < 1e-9
    tw = d.twono.cpu().numpy()
    indn, igem = host.ACCAS_pairs(s.occ, s.nele), host.geminals(s.nbasis, s.ninact, s.nact)
    rdm = host.pack_rdm2act(s.gamma_act)
    k, al = 1, 0.9
    ap, am, _, ci = host.AB_CAS(tw, None, s.occ, s.xone, indn, s.nbasis, s.ninact, s.nact, igem, rdm, al)
    y, eig, nneg = O.erpasymm1(ap, am)
    w, _ = O.aceneerpa(y, eig, tw, s.occ, ci, igem, indn)
    assert nneg > 0
    assert two["nneg"][k] == nneg and one["nneg"][k] == nneg and mix["nneg"][k] == nneg
    assert abs(two["walpha"][k] - w) < 1e-9 and abs(one["walpha"][k] - w) < 1e-9
    assert abs(mix["walpha"][k] - w) < 1e-6
    got = two["eig"][k].cpu().numpy()
    keep = eig > 1e-3
    assert np.max(np.abs(got[keep] - eig[keep])) < 1e-10 * np.max(eig)


def test_hopeless_basis_is_left_after_the_first_ritz_problem(cuda, monkeypatch, capfd):
    from gammcor_amd import host
    monkeypatch.setenv("GMC_OA_STATS", "1")
    _, d = _device_system(cuda, 150, 8, 8, 8, 450, 0.1, 3)
    a, w = np.array([0.6]), np.array([1.0])
    res = {}
    for prec in (host.GMC_FP64, host.GMC_MIXED):
        res[prec], err = _report(capfd, lambda: host.ACECORR(d, a, w, prec=prec))
        assert RITZ.findall(err)[:1] == ["832"] and TAKEN_OVER.findall(err) == [("no convergence", "832")]
        assert FACTORED not in err
    assert abs(res[host.GMC_FP64]["ecorr"] - res[host.GMC_MIXED]["ecorr"]) < 1e-6


def test_exhausted_space_is_noticed_before_the_ritz_problem(cuda, monkeypatch, capfd):
    import torch
    from gammcor_amd import host
    monkeypatch.setenv("GMC_OA_STATS", "1")
    n, ni, na = 140, 10, 8
    t = n * (n + 1) // 2
    tw = torch.zeros(t * (t + 1) // 2, dtype=torch.float64, device=cuda)
    eps = np.concatenate([np.full(ni, -10.0), np.linspace(-1.0, 1.0, na), np.full(n - ni - na, 10.0)])
    occ = np.concatenate([np.ones(ni), np.linspace(0.93, 0.07, na), np.zeros(n - ni - na)])
    i, j = np.tril_indices(n)
    d = host.DeviceSystem(tw, occ, np.diag(eps)[i, j], np.zeros((na,) * 4), n, ni, na, ni + na // 2, device=cuda)
    assert d.ndimx >= 2048
    r, err = _report(capfd, lambda: host.ACECORR(d, np.array([0.5]), np.array([1.0]), prec=host.GMC_FP64))
    (why, basis), = TAKEN_OVER.findall(err)
    assert why == "breakdown" and int(basis) < 832 and not RITZ.search(err)
    assert r["nneg"][0] == 0 and abs(r["ecorr"]) < 1e-12


def test_nan_among_the_integrals_breaks_down_and_ends(cuda, monkeypatch, capfd):
    import torch
    from gammcor_amd import host
    monkeypatch.setenv("GMC_OA_STATS", "1")
    _, d = _device_system(cuda, 150, 8, 8, 8, 450, 0.05, 3)
    # (p a | q b) with p, q inactive and a, b virtual: one element of A+ and its mirror
    pair = lambda x, y: max(x, y) * (max(x, y) + 1) // 2 + min(x, y)
    d.twono[pair(pair(1, 40), pair(3, 90))] = float("nan")
    r, err = _report(capfd, lambda: host.ACECORR(d, np.array([0.5]), np.array([1.0]), prec=host.GMC_FP64, return_eig=True))
    assert TAKEN_OVER.findall(err) == [("breakdown", "128")]
    assert bool(torch.isnan(r["eig"]).any())
