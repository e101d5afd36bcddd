"""Workloads of the AC-CAS library and their plain 64-bit values.

Each case is a dict of plain values.  ``prepare`` makes what a user's program
holds before the call (integrals, orbitals, RDMs on the GPU, or host arrays
for the Fortran-style drop-ins), ``run`` is one pass through the public entry
points of ``gammcor_amd.host``, ``work`` the bytes and operations the path
cannot do without, ``exact`` the same outputs from torch in 64 bits.

Inputs are those of ``gammcor_amd.synth``: AO integrals from Gaussian
Cholesky factors, random orthogonal orbitals, the exact RDMs of a CI vector
dominated by one determinant, and an h that puts the inactive, active and
virtual orbitals at separated energies as a CASSCF reference does.
"""
import math

import numpy as np
import torch

from gammcor_amd import _lib, host, synth


def listed():
    return [
        # The AO->NO transform alone: the first step of every in-core run.
        dict(name="transform_n48", kind="transform", n=48),
        dict(name="transform_n200", kind="transform", n=200),
        # AC-CAS of a minimal-basis diatomic: launches and latency.
        dict(name="accas_n16", kind="accas", n=16, ni=3, na=4, nalpha=4, prec="fp64"),
        # The small named system (n48_cas44), all alpha points in one call.
        dict(name="accas_n48", kind="accas", n=48, ni=6, na=4, nalpha=8, prec="fp64"),
        # The mid-size named system (n160_cas88) in plain double precision.
        dict(name="accas_n160", kind="accas", n=160, ni=10, na=8, nalpha=8, prec="fp64"),
        # The headline system (n240_cas88): a whole solve as bench.py runs it,
        # transform, assembly and 16 alpha points, mixed precision.
        dict(name="solve_mixed_n240", kind="solve", n=240, ni=12, na=8, nalpha=16, prec="mixed"),
        # One alpha point per call, as the reference's own ACEInteg loop asks
        # for it, with odd sizes.
        dict(name="alpha_n101", kind="accas", n=101, ni=8, na=6, nalpha=1, prec="fp64"),
        # The FOFO form: integral classes straight from the AO integrals, the
        # reference's five-point rule.
        dict(name="fofo_n121", kind="fofo", n=121, ni=6, na=6, nalpha=5, prec="fp64"),
        # The linearised correction, the cheap production variant.
        dict(name="ac0_n160", kind="ac0", n=160, ni=10, na=8),
        # Many small systems at once (points of a potential curve, fragments).
        dict(name="batch_8", kind="batch", sizes="34,41,48,53,60,67,72,80", nalpha=8),
        # SAPT dispersion of a dimer: two monomer responses and the energy.
        dict(name="sapt_n72", kind="sapt", n=72, ni=5, na=4),
        # The Fortran program's flow on host arrays: TwoNO1, then ACEInteg for
        # each of five alpha points.
        dict(name="dropin_n64", kind="dropin", n=64, ni=5, na=4, nalpha=5),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["transform", "accas", "accas", "alpha", "mixed", "fofo", "ac0", "batch", "sapt", "dropin"])
    na = rng.choice([2, 4, 6, 8])
    if kind == "transform":
        return dict(kind="transform", n=_logint(rng, 12, 220))
    if kind in ("accas", "alpha", "fofo"):
        n = _logint(rng, 20, 170)
        c = dict(kind="fofo" if kind == "fofo" else "accas", n=n, ni=max(1, int(n * rng.uniform(0.04, 0.09))), na=na,
                 nalpha=1 if kind == "alpha" else rng.randint(2, 12), prec="fp64")
        return c
    if kind == "mixed":
        n = _logint(rng, 100, 230)
        return dict(kind="solve", n=n, ni=max(2, int(n * 0.05)), na=rng.choice([6, 8]), nalpha=rng.randint(6, 16),
                    prec="mixed")
    if kind == "ac0":
        n = _logint(rng, 24, 200)
        return dict(kind="ac0", n=n, ni=max(1, n // 16), na=na)
    if kind == "batch":
        sizes = sorted(_logint(rng, 24, 110) for _ in range(rng.randint(3, 12)))
        return dict(kind="batch", sizes=",".join(map(str, sizes)), nalpha=rng.randint(4, 12))
    if kind == "sapt":
        n = _logint(rng, 24, 110)
        return dict(kind="sapt", n=n, ni=max(1, n // 14), na=rng.choice([4, 6]))
    n = _logint(rng, 20, 100)
    return dict(kind="dropin", n=n, ni=max(1, n // 13), na=rng.choice([4, 6]), nalpha=rng.randint(3, 6))


# ---------------------------------------------------------------- inputs
def _device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _normal(shape, seed, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, dtype=torch.float64, device=dev)


def _tril(n, dev):
    return torch.tril_indices(n, n, device=dev)


def _factors(n, sigma, seed, dev):
    """Symmetric Cholesky factors L_P (rank 3 n) of the AO integrals."""
    i, j = _tril(n, dev)
    v = sigma * _normal((3 * n, len(i)), seed, dev)
    full = torch.empty(3 * n, n, n, dtype=torch.float64, device=dev)
    full[:, i, j] = v
    full[:, j, i] = v
    return full


def _packed(fac):
    """The 8-fold packed (ij|kl) = sum_P F_P,ij F_P,kl, ij >= kl."""
    n, dev = fac.shape[1], fac.device
    i, j = _tril(n, dev)
    c = fac[:, i, j].contiguous()
    t = c.shape[1]
    out = torch.empty(t * (t + 1) // 2, dtype=torch.float64, device=dev)
    cols = torch.arange(t, device=dev)
    for r0 in range(0, t, 1024):
        r1 = min(t, r0 + 1024)
        block = c[:, r0:r1].T @ c[:, :r1]
        out[r0 * (r0 + 1) // 2: r1 * (r1 + 1) // 2] = block[cols[None, :r1] <= cols[r0:r1, None]]
    return out


def _orbitals(n, seed, dev):
    """U[no, ao]: the orthogonal factor of a Gaussian matrix."""
    q, _ = np.linalg.qr(np.random.default_rng(seed).standard_normal((n, n)))
    return torch.from_numpy(np.ascontiguousarray(q.T)).to(dev)


def _system(n, ni, na, seed, dev, ao_fac=None):
    """One system as a dict of tensors and arrays (ao: factors in the AO
    basis, b: in the NO basis)."""
    sigma = 0.1 if n < 150 else 0.05
    fac = _factors(n, sigma, seed, dev) if ao_fac is None else ao_fac
    u = _orbitals(n, seed + 1, dev)
    b = torch.matmul(torch.matmul(u, fac), u.T.contiguous())
    gamma, d = synth.cas_rdms(na, na, seed + 2)
    w, v = np.linalg.eigh(gamma)
    order = np.argsort(-w, kind="stable")
    w, v = w[order], v[:, order]
    g2 = 0.5 * np.einsum("pqrs,pa,qb,rc,sd->abcd", d, v, v, v, v, optimize=True)
    g2 = 0.5 * np.round(g2 + g2.transpose(2, 3, 0, 1), 12)
    occ = np.zeros(n)
    occ[:ni] = 1.0
    occ[ni:ni + na] = np.abs(w) / 2.0
    # mean field of the NO densities: h is designed so that h + G is diagonal
    # up to noise
    no = ni + na
    f = torch.from_numpy(occ[:no]).to(dev)
    bd = torch.einsum("ptt,t->p", b[:, :no, :no], f)
    bo = (b[:, :, :no] * f.sqrt()).permute(1, 0, 2).reshape(n, -1)
    gmf = 2.0 * torch.einsum("pij,p->ij", b, bd) - bo @ bo.T
    rng = np.random.default_rng(seed + 3)
    h = rng.standard_normal((n, n)) * synth.H_SIGMA
    h = np.tril(h) + np.tril(h, -1).T
    h += np.diag(synth.orbital_energies(ni, na, n - ni - na)) - gmf.cpu().numpy()
    h = 0.5 * (h + h.T)
    i, j = np.tril_indices(n)
    return dict(n=n, ni=ni, na=na, nele=ni + na // 2, fac=fac, u=u, b=b, occ=occ, h=h, xone=h[i, j], g2=g2)


def _ure(s):
    return s["u"].T.contiguous().reshape(-1)       # URe(NO, AO), column-major


def _dsys(s, twono):
    return host.DeviceSystem(twono, s["occ"], s["xone"], s["g2"], s["n"], s["ni"], s["na"], s["nele"])


def _grid(nalpha):
    return host.GauLeg(0.0, 1.0, nalpha)


_PREC = dict(fp64=host.GMC_FP64, mixed=host.GMC_MIXED)


def _inputs(case, seed, dev):
    k = case["kind"]
    if k == "transform":
        return dict(fac=_factors(case["n"], 0.1 if case["n"] < 150 else 0.05, seed * 10, dev),
                    u=_orbitals(case["n"], seed * 10 + 1, dev))
    if k == "batch":
        return [_system(n, max(1, n // 12), 4 if i % 2 == 0 else 6, seed * 1000 + 10 * i, dev)
                for i, n in enumerate(int(x) for x in case["sizes"].split(","))]
    s = _system(case["n"], case["ni"], case["na"], seed * 10, dev)
    if k == "sapt":
        return s, _system(case["n"], case["ni"], case["na"], seed * 10 + 5, dev, ao_fac=s["fac"])
    return s


def prepare(case, seed):
    dev = _device()
    k = case["kind"]
    inp = _inputs(case, seed, dev)
    if k == "transform":
        ao = _packed(inp["fac"])
        return dict(kind=k, n=case["n"], ao=ao, work=torch.empty_like(ao), ure=_ure(inp))
    if k == "batch":
        a, w = _grid(case["nalpha"])
        return dict(kind=k, systems=[_dsys(s, _packed(s["b"])) for s in inp], a=a, w=w)
    if k == "sapt":
        da, db = (_dsys(s, _packed(s["b"])) for s in inp)
        sel = lambda s, d: s["b"][:, d.indn_host[:, 0] - 1, d.indn_host[:, 1] - 1]
        vab = sel(inp[1], db).T.contiguous() @ sel(inp[0], da)       # row-major (B, A): column-major (A, B)
        return dict(kind=k, da=da, db=db, vab=vab.reshape(-1))
    s = inp
    if k == "dropin":
        ao = _packed(s["fac"]).cpu().numpy()
        a, w = _grid(case["nalpha"])
        return dict(kind=k, n=s["n"], ni=s["ni"], na=s["na"], ao=ao, work=np.empty_like(ao),
                    u=np.asfortranarray(s["u"].cpu().numpy()), occ=s["occ"], xone=s["xone"],
                    indn=host.ACCAS_pairs(s["occ"], s["nele"]), igem=host.geminals(s["n"], s["ni"], s["na"]),
                    rdm=host.pack_rdm2act(s["g2"]), a=a, w=w)
    if k == "ac0":
        return dict(kind=k, d=_dsys(s, _packed(s["b"])))
    a, w = _grid(case["nalpha"])
    st = dict(kind=k, a=a, w=w, prec=_PREC[case["prec"]])
    if k == "accas":
        st["d"] = _dsys(s, _packed(s["b"]))
    elif k == "fofo":
        st.update(ao=_packed(s["fac"]), ure=_ure(s), d=_dsys(s, torch.zeros(1, dtype=torch.float64, device=dev)))
    else:
        st["ao"] = _packed(s["fac"])
        st["work"] = torch.empty_like(st["ao"])
        st.update(ure=_ure(s), d=_dsys(s, st["work"]))
    return st


# ---------------------------------------------------------------- one pass
def run(st):
    k = st["kind"]
    if k == "transform":
        st["work"].copy_(st["ao"])
        return host.TwoNO1(st["work"], st["ure"], st["n"])
    if k == "accas":
        return host.ACECORR(st["d"], st["a"], st["w"], prec=st["prec"], return_eig=True)
    if k == "solve":
        st["work"].copy_(st["ao"])
        host.TwoNO1(st["work"], st["ure"], st["d"].nbasis)
        return host.ACECORR(st["d"], st["a"], st["w"], prec=st["prec"])
    if k == "fofo":
        return host.ACECORR_FOFO(st["ao"], st["ure"], st["d"], st["a"], st["w"], prec=st["prec"])
    if k == "ac0":
        return host.AC0CAS(st["d"])
    if k == "batch":
        return host.ACECORR_BATCH(st["systems"], st["a"], st["w"], prec=host.GMC_FP64)
    if k == "sapt":
        # the response vectors' signs are free; the energies do not depend on them
        ra, rb = host.SAPT_RESPONSE(st["da"]), host.SAPT_RESPONSE(st["db"])
        return dict(e2disp=host.E2DISP(ra, rb, st["vab"]), eig_a=ra["eig"], eig_b=rb["eig"])
    np.copyto(st["work"], st["ao"])
    _lib.call("gmc_forget_resident")
    tno = host.TwoNO1(st["work"], st["u"], st["n"])
    wa = []
    for al in st["a"]:
        r = host.ACEInteg(tno, None, st["occ"], st["xone"], st["indn"], st["n"], st["ni"], st["na"], st["igem"],
                          st["rdm"], al)
        wa.append(r["ecorr"])
    return dict(tno=tno, walpha=np.array(wa), ecorr=float(np.dot(st["w"], wa)), egone=r["egone"])


# ---------------------------------------------------------------- work
def _npair(n, ni, na):
    nv = n - ni - na
    return ni * na + ni * nv + na * (na - 1) // 2 + na * nv


def _w_transform(n):
    # both halves: U M for every pair column, then the lower half of (U M) U^T
    t = n * (n + 1) // 2
    return dict(bytes=2 * 8 * t * (t + 1) // 2, flops=6.0 * n ** 3 * t)


def _w_erpa(n, nalpha):
    # per alpha: a factor of A+ (n^3/3), M (3 n^3), one symmetric eigenproblem
    # with vectors (4/3 n^3 reduction, 2 n^3 back-transformation), Y (n^3 with a
    # triangular factor), the lower half of Y Y^T (n^3)
    return nalpha * (1 / 3 + 3 + 4 / 3 + 2 + 1 + 1) * n ** 3


def work(case):
    k = case["kind"]
    if k == "transform":
        return _w_transform(case["n"])
    packed = lambda n: 8 * (n * (n + 1) // 2) * (n * (n + 1) // 2 + 1) // 2
    if k == "batch":
        b = f = 0
        for i, n in enumerate(int(x) for x in case["sizes"].split(",")):
            b += packed(n)
            f += _w_erpa(_npair(n, max(1, n // 12), 4 if i % 2 == 0 else 6), case["nalpha"])
        return dict(bytes=b, flops=f)
    n, ni, na = case["n"], case["ni"], case["na"]
    nd = _npair(n, ni, na)
    if k == "accas":
        return dict(bytes=packed(n) + 8 * nd * case["nalpha"], flops=_w_erpa(nd, case["nalpha"]))
    if k in ("solve", "dropin"):
        t = _w_transform(n)
        return dict(bytes=t["bytes"] + packed(n), flops=t["flops"] + _w_erpa(nd, case["nalpha"]))
    if k == "fofo":
        no, t = ni + na, n * (n + 1) // 2
        # (fo|c) and (kl|c) per AO pair column, then U M U_O^T and U M U^T per row
        half = 2.0 * t * (n * n * no * 2 + no * no * n) + 2.0 * n * no * (n * n * no + n * no * no) + \
            2.0 * no * no * 2 * n ** 3
        return dict(bytes=packed(n), flops=half + _w_erpa(nd, case["nalpha"]))
    if k == "ac0":
        # the alpha=0 blocks are small; X^T A' X, Y^T A' Y and Y D Y^T remain
        return dict(bytes=packed(n), flops=(3 + 3 + 3) * float(nd) ** 3)
    return dict(bytes=2 * packed(n) + 8 * nd * nd, flops=2 * (1 / 3 + 3 + 4 / 3 + 2 + 1 + 2) * float(nd) ** 3 +
                4.0 * nd ** 3)


# ---------------------------------------------------------------- 64-bit values
def _ref_integrals(s):
    """(pq|tu) and (pt|qu) with t, u occupied, and the pair list."""
    b, n, no = s["b"], s["n"], s["ni"] + s["na"]
    r = b.shape[0]
    jj = (b.reshape(r, -1).T @ b[:, :no, :no].reshape(r, -1)).reshape(n, n, no, no)
    half = b[:, :, :no].reshape(r, -1)
    kk = (half.T @ half).reshape(n, no, n, no)     # (p t|q u) at [p, t, q, u]
    kind = np.where(s["occ"] == 0.0, 2, np.where(s["occ"] == 1.0, 0, 1))
    pairs = [(p, q) for p in range(n) for q in range(p)
             if not (kind[p] == kind[q] and kind[p] != 1)
             and not (kind[p] == kind[q] == 1 and abs(s["occ"][p] - s["occ"][q]) / s["occ"][p] < 1e-8)]
    gem = torch.tensor([0] * s["ni"] + [1] * s["na"] + [2] * (n - no), device=b.device)
    return jj, kk, np.array(pairs), gem


def _ref_gamma(s):
    """The two-particle density over all occupied orbitals: the active block
    and its antisymmetrised products with the inactive occupations."""
    ni, na = s["ni"], s["na"]
    no = ni + na
    f = torch.from_numpy(s["occ"][:no])
    e = torch.eye(no, dtype=torch.float64)
    g = 2.0 * torch.einsum("p,q,pr,qs->pqrs", f, f, e, e) - torch.einsum("p,q,ps,qr->pqrs", f, f, e, e)
    g[ni:, ni:, ni:, ni:] = torch.from_numpy(s["g2"])
    return g.to(s["b"].device)


def _ref_ab(s, ints, gam, alpha):
    """A+B and A-B of the alpha-scaled Hamiltonian over the pair list: the
    expectation value of the double commutator with every two-electron term
    that joins different geminals scaled by alpha."""
    jj, kk, pairs, gem = ints
    dev = jj.device
    n, no = s["n"], s["ni"] + s["na"]
    f = torch.from_numpy(s["occ"]).to(dev)
    h = torch.from_numpy(s["h"]).to(dev)
    same = gem[:, None] == gem[None, :]
    # one-electron part: coupling to other geminals' mean field enters as 1 - alpha
    out = torch.zeros_like(h)
    for g in range(3):
        w = torch.where(gem[:no] != g, f[:no], torch.zeros_like(f[:no]))
        m = gem == g
        mf = 2.0 * torch.einsum("ijtt,t->ij", jj, w) - torch.einsum("itjt,t->ij", kk, w)
        out[m] = torch.where(same[m], mf[m], out[m])
    h = torch.where(same, h + (1.0 - alpha) * out, alpha * h)
    fac = torch.where(same[:, :, None, None] & same[:no, :no][None, None] & same[:, None, :no, None],
                      torch.ones((), dtype=torch.float64, device=dev), torch.full((), alpha, dtype=torch.float64, device=dev))
    fj = fac * jj                                          # [p, q, t, u]
    fk = fac.permute(0, 2, 1, 3) * kk                      # [p, t, q, u]
    x1 = torch.einsum("sqtu,purt->sqpr", fj, gam) + torch.einsum("suqt,putr->sqpr", fk, gam)
    x5 = torch.einsum("ptsu,tuqr->psqr", fk, gam)
    wm = torch.zeros(n, n, dtype=torch.float64, device=dev)
    ju = fj[:, :no]                                        # (p u|t w) at [p, u, t, w]
    wm[:, :no] = torch.einsum("putw,wutr->pr", ju, gam) + torch.einsum("pwtu,wurt->pr", ju, gam)
    r = torch.from_numpy(pairs[:, 0]).to(dev)[:, None]
    sx = torch.from_numpy(pairs[:, 1]).to(dev)[:, None]

    def at(x, a, b, c, d):     # x[a, b, c, d], zero where c or d is virtual
        ok = (c < no) & (d < no)
        return torch.where(ok, x[a, b, c.clamp(max=no - 1), d.clamp(max=no - 1)], torch.zeros((), dtype=torch.float64, device=dev))

    def element(p, q):
        dpr, dsq = (p == r).double(), (sx == q).double()
        return (dpr * ((f[p] - f[sx]) * h[q, sx] - 0.5 * wm[q, sx]) + dsq * ((f[q] - f[r]) * h[p, r] - 0.5 * wm[p, r]) +
                at(x1, sx, q, p, r) + at(x1, p, r, sx, q) - at(x5, p, sx, q, r) - at(x5, r, q, sx, p))

    e1, e2 = element(r.T, sx.T), element(sx.T, r.T)
    c = f.sqrt() * torch.where(f < 0.5, -1.0, 1.0)
    cp, cm = c[r] + c[sx], c[r] - c[sx]
    return (e1 + e2) / cp / cp.T, (e1 - e2) / cm / cm.T


def _ref_ecas(s, ints, gam):
    no = s["ni"] + s["na"]
    jo = ints[0][:no, :no]
    return float(2.0 * np.sum(s["occ"] * np.diag(s["h"]))) + float(torch.einsum("pqrs,prqs->", gam, jo))


def _ref_erpa(ap, am):
    """Y, X and omega (omega^2 where that is at most 1e-6) of the symmetric
    ERPA problem, and the count of negative eigenvalues of A+."""
    ap, am = 0.5 * (ap + ap.T).cpu(), 0.5 * (am + am.T).cpu()
    lam, v = torch.linalg.eigh(ap)
    sq = (v * lam.abs().sqrt()) @ v.T
    m = sq @ (am @ sq)
    om2, z = torch.linalg.eigh(0.5 * (m + m.T))
    pos = om2 > 1e-6
    om = torch.where(pos, om2.clamp(min=1e-300).sqrt(), om2)
    y = torch.where(pos, (sq @ z) / (2.0 * om.abs()).sqrt(), torch.zeros_like(z))
    x = torch.where(pos, (am @ y) / om, torch.zeros_like(z))
    return y, x, om, int((lam < 0).sum())


def _ref_weights(s, ints):
    """(pr|qs) C-weighted over the pair list, zero within one geminal."""
    _, _, pairs, gem = ints
    b = s["b"]
    p, q = (torch.from_numpy(pairs[:, i]).to(b.device) for i in (0, 1))
    bp = b[:, p, q]
    f = torch.from_numpy(s["occ"]).to(b.device)
    c = f.sqrt() * torch.where(f < 0.5, -1.0, 1.0)
    own = gem[p] == gem[q]
    one = own[:, None] & own[None, :] & (gem[p][:, None] == gem[p][None, :])
    g = torch.where(one, torch.zeros((), dtype=torch.float64, device=b.device), bp.T @ bp)
    diag = (g.diagonal() * (f[p] * (1 - f[q]) + f[q] * (1 - f[p]))).sum()
    return (g * (c[p] + c[q])[:, None] * (c[p] + c[q])[None, :]).cpu(), float(diag)


def _ref_accas(s, nalpha):
    ints, gam = _ref_integrals(s), _ref_gamma(s)
    gw, diag = _ref_weights(s, ints)
    x, w = np.polynomial.legendre.leggauss(nalpha)
    wa, eig, nneg = [], [], []
    for al in 0.5 * (x + 1.0):
        y, _, om, neg = _ref_erpa(*_ref_ab(s, ints, gam, float(al)))
        k = y[:, (om > 1e-3) & (om < 1e8)]
        wa.append(2.0 * float((gw * (k @ k.T)).sum()) - diag)
        eig.append(om)
        nneg.append(neg)
    wa = np.array(wa)
    return dict(ecorr=float(np.dot(0.5 * w, wa)), walpha=wa, ecasscf=_ref_ecas(s, ints, gam),
                nneg=np.array(nneg, dtype=np.int32), eig=torch.stack(eig))


def _ref_ac0(s):
    ints, gam = _ref_integrals(s), _ref_gamma(s)
    pairs, ni, no = ints[2], s["ni"], s["ni"] + s["na"]
    (p0, m0), (p1, m1) = (_ref_ab(s, ints, gam, al) for al in (0.0, 1.0))
    index = {(int(a), int(b)): i for i, (a, b) in enumerate(pairs)}
    act, virt = range(ni, no), range(no, s["n"])
    blocks = [[index[(p, q)] for q in act for p in act if (p, q) in index]]
    blocks += [[index[(p, q)] for p in act] for q in range(ni)] + [[index[(p, q)] for q in act] for p in virt]
    single = [index[(p, q)] for p in virt for q in range(ni)]
    order = [i for b in blocks for i in b] + single
    pos = np.empty(len(order), dtype=np.int64)
    pos[order] = np.arange(len(order))
    low = torch.from_numpy(pos[:, None] >= pos[None, :]).to(p0.device)
    tri = lambda a: torch.where(low, a, a.T)            # the triangle at or below the diagonal in block order
    ap, am = tri(p0).cpu(), tri(m0).cpu()
    n = len(order)
    y, x, om = torch.zeros(n, n, dtype=torch.float64), torch.zeros(n, n, dtype=torch.float64), torch.zeros(n, dtype=torch.float64)
    for b in blocks:
        if b:
            i = torch.tensor(b)
            yb, xb, ob, _ = _ref_erpa(ap[i][:, i], am[i][:, i])
            y[i[:, None], i], x[i[:, None], i], om[i] = yb, xb, ob
    i = torch.tensor(single)
    y[i, i] = x[i, i] = math.sqrt(0.5)
    om[i] = ap[i, i]
    dev = p0.device
    y, x, om = y.to(dev), x.to(dev), om.to(dev)
    d = 2.0 * (x.T.contiguous() @ (tri(p1 - p0) @ x) - y.T.contiguous() @ (tri(m1 - m0) @ y)) / (om[:, None] + om[None, :])
    d = torch.where((om != 0)[:, None] & (om != 0)[None, :], d, torch.zeros_like(d))
    gw, _ = _ref_weights(s, ints)
    pm = y @ d @ y.T.contiguous()
    return dict(ecorr=float((gw.to(dev) * pm).sum()), ecasscf=_ref_ecas(s, ints, gam))


def _ref_sapt(pair):
    resp = []
    for s in pair:
        ints, gam = _ref_integrals(s), _ref_gamma(s)
        y, x, om, _ = _ref_erpa(*_ref_ab(s, ints, gam, 1.0))
        p, q = (torch.from_numpy(ints[2][:, i]) for i in (0, 1))
        f = torch.from_numpy(s["occ"])
        c = f.sqrt() * torch.where(f < 0.5, -1.0, 1.0)
        cm, cp = (c[p] - c[q])[:, None], (c[p] + c[q])[:, None]
        # X' = X / (C_p + C_q), Y' = Y / (C_p - C_q): (C_p - C_q)(EigY - EigX) = Y
        resp.append((cm * (y / cm), om, cp, s["b"].cpu()[:, p, q]))
    (ya, oa, ca, ba), (yb, ob, cb, bb) = resp
    t = (ya * ca).T @ (ba.T @ bb) @ (yb * cb)
    ka, kb = oa.abs() > 1e-3, ob.abs() > 1e-3
    t = t[ka][:, kb]
    return dict(e2disp=-16.0 * float((t * t / (oa[ka][:, None] + ob[kb][None, :])).sum()), eig_a=oa, eig_b=ob)


def exact(case, seed):
    k = case["kind"]
    if k in ("accas", "fofo", "solve", "dropin") and \
            case["nalpha"] * _npair(case["n"], case["ni"], case["na"]) ** 3 > 1.6e10:
        return None
    if k == "batch" and work(case)["flops"] > 1.6e11:
        return None
    inp = _inputs(case, seed, _device())
    if k == "transform":
        return _packed(torch.matmul(torch.matmul(inp["u"], inp["fac"]), inp["u"].T.contiguous()))
    if k == "batch":
        r = [_ref_accas(s, case["nalpha"]) for s in inp]
        return dict(ecorr=np.array([x["ecorr"] for x in r]), ecasscf=np.array([x["ecasscf"] for x in r]),
                    walpha=np.stack([x["walpha"] for x in r]))
    if k == "ac0":
        return _ref_ac0(inp)
    if k == "sapt":
        return _ref_sapt(inp)
    r = _ref_accas(inp, case["nalpha"])
    if k == "dropin":
        return dict(tno=_packed(inp["b"]).cpu().numpy(), walpha=r["walpha"], ecorr=r["ecorr"], egone=r["ecasscf"])
    if k != "accas":
        del r["eig"]
    return r
