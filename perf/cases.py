"""Performance cases of the LAPW setup library: what a ground-state program has it do.

Every case goes through the Python binding of the C-ABI (``exciting_amd.lapw``) on synthetic
crystals of ``exciting_amd.synth`` (orthorhombic cells of about 215 bohr^3 per atom, the radii,
basis sizes and local orbitals of its workloads).  Kinds (``case["kind"]``):

setup    match + H/O setup of all k-points in one grouped call, replayed as a hipGraph: the k
         loop of an SCF iteration (``split``: the modular split, else FP64)
scf      the same as an SCF program runs it, with a new potential each time: the muffin-tin
         integrals, V(G), then the grouped setup with the modular split
perk     one k-point after another on device arrays (match_dev, setup_dev)
host     one k-point after another on host arrays, as the Fortran driver calls the library
solve    after the setup: the generalized eigensolve of all k-points, the muffin-tin density
         matrix and density and the interstitial density.  Eigenvectors are defined up to a
         phase, so what they make (energies, density matrix, densities) is the output
density  the direct-route muffin-tin density of each k-point (rhovalk) and the interstitial one
forces   the adjoint of the setup (the IBS force term and dE/dV(G)) of each k-point
"""
import math

import numpy as np
import torch

from exciting_amd import lapw, synth

RMT = (2.0, 1.8, 2.2, 1.6)
VOLUME_PER_ATOM = 215.0
LMAXVR = 6                  # potential and density harmonics of the muffin-tin integrals
LMAXVR_DIRECT = 8           # of the direct-route density
MESH = (500, 460)           # radial mesh points of the species


def _case(name, kind, natm, nsp, lmax, lo, nk, n_lo, n_hi, split=False, nst=0):
    c = dict(kind=kind, natm=natm, nsp=nsp, lmax=lmax, lo=lo, nk=nk, n_lo=n_lo, n_hi=n_hi, split=split, nst=nst)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a two-atom cell at the coarsest cutoff: launches and latency
        _case("perk-2atom-N97", "perk", 2, 1, 8, "0011", 1, 97, 97),
        # a small cell with a k mesh (five atoms, as a perovskite): the everyday small calculation
        _case("setup-5atom-N260", "setup", 5, 3, 8, "01", 8, 235, 275),
        # workload 1's sizes: 8 atoms, 16 k-points
        _case("setup-8atom-N1200", "setup", 8, 2, 10, "01", 16, 1150, 1250),
        # the same sizes inside an SCF loop: every pass brings a new potential
        _case("scf-8atom-N1200-split", "scf", 8, 2, 10, "01", 8, 1150, 1250, split=True),
        # workload 4's sizes: 16 atoms, 8 k-points
        _case("setup-16atom-N2500", "setup", 16, 3, 10, "01", 8, 2475, 2525),
        # workload 3's sizes in FP64 (4 k-points) and with the modular split (8 k-points)
        _case("setup-32atom-N5000", "setup", 32, 4, 10, "01", 4, 4950, 5050),
        _case("setup-32atom-N5000-split", "setup", 32, 4, 10, "01", 8, 4950, 5050, split=True),
        # the Fortran driver's calls on host arrays, one k-point of workload 1
        _case("host-8atom-N1200", "host", 8, 2, 10, "01", 1, 1150, 1250),
        # the steps after the setup, 200 states
        _case("solve-8atom-N1200", "solve", 8, 2, 10, "01", 4, 1150, 1250, nst=200),
        _case("density-8atom-N1200", "density", 8, 2, 10, "01", 2, 1150, 1250, nst=200),
        # forces of workload 4: 64 states
        _case("forces-16atom-N2500", "forces", 16, 3, 10, "01", 2, 2475, 2525, nst=64),
    ]


def draw(rng):
    kind = rng.choice(["setup", "setup", "setup", "setup", "scf", "perk", "perk", "host", "solve", "density", "forces"])
    split = kind == "scf" or (kind == "setup" and rng.random() < 0.5)
    most = {"setup": 32, "scf": 16, "perk": 12, "host": 12, "solve": 8, "density": 12, "forces": 20}[kind]
    natm = max(2, min(most, round(2 * (most / 2) ** rng.random())))
    lmax = rng.choice([7, 8, 9, 10, 10, 10])
    if kind == "density":
        lmax = max(lmax, LMAXVR_DIRECT)
    # planewaves per atom: a coarse to a converged cutoff
    n_hi = round(natm * 50 * (162 / 50) ** rng.random())
    n_lo = max(16, n_hi - round(0.08 * n_hi * rng.random()) - rng.randint(0, 9))
    nsp = rng.randint(1, min(4, natm))
    lo = rng.choice(["01", "01", "0011", "012", "0"])
    # no more contraction work than four k-points of 32 atoms at N = 5000
    unit = natm * (lmax + 1) ** 2 * n_hi ** 2
    room = max(1, int(4 * 32 * 121 * 4950 ** 2 / unit))
    nk = min(room, round(16 ** rng.random())) if kind in ("setup", "scf") else min(4 if kind == "solve" else 2, room)
    nst = 0
    if kind in ("solve", "density", "forces"):
        nst = max(4, min(200, round(n_hi * rng.uniform(0.04, 0.16))))
    return _case(None, kind, natm, nsp, lmax, lo, nk, n_lo, n_hi, split=split, nst=nst)


# ------------------------------------------------------------------------------- inputs
def _inputs(case, seed):
    """Crystal, k-points and what the kind needs beside them, as host arrays, from the seed."""
    rng = np.random.default_rng([seed, 20261205])
    natm, nsp, nhi = case["natm"], case["nsp"], case["n_hi"]
    a = (VOLUME_PER_ATOM * natm) ** (1.0 / 3.0)
    per = [natm // nsp + (1 if s < natm % nsp else 0) for s in range(nsp)]
    # the G set of the crystal holds every difference G - G' of bases up to this size
    w = synth.make_small(natm_per_species=tuple(per), lmax=case["lmax"], lorbl=tuple(int(c) for c in case["lo"]),
                         n_target=nhi + nhi // 20 + 20, nk=1, seed=int(rng.integers(1 << 30)),
                         cell=(0.95 * a, a, a / 0.95), rmt=RMT[:nsp])
    cr = w.crystal
    # uneven basis sizes, the case's own
    sizes = np.random.default_rng([case["n_lo"], nhi, case["nk"]]).integers(case["n_lo"], nhi + 1, case["nk"])
    kps = [synth.make_kpoint(cr, rng, int(n), None) for n in sizes]
    ngkmax = max(k.ngp for k in kps)
    kps = [synth.pad_kpoint(k, ngkmax) for k in kps]
    more = {}
    if case["kind"] in ("scf", "solve", "density"):
        rd = synth.make_radial(cr, nr=MESH, lmaxvr=LMAXVR_DIRECT if case["kind"] == "density" else LMAXVR,
                               seed=int(rng.integers(1 << 30)))
        # normalised radial functions in a potential of valence depth
        for fr in (rd.apwfr, rd.lofr):
            for ia in range(cr.natm):
                n = int(rd.nrmt[cr.spidx[ia]])
                r = rd.spr[:n, cr.spidx[ia]]
                f = fr[:n, 0, ..., ia].reshape(n, -1)
                s = np.sqrt(np.trapezoid(f ** 2 * (r * r)[:, None], r, axis=0))
                fr[..., ia] /= s.reshape(fr.shape[2:-1])
        rd.veffmt *= 0.05
        more["rd"] = rd
    if case["kind"] == "scf":
        z = np.zeros(cr.ngrtot, dtype=np.complex128)
        z[_fft_index(cr)[:cr.ngvec]] = cr.veffig
        more["veffir"] = np.ascontiguousarray(np.fft.ifftn(z.reshape(_grid(cr)[::-1])).real.ravel() * cr.ngrtot)
    nst = case["nst"]
    if nst:
        # occupations falling from 2 to 0 over the upper states, one k-point weight
        t = (np.arange(nst) - 0.6 * nst) / (0.04 * nst)
        more["occ"] = [2.0 / (1.0 + np.exp(np.minimum(t, 40.0))) * rng.uniform(0.95, 1.0) for _ in kps]
        more["w"] = [1.0 / len(kps)] * len(kps)
    if case["kind"] in ("density", "forces"):
        more["C"] = [(rng.standard_normal((nst, k.ngp + cr.nlotot)) + 1j * rng.standard_normal((nst, k.ngp + cr.nlotot)))
                     / math.sqrt(2.0 * k.ngp) for k in kps]
        more["e"] = [np.sort(rng.uniform(-2.0, 2.0, nst)) for _ in kps]
    return cr, kps, more


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def prepare(case, seed):
    kind = case["kind"]
    cr, kps, more = _inputs(case, seed)
    stream = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=stream)
    s = dict(case=case, ctx=ctx, stream=stream, cr=cr, kps=kps)
    with torch.cuda.stream(stream):
        if kind == "host":
            s["apw"] = [np.zeros((k.igpig.shape[0], cr.apwordmax, cr.lmmaxapw, cr.natm), np.complex128, order="F")
                        for k in kps]
            s["ho"] = [tuple(np.zeros((k.ngp + cr.nlotot,) * 2, np.complex128, order="F") for _ in "ho") for k in kps]
            return s
        s["batch"] = b = lapw.DeviceBatch(cr, kps)
        for x in b.apw:
            x.zero_()                   # the rows past a k-point's basis are the caller's
        if kind == "scf":
            s.update(rd=more["rd"], veffir=more["veffir"])
            ctx.gencfun()
        if kind in ("solve", "density", "forces"):
            if kind != "forces":
                s["rd"] = more["rd"]
                ctx.hmlint(more["rd"], out=False)
            if kind == "solve":
                ctx.upload(cr)          # the seeded muffin-tin matrices; the radial functions stay
                ws = ctx.dmat_wfsize()
                s["eval"] = [torch.empty(case["nst"], dtype=torch.float64, device="cuda") for _ in kps]
                s["evec"] = [torch.empty((case["nst"], n), dtype=torch.complex128, device="cuda") for n in b.nmat]
                s["dm"] = torch.zeros((cr.natm, ws, ws), dtype=torch.complex128, device="cuda")
            else:
                s["evec"] = [_dev(c) for c in more["C"]]
            ctx.setup_batched_dev(b, lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE)
            s.update(occ=[_dev(o) for o in more["occ"]], w=more["w"])
            lmaxvr = LMAXVR_DIRECT if kind == "density" else LMAXVR
            s["rho_mt"] = torch.zeros((cr.natm, max(MESH[:cr.nspecies]), (lmaxvr + 1) ** 2), dtype=torch.float64,
                                      device="cuda")
            s["rho_ir"] = torch.zeros(cr.ngrtot, dtype=torch.float64, device="cuda")
            if kind == "density":
                zb, rf = _point_transform(LMAXVR_DIRECT)
                s.update(zb=_dev(zb.T), rf=_dev(rf.T))
            if kind == "forces":
                s["wh"] = [(w * o).contiguous() for w, o in zip(s["w"], s["occ"])]
                s["wo"] = [-w * o * _dev(e) for w, o, e in zip(s["w"], s["occ"], more["e"])]
                s["dtau"] = torch.zeros((cr.natm, 3), dtype=torch.float64, device="cuda")
                s["dv"] = torch.zeros(cr.ngvec, dtype=torch.complex128, device="cuda")
    stream.synchronize()
    return s


def run(s):
    case, ctx, kind = s["case"], s["ctx"], s["case"]["kind"]
    if kind == "host":
        for k, a, ho in zip(s["kps"], s["apw"], s["ho"]):
            ctx.match(k, out=a)
            ctx.hamiltonandoverlapsetup(k, a, out=ho, resident=True)
        return {"apwalm": s["apw"], "h": [x[0] for x in s["ho"]], "o": [x[1] for x in s["ho"]]}
    b = s["batch"]
    if kind in ("setup", "scf"):
        if kind == "scf":
            ctx.hmlint(s["rd"], out=False)
            ctx.genveffig(s["veffir"])
        ctx.setup_batched_dev(b, lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_GRAPH | lapw.EXC_BATCH_OLP_LEGENDRE |
                              (lapw.EXC_BATCH_SPLIT_CRT if case["split"] else 0))
        return {"apwalm": b.apw, "h": b.H, "o": b.O}
    if kind == "perk":
        for i, d in enumerate(b.dks):
            ctx.match_dev(d.ngp, d.ngkmax, d.gpc, d.tpgpc, d.sfacgp, b.apw[i])
            ctx.setup_dev(d.ngp, d.ngkmax, b.apw[i], d.igpig, d.vgpc, b.nmat[i], b.H[i], b.O[i])
        return {"apwalm": b.apw, "h": b.H, "o": b.O}
    nst = case["nst"]
    with torch.cuda.stream(s["stream"]):
        if kind == "forces":
            s["dtau"].zero_()
            s["dv"].zero_()
            for i, d in enumerate(b.dks):
                ctx.vjp_dev(d.ngp, d.ngkmax, b.apw[i], d.igpig, d.vgpc, d.sfacgp, s["evec"][i], b.nmat[i], nst,
                            s["wh"][i], s["wo"][i], s["dtau"], s["dv"])
            return {"dtau": s["dtau"], "dv": s["dv"]}
        s["rho_ir"].zero_()
        if kind == "density":
            s["rho_mt"].zero_()
            for i, d in enumerate(b.dks):
                ctx.rhovalk_dev(1, s["zb"], s["rf"], d.ngp, d.ngkmax, b.apw[i], nst, b.nmat[i], s["evec"][i],
                                s["occ"][i], s["w"][i], s["rho_mt"])
            ctx.genrhoir_batched_dev(b, nst, s["evec"], s["occ"], s["w"], s["rho_ir"])
            return {"rho_mt": s["rho_mt"], "rho_ir": s["rho_ir"]}
        ctx.eigen_batched_dev(b.nmat, b.H, b.O, nst, s["eval"], s["evec"])
        s["dm"].zero_()
        ctx.gendmatmt_batched_dev(b, nst, s["evec"], s["occ"], s["w"], s["dm"])
        ctx._call("exc_genrhomt_dev", ctx.h, s["dm"].data_ptr(), s["rho_mt"].data_ptr())
        ctx.genrhoir_batched_dev(b, nst, s["evec"], s["occ"], s["w"], s["rho_ir"])
        return {"eval": s["eval"], "dm": s["dm"], "rho_mt": s["rho_mt"], "rho_ir": s["rho_ir"]}


# ------------------------------------------------------------------------------- work
def work(case):
    """Bytes: every input read once, every output written once.  Flops, real, per k-point: the
    muffin-tin product h A and the upper triangle of conj(A) (h A) for H, the addition-theorem sum
    for O's upper triangle (three multiply-adds per atom and l); for the other kinds the
    products they are made of."""
    natm, L, nk, nst = case["natm"], case["lmax"], case["nk"], case["nst"]
    n = 0.5 * (case["n_lo"] + case["n_hi"])
    naa = 2 * (L + 1) ** 2
    K = natm * naa
    nlo = sum(2 * int(c) + 1 for c in case["lo"])
    nmat = n + natm * nlo
    apw, mats = 16.0 * K * n, 2 * 16.0 * nmat ** 2
    kind = case["kind"]
    tables = 16.0 * natm * naa * (naa + nlo) + 32.0 * 8 * n
    grid = 18.0 * n                                   # points of the G box
    npts = natm * MESH[0]
    if kind in ("setup", "scf", "perk", "host"):
        f = 8.0 * K * naa * n + 4.0 * K * n * n + 3.0 * natm * (L + 1) * n * n + 8.0 * K * nlo * n
        by = nk * (apw + mats + 16.0 * n * (natm + 4)) + tables
        if kind == "scf":
            by += 8.0 * npts * ((LMAXVR + 1) ** 2 + 4 * (L + 2)) + 8.0 * grid
        return {"bytes": by, "flops": nk * f}
    if kind == "forces":
        # V_l = (q_l C)^T A for q_0 .. q_3, their products with h, and D, W per pair with the G sum
        f = 4 * 8.0 * nst * n * K + 4 * 8.0 * nst * K * naa + 2 * 8.0 * nst * n * n / 2
        return {"bytes": nk * (apw + 16.0 * nst * nmat + 16.0 * n * (natm + 4)) + tables + 16.0 * grid,
                "flops": nk * f}
    fft = nst * 5.0 * grid * math.log2(grid)
    if kind == "density":
        lmv = (LMAXVR_DIRECT + 1) ** 2
        nf = 2 * (LMAXVR_DIRECT + 1) + len(case["lo"])
        f = 8.0 * 2 * natm * lmv * nst * n + 16.0 * natm * lmv * lmv * nst + 4.0 * natm * lmv * nst * nf * (nf + 1) / 2
        f += npts * (1.5 * nf * nf * lmv + 2.0 * lmv * lmv)
        return {"bytes": nk * (apw * lmv / (L + 1.0) ** 2 + 16.0 * nst * nmat) + 8.0 * npts * lmv + 8.0 * grid,
                "flops": nk * (f + fft)}
    # solve: Cholesky, reduction to standard form and tridiagonal form of order nmat, the
    # transformation of nst vectors, the density matrix of nst states
    f = 4.0 * (1 / 3 + 1 + 4 / 3) * nmat ** 3 + 8.0 * 1.5 * nmat ** 2 * nst + 8.0 * K * nst * n + 4.0 * K * naa * nst
    return {"bytes": nk * (mats + apw + 2 * 16.0 * nst * nmat) + 16.0 * natm * naa ** 2 + 8.0 * npts * 49 + 8.0 * grid,
            "flops": nk * (f + fft)}


# ------------------------------------------------------------------------------- values in 64 bits
def _grid(cr):
    return [int(cr.intgv[i, 1] - cr.intgv[i, 0] + 1) for i in range(3)]


def _fft_index(cr):
    n = _grid(cr)
    j = [np.mod(cr.ivg[i].astype(np.int64), n[i]) for i in range(3)]
    return j[0] + n[0] * (j[1] + n[1] * j[2])


def _bessel(lmax, x):
    """j_l(x) for l = 0 .. lmax, downward from far above lmax, normalised by sum (2l+1) j_l^2 = 1."""
    top = lmax + 30 + int(x.max())
    j = np.zeros((top + 2, x.size))
    j[top] = 1e-150
    for l in range(top, 0, -1):
        j[l - 1] = (2 * l + 1) / x * j[l] - j[l + 1]
        big = np.abs(j[l - 1]) > 1e100
        j[l - 1:, big] *= 1e-100
    j /= np.sqrt((np.arange(1, 2 * top + 4, 2)[:, None] * j * j).sum(axis=0))
    return j[:lmax + 1] * np.sign(np.where(np.abs(j[0]) > np.abs(j[1]), np.sin(x) / x / j[0],
                                           (np.sin(x) / x - np.cos(x)) / x / j[1]))


def _ylm(lmax, theta, phi):
    """Y_lm at points, rows l(l+1)+m, from the normalised Legendre recurrence."""
    y = np.zeros(((lmax + 1) ** 2, theta.size), dtype=np.complex128)
    c, s = np.cos(theta), np.sin(theta)
    p = np.full(theta.size, math.sqrt(0.25 / math.pi))
    for m in range(lmax + 1):
        if m:
            p = -p * s * math.sqrt((2 * m + 1) / (2.0 * m))
        q0, q1 = np.zeros_like(p), p
        for l in range(m, lmax + 1):
            if l > m:
                a = math.sqrt((4.0 * l * l - 1) / (l * l - m * m))
                b = math.sqrt(((l - 1.0) ** 2 - m * m) / (4.0 * (l - 1) ** 2 - 1)) if l > m + 1 else 0.0
                q0, q1 = q1, a * (c * q1 - b * q0)
            v = q1 * np.exp(1j * m * phi)
            y[l * l + l + m] = v
            y[l * l + l - m] = (-1) ** m * v.conj()
    return y


def _real_ylm(lmax, theta, phi):
    y = _ylm(lmax, theta, phi)
    r = np.empty(y.shape)
    for l in range(lmax + 1):
        for m in range(-l, l + 1):
            v = y[l * l + l + m]
            r[l * l + l + m] = v.real if m == 0 else math.sqrt(2.0) * (v.real if m > 0 else v.imag)
    return r


def _point_transform(lmax):
    """Y_lm at (lmax+1)^2 points on a spiral over the sphere, (point, lm), and the inverse of the
    real harmonics at those points, (lm, point)."""
    n = (lmax + 1) ** 2
    h = 2.0 * np.arange(n) / (n - 1) - 1.0
    theta = np.arccos(h)
    step = np.zeros(n)
    step[1:-1] = math.sqrt(8.0 * math.pi / math.sqrt(3.0) / n) / np.sqrt(1.0 - h[1:-1] ** 2)
    phi = np.mod(np.cumsum(step), 2.0 * math.pi)
    phi[-1] = 0.0
    return _ylm(lmax, theta, phi).T.copy(), np.linalg.inv(_real_ylm(lmax, theta, phi).T)


def _x_apw(cr, kp):
    """apwalm as (natm, lm, io, G) on the GPU."""
    n, L = kp.ngp, cr.lmaxapw
    g = kp.gpc[:n]
    y = _ylm(L, kp.tpgpc[0, :n], kp.tpgpc[1, :n]).conj()
    lof = np.repeat(np.arange(L + 1), 2 * np.arange(L + 1) + 1)
    pre = y * (4.0 * math.pi / math.sqrt(cr.omega) * 1j ** lof)[:, None]
    out = torch.empty((cr.natm, (L + 1) ** 2, 2, n), dtype=torch.complex128, device="cuda")
    pre = _dev(pre)
    for s in range(cr.nspecies):
        x = g * cr.rmt[s]
        j = _bessel(L + 1, x)
        l = np.arange(L + 1)[:, None]
        f = np.stack([j[:L + 1], g * (l / x * j[:L + 1] - j[1:])], axis=1)            # (l, order, G)
        for a in np.nonzero(cr.spidx == s)[0]:
            r = np.linalg.solve(np.moveaxis(cr.dmat[:, :, :, a], 2, 0), f)            # (l, io, G)
            out[a] = pre[:, None, :] * (_dev(r[lof]) * _dev(kp.sfacgp[:n, a]))
    return out


def _x_pairs(cr, kp):
    """Index of G_i - G_j (0-based) and whether it is one of the first ngvec, on the GPU."""
    iv = torch.from_numpy(cr.ivg[:, kp.igpig[:kp.ngp] - 1].astype(np.int64)).cuda()
    box = _dev(cr.ivgig.astype(np.int64))
    lin, ok = 0, True
    for q in range(3):
        d = iv[q][:, None] - iv[q][None, :] - int(cr.intgv[q, 0])
        ok = ok & (d >= 0) & (d < box.shape[q])
        lin = lin * box.shape[q] + d.clamp(0, box.shape[q] - 1)
    ig = box.reshape(-1)[lin]
    ok = ok & (ig > 0) & (ig <= cr.ngvec)
    return torch.where(ok, ig - 1, 0), ok


def _x_setup(cr, kp, mt=None, veffig=None):
    """(apwalm, H, O) of one k-point, matrices as (row, column)."""
    haa, loa, lolo, oalo, ololo = mt or (cr.haa, cr.loa, cr.lolo, cr.oalo, cr.ololo)
    A = _x_apw(cr, kp)
    n, nm, naa = kp.ngp, kp.ngp + cr.nlotot, cr.maxaa
    H = torch.zeros((nm, nm), dtype=torch.complex128, device="cuda")
    O = torch.zeros_like(H)
    for a in range(cr.natm):
        f = A[a].reshape(naa, n)
        fh = f.conj().T.contiguous()
        H[:n, :n] += fh @ (_dev(haa[:, :, a]) @ f)
        O[:n, :n] += fh @ f
        s = cr.spidx[a]
        r = n + int(cr.idxlo[:, :, a][cr.idxlo[:, :, a] > 0].min()) - 1
        ns = int(cr.losize[s])
        H[r:r + ns, :n] = _dev(loa[:ns, :, a]) @ f
        H[:n, r:r + ns] = H[r:r + ns, :n].conj().T
        H[r:r + ns, r:r + ns] += _dev(lolo[:ns, :ns, a])
        for i in range(int(cr.nlorb[s])):
            l = int(cr.lorbl[i, s])
            p = n + int(cr.idxlo[l * l, i, a]) - 1
            w = _dev(oalo[:, i, a]).to(torch.complex128)
            blk = (A[a, l * l:(l + 1) ** 2] * w[None, :, None]).sum(1)
            O[p:p + 2 * l + 1, :n] += blk
            O[:n, p:p + 2 * l + 1] += blk.conj().T
            for q in range(int(cr.nlorb[s])):
                if int(cr.lorbl[q, s]) == l:
                    p2 = n + int(cr.idxlo[l * l, q, a]) - 1
                    for m in range(2 * l + 1):
                        O[p + m, p2 + m] += float(ololo[i, q, a])
    ig, ok = _x_pairs(cr, kp)
    v = _dev(kp.vgpc[:, :n])
    th = torch.where(ok, _dev(cr.cfunig)[ig], 0.0)
    H[:n, :n] += torch.where(ok, _dev(cr.veffig if veffig is None else veffig)[ig], 0.0) + 0.5 * (v.T @ v) * th
    O[:n, :n] += th
    return A, H, O


def _quadrature(w):
    """Weights of the integral of the interpolating cubic spline on a mesh: second derivatives
    continuous, those of the end points from the second divided differences there."""
    x, n = w, w.size
    h = np.diff(x)
    D = np.zeros((n, n))                               # right-hand sides on the samples
    M = np.zeros((n, n))
    for i, k in ((0, 0), (n - 1, n - 3)):
        M[i, i] = 1.0
        for p in range(3):
            D[i, k + p] = 1.0 / np.prod([x[k + p] - x[k + q] for q in range(3) if q != p])
    for i in range(1, n - 1):
        M[i, i - 1:i + 2] = h[i - 1], 2.0 * (h[i - 1] + h[i]), h[i]
        D[i, i - 1:i + 2] = 3.0 / h[i - 1], -3.0 / h[i - 1] - 3.0 / h[i], 3.0 / h[i]
    t, c = np.zeros(n), np.zeros(n)
    for e in (slice(None, -1), slice(1, None)):
        t[e] += 0.5 * h
        c[e] -= h ** 3 / 12.0
    return t + np.linalg.solve(M.T, c) @ D


def _gaunt(L, lv):
    """int conj(Y_1) R_2 Y_3 over the sphere as (lm1, lm2, lm3), by Gauss quadrature."""
    ct, w = np.polynomial.legendre.leggauss(L + lv // 2 + 2)
    nph = 2 * L + lv + 2
    ph = 2.0 * math.pi * np.arange(nph) / nph
    th, ph = np.repeat(np.arccos(ct), nph), np.tile(ph, ct.size)
    w = np.repeat(w, nph) * 2.0 * math.pi / nph
    y, r = _ylm(L, th, ph), _real_ylm(lv, th, ph)
    return np.stack([(y.conj() * (w * r[k])) @ y.T for k in range(r.shape[0])], axis=1)


def _functions(cr, rd, a):
    """Radial functions of an atom: u, u', l; APW (l, io) io fastest, then the local orbitals."""
    s = cr.spidx[a]
    n = int(rd.nrmt[s])
    f = rd.apwfr[:n, :, :, :, a]                       # (r, 2, io, l)
    u = np.transpose(f, (1, 3, 2, 0)).reshape(2, -1, n)
    lo = np.transpose(rd.lofr[:n, :, :int(cr.nlorb[s]), a], (1, 2, 0))
    l = np.concatenate([np.repeat(np.arange(cr.lmaxapw + 1), 2), cr.lorbl[:int(cr.nlorb[s]), s]]).astype(int)
    u = np.concatenate([u, lo], axis=1)
    return u[0], u[1], l, rd.spr[:n, s]


def _x_hmlint(cr, rd):
    """The muffin-tin matrices of the radial data: haa, loa, lolo, oalo, ololo."""
    L, na = cr.lmaxapw, cr.natm
    haa, loa, lolo = np.zeros_like(cr.haa), np.zeros_like(cr.loa), np.zeros_like(cr.lolo)
    oalo, ololo = np.zeros_like(cr.oalo), np.zeros_like(cr.ololo)
    G = _gaunt(L, rd.lmaxvr)
    for a in range(na):
        u, du, l, r = _functions(cr, rd, a)
        w = _quadrature(r)
        P = np.einsum("ar,vr,br->vab", u, rd.veffmt[:, :r.size, a] * (w * r * r), u, optimize=True)
        same = l[:, None] == l[None, :]
        Kin = same * 0.5 * ((du * (w * r * r)) @ du.T + (l * (l + 1))[:, None] * ((u * w) @ u.T))
        S = (u * (w * r * r)) @ u.T
        # every function with its m: APW (lm, io) io fastest, then the local orbitals
        fn, lm = [], []
        for ll in range(L + 1):
            for m in range(-ll, ll + 1):
                fn += [2 * ll, 2 * ll + 1]
                lm += [ll * ll + ll + m] * 2
        for i in range(2 * (L + 1), l.size):
            fn += [i] * (2 * l[i] + 1)
            lm += list(range(l[i] ** 2, (l[i] + 1) ** 2))
        fn, lm = np.array(fn), np.array(lm)
        h = (G[lm[:, None], :, lm[None, :]] * np.moveaxis(P, 0, 2)[fn[:, None], fn[None, :]]).sum(2)
        h += (lm[:, None] == lm[None, :]) * Kin[fn[:, None], fn[None, :]]
        q = cr.maxaa
        ns = fn.size - q
        haa[:, :, a], loa[:ns, :, a], lolo[:ns, :ns, a] = h[:q, :q], h[q:, :q], h[q:, q:]
        for i in range(l.size - 2 * (L + 1)):
            b = 2 * (L + 1) + i
            oalo[:, i, a] = S[2 * l[b]:2 * l[b] + 2, b]
            ololo[i, :l.size - 2 * (L + 1), a] = np.where(l[2 * (L + 1):] == l[b], S[b, 2 * (L + 1):], 0.0)
    return haa, loa, lolo, oalo, ololo


def _x_rhoir(cr, kp, C, t):
    """Interstitial density of states C (state, G + lo) with weights t / Omega on the FFT grid."""
    idx = torch.from_numpy(_fft_index(cr)[kp.igpig[:kp.ngp] - 1]).cuda()
    rho = torch.zeros(cr.ngrtot, dtype=torch.float64, device="cuda")
    for j in range(C.shape[0]):
        z = torch.zeros(cr.ngrtot, dtype=torch.complex128, device="cuda")
        z[idx] = C[j, :kp.ngp]
        z = torch.fft.ifftn(z.reshape(_grid(cr)[::-1]), norm="forward").reshape(-1)
        rho += (t[j] / cr.omega) * (z.real ** 2 + z.imag ** 2)
    return rho


def _lo_rows(cr, a):
    """First local-orbital row of an atom and their number."""
    q = cr.idxlo[:, :, a]
    return int(q[q > 0].min()) - 1, int(cr.losize[cr.spidx[a]])


def _x_solve(cr, kps, more, nst):
    L = cr.lmaxapw
    order = np.array([2 * (l * l + m) + io for l in range(L + 1) for io in (0, 1) for m in range(2 * l + 1)])
    ws = cr.maxaa + cr.maxnlo
    dm = torch.zeros((cr.natm, ws, ws), dtype=torch.complex128, device="cuda")     # (atom, row, column)
    rho_ir, evals = 0.0, []
    for i, kp in enumerate(kps):
        A, H, O = _x_setup(cr, kp)
        h, o = H.cpu().numpy(), O.cpu().numpy()
        Li = np.linalg.inv(np.linalg.cholesky(o))
        e, v = np.linalg.eigh(Li @ h @ Li.conj().T)
        C = _dev((Li.conj().T @ v[:, :nst]).T)
        evals.append(_dev(e[:nst]))
        t = _dev(more["w"][i] * more["occ"][i])
        for a in range(cr.natm):
            wf = torch.zeros((ws, nst), dtype=torch.complex128, device="cuda")
            wf[:cr.maxaa] = A[a].reshape(cr.maxaa, -1)[order] @ C[:, :kp.ngp].T.contiguous()
            r, ns = _lo_rows(cr, a)
            wf[cr.maxaa:cr.maxaa + ns] = C[:, kp.ngp + r:kp.ngp + r + ns].T
            dm[a] += (wf * t) @ wf.conj().T.contiguous()
        rho_ir = rho_ir + _x_rhoir(cr, kp, C, t)
    # the muffin-tin density: sum over pairs of functions of u u' Re(dm conj(G))
    rd = more["rd"]
    lv = (rd.lmaxvr + 1) ** 2
    G = _gaunt(max(L, int(cr.lorbl.max())), rd.lmaxvr)
    rho = np.zeros((cr.natm, rd.spr.shape[0], lv))
    for a in range(cr.natm):
        u, _, l, r = _functions(cr, rd, a)
        d = dm[a].cpu().numpy()
        off = np.concatenate([[0], np.cumsum(2 * l + 1)])
        nf = 2 * (L + 1)
        F = np.zeros((lv, l.size, l.size))
        for p in range(l.size):
            for q in range(l.size):
                if p >= nf > q:
                    continue                           # twice the APW-lo block instead
                blk = d[off[p]:off[p + 1], off[q]:off[q + 1]]
                g = G[l[p] ** 2:(l[p] + 1) ** 2, :, l[q] ** 2:(l[q] + 1) ** 2]
                F[:, p, q] = (2.0 if p < nf <= q else 1.0) * np.einsum("ab,avb->v", blk, g.conj()).real
        rho[a, :r.size] = np.einsum("vab,ar,br->rv", F, u, u, optimize=True)
    # run's density matrix is column-major per atom
    return {"eval": evals, "dm": dm.transpose(1, 2), "rho_mt": rho, "rho_ir": rho_ir}


def _x_density(cr, kps, more, nst):
    rd, L = more["rd"], LMAXVR_DIRECT
    lv = (L + 1) ** 2
    zb, rf = (_dev(x) for x in _point_transform(L))
    rho, rho_ir = torch.zeros((cr.natm, rd.spr.shape[0], lv), dtype=torch.float64, device="cuda"), 0.0
    for i, kp in enumerate(kps):
        A, C = _x_apw(cr, kp), _dev(more["C"][i])
        t = _dev(more["w"][i] * more["occ"][i])
        rho_ir = rho_ir + _x_rhoir(cr, kp, C, t)
        Ct = C[:, :kp.ngp].T.contiguous()
        for a in range(cr.natm):
            s = cr.spidx[a]
            n = int(rd.nrmt[s])
            coef = (A[a, :min(lv, A.shape[1])].reshape(-1, kp.ngp) @ Ct).reshape(-1, 2, nst)
            u = _dev(np.transpose(rd.apwfr[:n, 0, :, :, a], (2, 1, 0)).copy())         # (l, io, r)
            lo, ns = _lo_rows(cr, a)
            pts = torch.zeros((lv, n), dtype=torch.float64, device="cuda")
            for j in range(nst):
                if abs(more["w"][i] * more["occ"][i][j]) <= 1e-8:
                    continue
                wf = torch.zeros((lv, n), dtype=torch.complex128, device="cuda")
                for l in range(min(L, cr.lmaxapw) + 1):
                    wf[l * l:(l + 1) ** 2] = coef[l * l:(l + 1) ** 2, :, j] @ u[l].to(torch.complex128)
                p = kp.ngp + lo
                for q in range(int(cr.nlorb[s])):
                    l = int(cr.lorbl[q, s])
                    wf[l * l:(l + 1) ** 2] += C[j, p:p + 2 * l + 1, None] * _dev(rd.lofr[:n, 0, q, a])
                    p += 2 * l + 1
                z = zb @ wf
                pts += t[j] * (z.real ** 2 + z.imag ** 2)
            rho[a, :n] += (rf @ pts).T
    return {"rho_mt": rho, "rho_ir": rho_ir}


def _x_forces(cr, kps, more):
    dtau = torch.zeros((cr.natm, 3), dtype=torch.float64, device="cuda")
    dv = torch.zeros(cr.ngvec, dtype=torch.complex128, device="cuda")
    vgc, pos = _dev(cr.vgc[:, :cr.ngvec]), _dev(cr.atposc)
    ffac = _dev(cr.ffacg)
    for i, kp in enumerate(kps):
        n = kp.ngp
        A, C = _x_apw(cr, kp), _dev(more["C"][i])
        wh = more["w"][i] * more["occ"][i]
        wh, wo = _dev(wh), _dev(-wh * more["e"][i])
        # D_ji and W_ji as (i, j) arrays: conj(C_i) w C_j
        Cc = C.conj().T.contiguous()
        D, W = Cc @ (wh[:, None] * C), Cc @ (wo[:, None] * C)
        ig, ok = _x_pairs(cr, kp)
        Dg = torch.where(ok, D[:n, :n], 0.0)
        dv.real.index_add_(0, ig.reshape(-1), Dg.real.reshape(-1).contiguous())
        dv.imag.index_add_(0, ig.reshape(-1), Dg.imag.reshape(-1).contiguous())
        q = _dev(kp.vgpc[:, :n])
        E = torch.where(ok, 0.5 * (q.T @ q) * D[:n, :n] + W[:n, :n], 0.0)
        th = torch.zeros(cr.ngvec, dtype=torch.complex128, device="cuda")       # sum of E per G_i - G_j
        th.real.index_add_(0, ig.reshape(-1), E.real.reshape(-1).contiguous())
        th.imag.index_add_(0, ig.reshape(-1), E.imag.reshape(-1).contiguous())
        for a in range(cr.natm):
            s = int(cr.spidx[a])
            f = A[a].reshape(cr.maxaa, n)
            fh = f.conj().T.contiguous()
            X = (fh @ (_dev(cr.haa[:, :, a]) @ f)) * D[:n, :n] + (fh @ f) * W[:n, :n]
            r, ns = _lo_rows(cr, a)
            r += n
            y = ((_dev(cr.loa[:ns, :, a]) @ f).conj().T * D[:n, r:r + ns]).sum(1)
            p = r
            for b in range(int(cr.nlorb[s])):
                l = int(cr.lorbl[b, s])
                w = _dev(cr.oalo[:, b, a]).to(torch.complex128)
                o = (A[a, l * l:(l + 1) ** 2] * w[None, :, None]).sum(1).conj().T
                y += (o * W[:n, p:p + 2 * l + 1]).sum(1)
                p += 2 * l + 1
            g = X.sum(1) - X.sum(0)
            ph = -ffac[:, s] * torch.exp(-1j * (vgc.T @ pos[:, a]).to(torch.complex128))
            for d in range(3):
                dtau[a, d] += (q[d] * (g + 2.0 * y)).sum().imag + (vgc[d] * ph * th).sum().imag
    return {"dtau": dtau, "dv": dv}


def exact(case, seed):
    cr, kps, more = _inputs(case, seed)
    kind = case["kind"]
    if kind == "solve":
        return _x_solve(cr, kps, more, case["nst"])
    if kind == "density":
        return _x_density(cr, kps, more, case["nst"])
    if kind == "forces":
        return _x_forces(cr, kps, more)
    mt = veffig = None
    if kind == "scf":
        mt = _x_hmlint(cr, more["rd"])
        idx, shape = _fft_index(cr), _grid(cr)[::-1]
        z = np.zeros(cr.ngrtot, dtype=np.complex128)
        z[idx] = cr.cfunig
        z = np.fft.ifftn(z.reshape(shape)).real * cr.ngrtot
        veffig = (np.fft.fftn(z * more["veffir"].reshape(shape)) / cr.ngrtot).ravel()[idx[:cr.ngvec]]
    out = {"apwalm": [], "h": [], "o": []}
    for kp in kps:
        A, H, O = _x_setup(cr, kp, mt, veffig)
        if kind == "host":                            # Fortran-ordered host arrays: (G, io, lm, atom), (row, column)
            out["apwalm"].append(_padded(A, kp).permute(3, 2, 1, 0).cpu().numpy())
            out["h"].append(H.cpu().numpy())
            out["o"].append(O.cpu().numpy())
        else:                                          # (atom, lm, io, G), (column, row)
            out["apwalm"].append(_padded(A, kp))
            out["h"].append(H.T)
            out["o"].append(O.T)
        del A, H, O
    return out


def _padded(A, kp):
    out = torch.zeros(A.shape[:3] + (kp.igpig.shape[0],), dtype=A.dtype, device=A.device)
    out[..., :kp.ngp] = A
    return out
