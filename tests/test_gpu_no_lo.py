"""Crystals without local orbitals, and with a species that has none: the setup (per-k and grouped, the
narrow tiles the small sizes take and the 64-wide ones) and the adjoint, whose lo kernels then
launch nothing or skip the atom, against the oracle.

Bars: H and O within 1e-12 of the oracle's norm (test_gpu_setup.py), the adjoint within 1e-9
(test_gpu_vjp.py)."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _without(cr, species):
    """The crystal without the local orbitals of these species (columns numbered anew)."""
    nlorb, losize = cr.nlorb.copy(), cr.losize.copy()
    nlorb[list(species)] = 0
    losize[list(species)] = 0
    idxlo, n = np.zeros_like(cr.idxlo), 0
    loa, lolo, oalo, ololo = cr.loa.copy(), cr.lolo.copy(), cr.oalo.copy(), cr.ololo.copy()
    for a in range(cr.natm):
        s = cr.spidx[a]
        for i in range(nlorb[s]):
            l = int(cr.lorbl[i, s])
            for m in range(l * l, (l + 1) ** 2):
                n += 1
                idxlo[m, i, a] = n
        if nlorb[s] == 0:
            loa[:, :, a], lolo[:, :, a], oalo[:, :, a], ololo[:, :, a] = 0.0, 0.0, 0.0, 0.0
    return dataclasses.replace(cr, nlorb=nlorb, losize=losize, idxlo=idxlo, nlotot=n, loa=loa, lolo=lolo, oalo=oalo,
                               ololo=ololo)


@pytest.mark.parametrize("n,lmax,species", [(17, 2, (0, 1)), (97, 4, (0, 1)), (97, 4, (0,)), (130, 3, (1,))])
def test_without_local_orbitals(n, lmax, species):
    import torch
    from exciting_amd import lapw, synth
    from oracle import lapw_ref as R
    w = synth.make_small(natm_per_species=(2, 1), lmax=lmax, lorbl=(0, 1), n_target=n, nk=2, seed=21 + n,
                         cell=(9.0, 9.5, 10.0))
    cr = _without(w.crystal, species)
    assert (cr.nlotot == 0) == (len(species) == 2)
    ref = [R.setup(cr, kp) for kp in w.kpoints]
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    assert ctx.nlotot == cr.nlotot
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, w.kpoints)

        def perk():
            for i, d in enumerate(b.dks):
                ctx.match_dev(d.ngp, d.ngkmax, d.gpc, d.tpgpc, d.sfacgp, b.apw[i])
                ctx.setup_dev(d.ngp, d.ngkmax, b.apw[i], d.igpig, d.vgpc, b.nmat[i], b.H[i], b.O[i])

        runs = [("per-k", perk)] + [(f"flags {f}", lambda f=f: ctx.setup_batched_dev(b, f)) for f in (
            lapw.EXC_BATCH_MATCH, lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE | lapw.EXC_BATCH_GRAPH)]
        for v in (-1, 0):
            for stage in ("mt", "bmt", "ystage"):
                ctx.set_variant(stage, v)
            for name, run in runs:
                for t in b.H + b.O:
                    t.fill_(float("nan"))
                print(f"no lo: N={n} species {species} variant {v} {name}", flush=True)
                run()
                torch.cuda.synchronize()
                for i, (hr, orf, _) in enumerate(ref):
                    for m, r in ((b.H[i], hr), (b.O[i], orf)):
                        m = m.cpu().numpy().T
                        assert np.linalg.norm(m - r) <= 1e-12 * np.linalg.norm(r)
    # the adjoint of the first k-point
    kp, d, rng, nst = w.kpoints[0], b.dks[0], np.random.default_rng(n), 5
    nmat = kp.ngp + cr.nlotot
    C = (rng.standard_normal((nmat, nst)) + 1j * rng.standard_normal((nmat, nst))) / np.sqrt(2.0 * n)
    wh, wo = rng.uniform(0.0, 2.0, nst), rng.uniform(-2.0, 2.0, nst)
    ref_t, ref_v = R.setup_vjp(cr, kp, (C * wh) @ C.conj().T, (C * wo) @ C.conj().T)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    dt = torch.zeros((cr.natm, 3), dtype=torch.float64, device="cuda")
    dv = torch.zeros(cr.ngvec, dtype=torch.complex128, device="cuda")
    c, h, o = dev(C.T), dev(wh), dev(wo)
    torch.cuda.synchronize()
    ctx.vjp_dev(kp.ngp, d.ngkmax, b.apw[0], d.igpig, d.vgpc, d.sfacgp, c, nmat, nst, h, o, dt, dv)
    torch.cuda.synchronize()
    assert np.linalg.norm(dt.cpu().numpy().T - ref_t) <= 1e-9 * np.linalg.norm(ref_t)
    assert np.linalg.norm(dv.cpu().numpy() - ref_v) <= 1e-9 * np.linalg.norm(ref_v)
    ctx.status()
    ctx.close()
