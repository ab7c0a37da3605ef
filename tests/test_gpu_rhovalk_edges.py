"""The direct-route density's matrix products at the edges of their tiles of 16 (states, points,
mesh points, pairs of radial functions), and the interstitial density over chunks of states.

Bars: rhovalk within 1e-12 of the oracle relative to its largest value (the same sums in another
order, as test_gpu_rhovalk.py); the interstitial density of many states within 64 eps nst of the
sum over calls of one state each, relative to its largest value (positive terms, the same
transforms, nst terms in two orders of summation)."""
import numpy as np
import pytest

from conftest import small

pytestmark = pytest.mark.gpu


def _states(cr, ngp, nst, seed):
    rng = np.random.default_rng(seed)
    C = np.asfortranarray(rng.standard_normal((ngp + cr.nlotot, nst)) + 1j * rng.standard_normal((ngp + cr.nlotot, nst)))
    occ = rng.uniform(0.1, 2.0, nst)
    if nst > 2:
        occ[1] = 0.0
    return C, occ


@pytest.mark.parametrize("nst,lmaxvr,nr,lradstep", [(1, 0, (17, 16), 1), (4, 1, (33, 15), 1), (15, 2, (40, 64), 7),
                                                    (16, 3, (100, 49), 3), (17, 4, (65, 120), 1), (65, 4, (48, 31), 2)])
def test_rhovalk_tile_edges(nst, lmaxvr, nr, lradstep):
    from exciting_amd import lapw, synth
    from oracle import lapw_ref as R
    from oracle import rhovalk_ref as V
    w = small("d")
    cr, kp = w.crystal, w.kpoints[0]
    rd = synth.make_radial(cr, nr=nr, lmaxvr=lmaxvr, seed=nst)
    apw = R.match(cr, kp)
    C, occ = _states(cr, kp.ngp, nst, nst)
    ctx = lapw.Context(cr)
    ctx.hmlint(rd, out=False)
    zb, _, rf = V.genshtmat(lmaxvr)
    nrmtmax = rd.spr.shape[0]
    got = ctx.rhovalk(np.asfortranarray(apw), kp.ngp, C, occ, 0.35, zb, rf, lmaxvr, nrmtmax, lradstep=lradstep)
    ref = V.rhovalk(cr, rd, apw, kp.ngp, C, occ, 0.35, lradstep=lradstep, sht=(zb, None, rf))
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("nst", [1, 2, 3, 63, 64, 65, 130])
def test_interstitial_density_chunks(nst):
    import torch
    from exciting_amd import lapw
    w = small("d")
    cr, kp = w.crystal, w.kpoints[0]
    C, occ = _states(cr, kp.ngp, nst, 3)
    occ = np.where(occ > 0.0, occ, 1e-12)      # below epsocc
    ctx = lapw.Context(cr)
    ctx.gencfun()
    got = ctx.genrhoir(kp, C, occ, 0.4)
    ref = np.zeros_like(got)
    for j in range(nst):
        ref += ctx.genrhoir(kp, np.asfortranarray(C[:, j:j + 1]), occ[j:j + 1], 0.4)
    assert np.abs(got - ref).max() <= 64 * 2.2e-16 * nst * max(np.abs(ref).max(), 1e-300)
