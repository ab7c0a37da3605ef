"""The radial integrals' matrix-core tiles (k_hmlint.hip) at their edges: 15, 16, 17, 33 and 41 radial
functions (tiles of 16), meshes of 4 points up to the largest accepted, mesh lengths that the four
waves share unevenly, two species of different length.

Bar: max |difference| <= 1e-12 of the largest element against the oracle, as test_gpu_hmlint.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,lo,nr,lmaxvr", [(6, (0,), (4, 7), 2), (6, (0, 1), (16, 17), 3), (7, (0,), (63, 65), 1),
                                               (3, (0, 1, 2), (100, 33), 4), (12, (0, 1, 0, 1, 0, 1, 2), (40, 21), 0),
                                               (1, (0,), (8192, 500), 0), (12, (0, 1, 2) * 5, (30, 18), 1)])
def test_hmlint_tiles(lmax, lo, nr, lmaxvr):
    from exciting_amd import lapw, synth
    from oracle import hmlint_ref as M
    w = synth.make_small(natm_per_species=(1, 1), lmax=lmax, lorbl=lo, n_target=30, nk=1, seed=lmax + len(lo))
    cr = w.crystal
    rd = synth.make_radial(cr, nr=nr, lmaxvr=lmaxvr, seed=3)
    ctx = lapw.Context(cr)
    print(f"hmlint lmax {lmax}, lo {lo}, mesh {nr}, lmaxvr {lmaxvr}", flush=True)
    haa, loa, lolo, oalo, ololo = ctx.hmlint(rd)
    rh, rl, rll = M.hmlint(cr, rd)
    ro, roo = M.olprad(cr, rd)
    mn, nl = cr.maxnlo, cr.nlomax
    for a, b in ((haa, rh), (loa[:mn], rl[:mn]), (lolo[:mn, :mn], rll[:mn, :mn]), (oalo[:, :nl], ro[:, :nl]),
                 (ololo[:nl, :nl], roo[:nl, :nl])):
        assert np.abs(a - b).max() <= 1e-12 * max(np.abs(b).max(), 1e-300)
    ctx.close()
