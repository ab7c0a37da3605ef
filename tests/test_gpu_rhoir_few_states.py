"""The interstitial density on large grids around the number of states from which the DFT products take
over from the batched FFT: 60^3 points with a basis that fills its share of the grid and one far
smaller, a slab of 18 x 75 x 75, two k-points of unequal bases; the same context changing
between the two routes and back.

Bar as test_gpu_rhoir_edges.py: 64 eps nst of the density that numpy's FFT gives."""
import numpy as np
import pytest

from test_gpu_rhoir_edges import _crystal, _ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell,n,share,states", [((42.0, 42.0, 42.0), 13000, 1.0, (1, 6, 12, 1)),
                                                 ((42.0, 42.0, 42.0), 13000, 0.15, (1, 2, 1)),
                                                 ((12.0, 52.5, 52.5), 5800, 1.0, (3, 9, 3))])
def test_few_states(cell, n, share, states):
    import torch
    from exciting_amd import lapw
    w = _crystal(cell, n)
    cr, kp = w.crystal, w.kpoints[0]
    rng = np.random.default_rng(n)
    order = np.argsort(kp.gpc[:kp.ngp], kind="stable")
    bases = [np.ascontiguousarray(np.sort(kp.igpig[:kp.ngp][order[:max(1, int(kp.ngp * s))]])) for s in (share, 0.8 * share)]
    ctx = lapw.Context(cr)
    for nst in states:
        rho = torch.full((cr.ngrtot,), 0.25, dtype=torch.float64, device="cuda")
        ref = np.zeros(cr.ngrtot)
        for ig in bases:
            c = (rng.standard_normal((nst, ig.size)) + 1j * rng.standard_normal((nst, ig.size))) / np.sqrt(2.0 * ig.size)
            occ = rng.uniform(0.1, 2.0, nst)
            print(f"rhoir {cell}, basis {ig.size}, {nst} states", flush=True)
            dig, dc, do = (torch.from_numpy(x).cuda() for x in (ig, c, occ))
            ctx._call("exc_genrhoir_dev", ctx.h, ig.size, dig.data_ptr(), nst, c.shape[1], dc.data_ptr(), do.data_ptr(),
                      0.35, 1e-8, rho.data_ptr())
            torch.cuda.synchronize()
            ref += _ref(cr, ig, c, occ, 0.35)
        err = np.abs(rho.cpu().numpy() - 0.25 - ref).max()
        assert err <= 64 * 2.2e-16 * max(nst, 4) * max(np.abs(ref).max(), 1.0)
    ctx.close()
