"""The adjoint's tiles at their edges: exc_ho_vjp_dev against the oracle's VJP (dense D and W) to
the same 1e-9 relative bar as test_gpu_vjp.py, at bases around the 64-wide tiles, state counts
around 16, 32 and 64, and a cell long along one axis (few lines of G per tile: the sums per
difference in LDS) as well as small cubic ones (many short lines: added pair by pair)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nst,lmax,lo,cell", [(20, 1, 2, (0,), (7.0, 7.5, 8.0)), (64, 16, 3, (0, 1), (7.0, 7.5, 8.0)),
                                                (65, 33, 3, (0, 1, 1), (8.0, 8.5, 9.0)),
                                                (150, 65, 4, (0, 1), (6.0, 6.2, 40.0)),
                                                (130, 17, 4, (0, 2), (38.0, 6.0, 6.5)),
                                                (200, 31, 5, (0, 1), (6.0, 36.0, 6.5))])
def test_vjp_edges(n, nst, lmax, lo, cell):
    import torch
    from exciting_amd import lapw, synth
    from oracle import lapw_ref as R
    w = synth.make_small(natm_per_species=(1, 2), lmax=lmax, lorbl=lo, n_target=n, nk=1, seed=5 + n, cell=cell)
    cr, kp = w.crystal, w.kpoints[0]
    rng = np.random.default_rng(n)
    nmat = kp.ngp + cr.nlotot
    C = (rng.standard_normal((nmat, nst)) + 1j * rng.standard_normal((nmat, nst))) / np.sqrt(2.0 * n)
    wh, wo = rng.uniform(0.0, 2.0, nst), rng.uniform(-2.0, 2.0, nst)
    ref_t, ref_v = R.setup_vjp(cr, kp, (C * wh) @ C.conj().T, (C * wo) @ C.conj().T)
    ctx = lapw.Context(cr)
    d = lapw.DeviceKPoint(kp)
    apw = torch.from_numpy(np.ascontiguousarray(np.transpose(R.match(cr, kp), (3, 2, 1, 0)))).cuda()
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    dt = torch.zeros((cr.natm, 3), dtype=torch.float64, device="cuda")
    dv = torch.zeros(cr.ngvec, dtype=torch.complex128, device="cuda")
    print(f"adjoint N={kp.ngp} nst={nst} cell={cell}", flush=True)
    ctx.vjp_dev(kp.ngp, d.ngkmax, apw, d.igpig, d.vgpc, d.sfacgp, dev(C.T), nmat, nst, dev(wh), dev(wo), dt, dv)
    torch.cuda.synchronize()
    ctx.status()
    et = np.linalg.norm(dt.cpu().numpy().T - ref_t) / np.linalg.norm(ref_t)
    ev = np.linalg.norm(dv.cpu().numpy() - ref_v) / np.linalg.norm(ref_v)
    print(f"dE/dtau {et:.2e} dE/dV {ev:.2e}", flush=True)
    assert et <= 1e-9 and ev <= 1e-9
    ctx.close()
