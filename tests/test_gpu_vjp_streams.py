"""The adjoint adds to dE/dtau and dE/dV(G): contexts on streams of their own may add their
k-points to the same two arrays at once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_two_contexts_add_to_the_same_arrays():
    """200 calls on each of two streams against 400 times one call's result: equal to rounding
    (400 additions, each to half an ulp of a sum that grows evenly; the bar allows every one of
    them an ulp and the per-call sums 1e-13); one lost addition alone would be 1/400."""
    import torch
    from exciting_amd import lapw, synth
    w = synth.make_small(natm_per_species=(1, 1), lmax=3, lorbl=(0, 1), n_target=60, nk=1, seed=8, cell=(8.0, 8.5, 9.0))
    cr, kp = w.crystal, w.kpoints[0]
    rng = np.random.default_rng(2)
    nst, nmat, calls = 9, kp.ngp + cr.nlotot, 200
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    C = dev((rng.standard_normal((nst, nmat)) + 1j * rng.standard_normal((nst, nmat))) / np.sqrt(2.0 * kp.ngp))
    wh, wo = dev(rng.uniform(0.5, 2.0, nst)), dev(rng.uniform(-2.0, 2.0, nst))
    d = lapw.DeviceKPoint(kp)
    streams = [torch.cuda.Stream() for _ in range(2)]
    ctxs = [lapw.Context(cr, stream=s) for s in streams]
    apw = lapw.alloc_apwalm_dev(cr, d.ngkmax, "cuda")
    ctxs[0].match_dev(d.ngp, d.ngkmax, d.gpc, d.tpgpc, d.sfacgp, apw)
    new = lambda: (torch.zeros((cr.natm, 3), dtype=torch.float64, device="cuda"),
                   torch.zeros(cr.ngvec, dtype=torch.complex128, device="cuda"))
    torch.cuda.synchronize()
    add = lambda c, out: c.vjp_dev(d.ngp, d.ngkmax, apw, d.igpig, d.vgpc, d.sfacgp, C, nmat, nst, wh, wo, *out)
    one, both = new(), new()
    torch.cuda.synchronize()
    print("adjoint: one call, then two streams", flush=True)
    warm = [new(), new()]                            # workspaces are made at the first call
    torch.cuda.synchronize()
    for c, out in zip(ctxs, warm):
        add(c, out)
    torch.cuda.synchronize()
    add(ctxs[0], one)
    torch.cuda.synchronize()
    for _ in range(calls):
        for c in ctxs:
            add(c, both)
    torch.cuda.synchronize()
    for x, y in zip(both, one):
        err = (x - 2 * calls * y).abs().max().item()
        assert err <= (2 * calls * 2.2e-16 + 1e-13) * 2 * calls * y.abs().max().item()
    for c in ctxs:
        c.status()
        c.close()
