"""The Gram form's table (k_gram.hip) at the orders it meets: naa = 2 (lmax + 1)^2 from 8 to 338 (one
to six 64-row chunks, orders that are no multiple of the 16-column panel), h_a indefinite,
positive definite, with a repeated smallest eigenvalue, diagonal (no off-diagonal element to
reduce), and not finite.

sigma against numpy's eigenvalues to 1e-12 max(1, |min lambda|) (the bar of test_gpu_crt.py), the
form the library reports, and H against the oracle's within the split's own bar (1e-9 relative,
as test_gpu_crt.py holds it)."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _h(kind, rng, n, natm, haa):
    out = haa.copy()
    for a in range(natm):
        if kind == "positive":
            out[:, :, a] += 3.0 * np.eye(n)
        elif kind == "diagonal":
            out[:, :, a] = np.diag(rng.uniform(-0.5, 4.0, n))
        elif kind == "repeated":
            q, _ = np.linalg.qr(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)))
            lam = rng.uniform(0.0, 6.0, n)
            lam[:3] = -1.25
            h = (q * lam) @ q.conj().T
            out[:, :, a] = 0.5 * (h + h.conj().T)
    return out


@pytest.mark.parametrize("lmax,kind", [(1, "plain"), (2, "diagonal"), (3, "plain"), (5, "repeated"), (7, "positive"),
                                       (8, "diagonal"), (10, "repeated"), (11, "plain"), (12, "plain")])
def test_gram_table(lmax, kind):
    import torch
    from exciting_amd import lapw, synth
    from oracle import lapw_ref as R
    w = synth.make_small(natm_per_species=(1, 2), lmax=lmax, lorbl=(0, 1), n_target=70, nk=1, seed=31 + lmax)
    rng = np.random.default_rng(lmax)
    cr = dataclasses.replace(w.crystal, haa=_h(kind, rng, w.crystal.maxaa, w.crystal.natm, w.crystal.haa))
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, w.kpoints)
        print(f"Gram table lmax={lmax} {kind}", flush=True)
        ctx.set_variant("crtform", 1)
        ctx.setup_batched_dev(b, lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_SPLIT_CRT | lapw.EXC_BATCH_OLP_LEGENDRE)
        torch.cuda.synchronize()
    form, nmod, sigma = ctx.crt_form()
    lam = [np.linalg.eigvalsh(cr.haa[:, :, a]) for a in range(cr.natm)]
    lmin, lmax_ = min(x[0] for x in lam), max(np.abs(x).max() for x in lam)
    ref = max(0.0, -lmin) * (1 + 1e-6) + 1e-10 * lmax_
    H_ref, _, _ = R.setup(cr, w.kpoints[0])
    eh = np.linalg.norm(b.H[0].cpu().numpy().T - H_ref) / np.linalg.norm(H_ref)
    print(f"sigma {sigma:.12f} (min lambda {lmin:.6f}), |dH|/|H| {eh:.2e}", flush=True)
    assert form == 1 and nmod == 10
    assert abs(sigma - ref) <= 1e-12 * max(1.0, abs(lmin))
    assert eh <= 1e-9
    ctx.close()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_gram_not_finite(bad):
    """An h_a that is not finite leaves the Gram form unused (no table), as before."""
    import torch
    from exciting_amd import lapw, synth
    w = synth.make_small(natm_per_species=(1, 1), lmax=3, lorbl=(0,), n_target=40, nk=1, seed=9)
    haa = w.crystal.haa.copy()
    haa[2, 2, 1] = bad
    cr = dataclasses.replace(w.crystal, haa=haa)
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, w.kpoints)
        ctx.setup_batched_dev(b, lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_SPLIT_CRT | lapw.EXC_BATCH_OLP_LEGENDRE)
        torch.cuda.synchronize()
    assert ctx.crt_form()[:2] == (0, 11)
    ctx.close()
