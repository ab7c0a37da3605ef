"""The tridiagonal reduction of the grouped eigensolve (k_trd.hip) and the Gram table (k_gram.hip) on
matrices with columns whose squares underflow: blocks coupled by 1e-149, 1e-156 and 1e-170, a
diagonal with off-diagonal elements of 1e-160, and a coupling that is imaginary alone.

Bars, as test_gpu_trd.py: eigenvalues within 1e-10 of LAPACK's (of the matrix without the tiny
elements: they move an eigenvalue by no more than their norm), |H C - O C e| and |C^H C - 1| within
1e-10 of the norm of H."""
import dataclasses

import numpy as np
import pytest

from conftest import small

pytestmark = pytest.mark.gpu


def _matrix(rng, n, kind):
    x = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    h, t = 0.5 * (x + x.conj().T), rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    t = t + t.conj().T
    if kind == "diagonal":
        return np.diag(np.linspace(-2.0, 2.0, n)) + 1e-160 * (t - np.diag(np.diag(t)))
    m = n // 2
    h[:m, m:] = 0.0
    if kind == "imaginary":
        h[m - 1, m] = 1e-165j
    else:
        h[:m, m:] = float(kind) * t[:m, m:]
    h[m:, :m] = h[:m, m:].conj().T
    return h


@pytest.mark.parametrize("sizes", [(7, 66), (97, 130)])
@pytest.mark.parametrize("kind", ["1e-149", "1e-156", "1e-170", "imaginary", "diagonal"])
def test_tiny_columns(sizes, kind):
    import torch
    from exciting_amd import lapw
    rng = np.random.default_rng(sum(sizes))
    ctx = lapw.Context(small("a").crystal)
    hs = [_matrix(rng, n, kind) for n in sizes]
    nev = min(sizes)
    dev = [torch.from_numpy(np.ascontiguousarray(h.T)).cuda() for h in hs]
    one = [torch.eye(n, dtype=torch.complex128, device="cuda") for n in sizes]
    evs = [torch.zeros(nev, dtype=torch.float64, device="cuda") for _ in sizes]
    vecs = [torch.zeros((nev, n), dtype=torch.complex128, device="cuda") for n in sizes]
    print(f"tiny columns {sizes} {kind}", flush=True)
    ctx.eigen_batched_dev(list(sizes), dev, one, nev, evs, vecs)
    torch.cuda.synchronize()
    for h, e, c in zip(hs, evs, vecs):
        e, c = e.cpu().numpy(), c.cpu().numpy().T
        h = np.where(np.abs(h) < 1e-140, 0.0, h)
        scale = max(1.0, np.linalg.norm(h))
        assert np.abs(e - np.linalg.eigvalsh(h)[:nev]).max() <= 1e-10
        assert np.linalg.norm(h @ c - c * e) <= 1e-10 * scale
        assert np.linalg.norm(c.conj().T @ c - np.eye(nev)) <= 1e-10 * scale
    ctx.close()


@pytest.mark.parametrize("kind", ["1e-156", "1e-170", "imaginary", "diagonal"])
def test_gram_table_of_tiny_columns(kind):
    """The table is made, with the shift of the matrix without the tiny elements (bar of test_gpu_gram.py)."""
    import torch
    from exciting_amd import lapw, synth
    w = synth.make_small(natm_per_species=(1, 1), lmax=3, lorbl=(0,), n_target=40, nk=1, seed=9)
    rng, haa = np.random.default_rng(5), w.crystal.haa.copy()
    for a in range(w.crystal.natm):
        haa[:, :, a] = _matrix(rng, haa.shape[0], kind)
    cr = dataclasses.replace(w.crystal, haa=haa)
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    ctx.set_variant("crtform", 1)
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, w.kpoints)
        print(f"Gram table of tiny columns {kind}", flush=True)
        ctx.setup_batched_dev(b, lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_SPLIT_CRT | lapw.EXC_BATCH_OLP_LEGENDRE)
        torch.cuda.synchronize()
    form, _, sigma = ctx.crt_form()
    lam = [np.linalg.eigvalsh(np.where(np.abs(haa[:, :, a]) < 1e-140, 0.0, haa[:, :, a])) for a in range(cr.natm)]
    lmin, lmax = min(x[0] for x in lam), max(np.abs(x).max() for x in lam)
    assert form == 1
    assert abs(sigma - (max(0.0, -lmin) * (1 + 1e-6) + 1e-10 * lmax)) <= 1e-12 * max(1.0, abs(lmin))
    ctx.close()
