"""The grouped eigensolve's Cholesky factor and inverse (k_chol.hip) around its blocks of 16 and 64
columns, alone and in batches of unequal orders, with O graded over 8 decades, and with O whose
leading minor of a given order is the first that is not positive (LAPACK's info, order + minor).

Bars, as test_gpu_trd.py: eigenvalues within 1e-10 of LAPACK's, residual and O-orthonormality within 1e-10
of the norm of H; for the graded O, D O D with its D^-1 H D^-1 scaled alike, whose eigenvalues are those of the
pair it comes from, within 1e-10 too (Cholesky does not see a diagonal scaling)."""
import numpy as np
import pytest

from conftest import small

pytestmark = pytest.mark.gpu


def _pair(rng, n, kind):
    x = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    h = 0.5 * (x + x.conj().T)
    y = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(2 * n)
    o = np.eye(n) + 0.1 * (y + y.conj().T)
    if kind == "graded":
        s = np.logspace(-4, 4, n)
        rng.shuffle(s)
        return h * s[:, None] * s, o * s[:, None] * s, h, o
    return h, o, h, o


def _solve(pairs, nev):
    import torch
    from exciting_amd import lapw
    ctx = lapw.Context(small("a").crystal)
    sizes = [h.shape[0] for h, _ in pairs]
    dev = [[torch.from_numpy(np.ascontiguousarray(m.T)).cuda() for m in p] for p in pairs]
    evs = [torch.zeros(nev, dtype=torch.float64, device="cuda") for _ in sizes]
    vecs = [torch.zeros((nev, n), dtype=torch.complex128, device="cuda") for n in sizes]
    try:
        ctx.eigen_batched_dev(sizes, [d[0] for d in dev], [d[1] for d in dev], nev, evs, vecs)
        torch.cuda.synchronize()
    finally:
        ctx.close()
    return [e.cpu().numpy() for e in evs], [v.cpu().numpy().T for v in vecs]


@pytest.mark.parametrize("sizes,kind", [([1], "plain"), ([2, 15], "plain"), ([16, 17, 31], "plain"), ([47, 48, 49], "plain"),
                                        ([63, 64, 65], "plain"), ([80, 81], "plain"), ([127, 128, 129], "plain"),
                                        ([200, 33], "graded"), ([257], "plain"), ([64, 130], "graded")])
def test_cholesky_orders(sizes, kind):
    import scipy.linalg
    rng = np.random.default_rng(sum(sizes) + 1)
    quad = [_pair(rng, n, kind) for n in sizes]
    nev = min(sizes)
    print(f"Cholesky and inverse {sizes} {kind}", flush=True)
    evs, vecs = _solve([q[:2] for q in quad], nev)
    for (h, o, h0, o0), e, c in zip(quad, evs, vecs):
        ref = scipy.linalg.eigh(h0, o0, eigvals_only=True, subset_by_index=[0, nev - 1])
        assert np.abs(e - ref).max() <= 1e-10
        scale = max(1.0, np.linalg.norm(h0))
        s = np.sqrt(np.abs(np.diag(o) / np.diag(o0)))
        c = c * s[:, None]
        assert np.linalg.norm(h0 @ c - (o0 @ c) * e) <= 1e-10 * scale
        assert np.linalg.norm(c.conj().T @ o0 @ c - np.eye(nev)) <= 1e-10 * scale


@pytest.mark.parametrize("n,minor", [(5, 1), (40, 16), (40, 17), (70, 64), (70, 65), (150, 100), (150, 150)])
def test_not_positive_definite(n, minor):
    from exciting_amd import lapw
    rng = np.random.default_rng(n + minor)
    h, o, _, _ = _pair(rng, n, "plain")
    o[minor - 1, minor - 1] = -0.5
    print(f"O of order {n}, minor {minor} not positive", flush=True)
    good = _pair(rng, 60, "plain")[:2]
    with pytest.raises(lapw.ExcError) as ei:
        _solve([good, (h, o)], 2)
    assert ei.value.code == n + minor
