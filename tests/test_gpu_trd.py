"""The tridiagonal reduction of the grouped eigensolve (k_trd.hip) at the orders where it changes:
the smallest, around its panels of 32 columns, its 64-row workgroups and the 64-reflector blocks of
the back-transform, batches of unequal orders; and matrices it has nothing to do on (diagonal),
with zero subdiagonal blocks, and real ones.

Bars, as test_gpu_eigen.py: eigenvalues within 1e-10 of LAPACK's, the residual |H C - O C e| and
|C^H O C - 1| within 1e-10 of the norm of H (all pairs of the order asked for)."""
import numpy as np
import pytest

from conftest import small

pytestmark = pytest.mark.gpu


def _pair(rng, n, kind):
    x = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    h = 0.5 * (x + x.conj().T)
    y = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(2 * n)
    o = np.eye(n) + 0.1 * (y + y.conj().T)
    if kind == "diagonal":
        return np.diag(rng.uniform(-2, 2, n)).astype(complex), np.eye(n, dtype=complex)
    if kind == "blocks":                       # exactly decoupled: zero columns above the subdiagonal
        h[: n // 2, n // 2:] = 0.0
        h[n // 2:, : n // 2] = 0.0
        o = np.eye(n, dtype=complex)
    if kind == "real":
        return h.real.astype(complex), o.real.astype(complex)
    return h, o


@pytest.mark.parametrize("sizes,kind", [([1, 2, 3], "plain"), ([4, 31, 32], "plain"), ([33, 34, 63], "plain"),
                                        ([64, 65, 66], "plain"), ([97, 96], "plain"), ([128, 130, 5], "plain"),
                                        ([70, 40], "diagonal"), ([75, 130], "blocks"), ([66, 67], "real"), ([193], "plain")])
def test_tridiagonal_orders(sizes, kind):
    import scipy.linalg
    import torch
    from exciting_amd import lapw
    rng = np.random.default_rng(sum(sizes))
    ctx = lapw.Context(small("a").crystal)
    pairs = [_pair(rng, n, kind) for n in sizes]
    nev = min(sizes)
    dev = [[torch.from_numpy(np.ascontiguousarray(m.T)).cuda() for m in p] for p in pairs]
    evs = [torch.zeros(nev, dtype=torch.float64, device="cuda") for _ in sizes]
    vecs = [torch.zeros((nev, n), dtype=torch.complex128, device="cuda") for n in sizes]
    print(f"tridiagonal reduction {sizes} {kind}", flush=True)
    ctx.eigen_batched_dev(sizes, [d[0] for d in dev], [d[1] for d in dev], nev, evs, vecs)
    torch.cuda.synchronize()
    for (h, o), e, c in zip(pairs, evs, vecs):
        e, c = e.cpu().numpy(), c.cpu().numpy().T
        ref = scipy.linalg.eigh(h, o, eigvals_only=True, subset_by_index=[0, nev - 1])
        assert np.abs(e - ref).max() <= 1e-10
        scale = max(1.0, np.linalg.norm(h))
        assert np.linalg.norm(h @ c - (o @ c) * e) <= 1e-10 * scale
        assert np.linalg.norm(c.conj().T @ o @ c - np.eye(nev)) <= 1e-10 * scale
    ctx.close()
