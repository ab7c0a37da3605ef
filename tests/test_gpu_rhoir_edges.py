"""The interstitial density's DFT products (k_rhoir.hip) at the edges of their 16-wide tiles: grids
longer and shorter than one tile an edge and unequal ones up to the largest that take this route
(80) and the first that does not; bases of one function, of a line of G, and of every G of the box; states that
do not count, more k-points than one launch takes, results added over two calls.

Bar: within 64 eps nst of the density that numpy's FFT gives, relative to its largest value, as
test_gpu_rhovalk_edges.py (positive terms; the transform's rounding is a few eps of psi's norm)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _crystal(cell, n):
    from exciting_amd import synth
    return synth.make_small(natm_per_species=(1,), lmax=2, lorbl=(0,), n_target=n, nk=1, seed=5, cell=cell)


def _ref(cr, igpig, c, occ, w):
    n = [int(cr.intgv[i, 1] - cr.intgv[i, 0] + 1) for i in range(3)]
    j = [np.mod(cr.ivg[i].astype(np.int64)[igpig - 1], n[i]) for i in range(3)]
    at = j[0] + n[0] * (j[1] + n[1] * j[2])
    rho = np.zeros(cr.ngrtot)
    for s in range(c.shape[0]):
        z = np.zeros(cr.ngrtot, complex)
        z[at] = c[s]
        psi = np.fft.ifftn(z.reshape(n[::-1])).ravel() * cr.ngrtot
        if abs(w * occ[s]) > 1e-8:
            rho += w * occ[s] / cr.omega * np.abs(psi) ** 2
    return rho


@pytest.mark.parametrize("cell,n,basis,nst", [((5.0, 5.5, 6.0), 9, "all", 1), ((6.0, 6.5, 7.0), 40, "k", 7),
                                              ((7.0, 9.0, 22.0), 120, "k", 9), ((30.0, 6.0, 7.0), 150, "line", 17),
                                              ((6.0, 30.0, 9.0), 150, "one", 3), ((12.0, 13.0, 14.0), 300, "all", 10),
                                              ((5.0, 6.0, 56.0), 220, "k", 65), ((56.0, 5.0, 6.0), 220, "k", 5),
                                              ((5.0, 56.0, 6.0), 220, "k", 33), ((5.0, 6.0, 60.0), 220, "k", 4)])
def test_rhoir_grids(cell, n, basis, nst):
    import torch
    from exciting_amd import lapw
    w = _crystal(cell, n)
    cr, kp = w.crystal, w.kpoints[0]
    rng = np.random.default_rng(n)
    grid = [int(cr.intgv[i, 1] - cr.intgv[i, 0] + 1) for i in range(3)]
    ig = {"k": kp.igpig[:kp.ngp], "one": kp.igpig[:1], "all": np.arange(1, cr.ngrtot + 1, dtype=np.int32),
          "line": np.flatnonzero((cr.ivg[1] == cr.ivg[1, 3]) & (cr.ivg[2] == cr.ivg[2, 3])).astype(np.int32) + 1}[basis]
    ig = np.ascontiguousarray(ig, dtype=np.int32)
    c = (rng.standard_normal((nst, ig.size + 2)) + 1j * rng.standard_normal((nst, ig.size + 2))) / np.sqrt(2.0 * ig.size)
    occ = rng.uniform(0.1, 2.0, nst)
    if nst > 3:
        occ[2] = 0.0
        occ[3] *= -1.0
    print(f"rhoir grid {grid}, basis {basis} of {ig.size}, {nst} states", flush=True)
    ctx = lapw.Context(cr)
    dig, dc, do = torch.from_numpy(ig).cuda(), torch.from_numpy(c).cuda(), torch.from_numpy(occ).cuda()
    rho = torch.full((cr.ngrtot,), 0.5, dtype=torch.float64, device="cuda")
    for _ in range(2):
        ctx._call("exc_genrhoir_dev", ctx.h, ig.size, dig.data_ptr(), nst, c.shape[1], dc.data_ptr(), do.data_ptr(),
                  0.35, 1e-8, rho.data_ptr())
    torch.cuda.synchronize()
    ref = _ref(cr, ig, c[:, :ig.size], occ, 0.35)
    got = 0.5 * (rho.cpu().numpy() - 0.5)
    err = np.abs(got - ref).max()
    print(f"largest difference {err / np.abs(ref).max():.2e}", flush=True)
    assert err <= 64 * 2.2e-16 * max(nst, 4) * max(np.abs(ref).max(), 1.0)
    ctx.close()


def test_rhoir_many_kpoints():
    """18 k-points of unequal bases in one call (16 a launch)."""
    import torch
    from exciting_amd import lapw, synth
    w = _crystal((8.0, 8.5, 9.0), 90)
    cr, rng = w.crystal, np.random.default_rng(1)
    kps = [synth.make_kpoint(cr, rng, int(m), None) for m in rng.integers(20, 90, 18)]
    top = max(k.ngp for k in kps)
    kps = [synth.pad_kpoint(k, top) for k in kps]
    nst = 11
    c = [rng.standard_normal((nst, k.ngp + cr.nlotot)) + 1j * rng.standard_normal((nst, k.ngp + cr.nlotot)) for k in kps]
    occ, wk = [rng.uniform(0.0, 2.0, nst) for _ in kps], rng.uniform(0.01, 0.1, len(kps))
    ctx = lapw.Context(cr)
    b = lapw.DeviceBatch(cr, kps)
    rho = torch.zeros(cr.ngrtot, dtype=torch.float64, device="cuda")
    print("rhoir 18 k-points", flush=True)
    dev = lambda a: [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in a]
    ctx.genrhoir_batched_dev(b, nst, dev(c), dev(occ), list(wk), rho)
    torch.cuda.synchronize()
    ref = sum(_ref(cr, k.igpig[:k.ngp], x[:, :k.ngp], o, float(v)) for k, x, o, v in zip(kps, c, occ, wk))
    assert np.abs(rho.cpu().numpy() - ref).max() <= 64 * 2.2e-16 * nst * np.abs(ref).max()
    ctx.close()
