"""The FP64 path's exact integer products (the muffin-tin contraction of large batches: 16 moduli,
57-bit integers, k_crt.hip) against the FP64 MFMA tiles (EXC_STAGE_BMT pinned) and the oracle.

* H (and O without the addition theorem) within 1e-14 of the MFMA tiles' norm, the bar between
  the FP64 summation orders, and 1e-12 of the oracle's; uneven sizes, bases that are no multiple
  of the 128- and 256-wide tiles, with the match and on the caller's apwalm;
* rows the integers do not take (NaN, infinity, norms whose square over- or underflows): the
  same NaN and infinity pattern as the MFMA tiles, the other elements as above;
* a batch whose residue planes are more than the workspace holds at a time: the same k-point in
  every group gives the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _workload(nk, sizes, natm=(12, 12), lmax=10, seed=3):
    from exciting_amd import synth
    n = sum(natm)
    a = (215.0 * n) ** (1.0 / 3.0)
    w = synth.make_small(natm_per_species=natm, lmax=lmax, lorbl=(0, 1), n_target=max(sizes) + 90, nk=1, seed=seed,
                         cell=(0.95 * a, a, a / 0.95), rmt=(1.6, 1.5))
    rng = np.random.default_rng(seed)
    kps = [synth.make_kpoint(w.crystal, rng, n, None) for n in sizes]
    m = max(k.ngp for k in kps)
    return w.crystal, [synth.pad_kpoint(k, m) for k in kps]


def _run(ctx, b, flags, variant):
    import torch
    ctx.set_variant("bmt", variant)
    for t in b.H + b.O:
        t.fill_(float("nan"))
    ctx.setup_batched_dev(b, flags)
    torch.cuda.synchronize()
    return [(h.clone(), o.clone()) for h, o in zip(b.H, b.O)]


def _near(x, ref, tol=1e-14):
    import torch
    return (torch.linalg.norm(x - ref) / torch.linalg.norm(ref)).item() <= tol


@pytest.mark.parametrize("sizes,natm,lmax", [((1279, 1281), (12, 12), 10), ((2050, 1400), (8, 8), 10)])
def test_exact_products(sizes, natm, lmax):
    import torch
    from exciting_amd import lapw
    from oracle import lapw_ref as R
    cr, kps = _workload(2, sizes, natm, lmax)
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, kps)
        for name, flags in (("addition theorem", lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE),
                            ("graph", lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE | lapw.EXC_BATCH_GRAPH),
                            ("both matrices", lapw.EXC_BATCH_MATCH), ("caller's apwalm", 0)):
            print(f"exact products {sizes} K={cr.natm * cr.maxaa}: {name}", flush=True)
            ref = _run(ctx, b, flags, 0)
            got = _run(ctx, b, flags, -1)
            for (h, o), (h0, o0) in zip(got, ref):
                assert not torch.equal(h, h0)          # the other route did run
                assert _near(h, h0) and _near(o, o0)
                il = torch.tril_indices(*h.shape, -1)
                for m in (h, o):                       # the strict triangles are conjugates bit for bit
                    assert torch.equal(m[il[0], il[1]], m[il[1], il[0]].conj())
    H_ref, O_ref, _ = R.setup(cr, kps[1])
    for m, r in zip((x[1].cpu().numpy().T for x in (b.H, b.O)), (H_ref, O_ref)):
        assert np.linalg.norm(m - r) <= 1e-12 * np.linalg.norm(r)
    ctx.status()
    ctx.close()


def test_exact_products_rows_left_to_mfma():
    import torch
    from exciting_amd import lapw
    cr, kps = _workload(2, (1290, 1301))
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    flags = lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, kps)
        for i, (row, f) in enumerate(((5, float("nan")), (700, float("inf")))):
            b.dks[i].sfacgp[:, row] *= f
        b.dks[0].tpgpc[40, 0] = float("nan")
        b.dks[1].sfacgp[:, 64] *= 1e200
        b.dks[1].sfacgp[:, 1300] *= 1e-200
        print("exact products: rows left to the MFMA tiles", flush=True)
        ref = _run(ctx, b, flags, 0)
        got = _run(ctx, b, flags, -1)
    for k, ((h, _), (h0, _)) in enumerate(zip(got, ref)):
        for x, y in ((h.real, h0.real), (h.imag, h0.imag)):
            assert torch.equal(x.isnan(), y.isnan()) and torch.equal(x.isinf(), y.isinf())
        fin = torch.isfinite(h0.real) & torch.isfinite(h0.imag)
        # the marked rows by themselves (they come from the same tiles), the others by their norm
        rows = [5, 40] if k == 0 else [64, 700, 1300]
        keep = torch.ones(h.shape[0], dtype=torch.bool, device=h.device)
        keep[rows] = False
        assert _near(h[keep][:, keep], h0[keep][:, keep])
        f = fin[rows]
        assert torch.equal(h[rows][f], h0[rows][f])
    ctx.close()


def test_exact_products_in_groups():
    import torch
    from exciting_amd import lapw
    cr, kps = _workload(1, (1270,))
    # planes: 2 operands x 2 maps x 16 moduli x K bytes for each of 1280 rows; more than 24 GiB in all
    nk = int(24 * 2 ** 30 / (64 * cr.natm * cr.maxaa * 1280)) + 3
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, kps * nk)
        print(f"exact products: {nk} k-points in groups", flush=True)
        got = _run(ctx, b, lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE | lapw.EXC_BATCH_GRAPH, -1)
    for h, o in got[1:]:
        assert torch.equal(h, got[0][0]) and torch.equal(o, got[0][1])
    del got, b
    torch.cuda.empty_cache()
    ctx.close()
