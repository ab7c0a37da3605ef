"""Device memory of the FP64 path's exact integer products: fewer k-points share the workspace where
less memory is free, with the same bits; where one k-point's would be more than half of it the batch
runs on the FP64 MFMA tiles, and exc_ctx_exact_products says so; another allocation of the context
that would fail gets the workspace back."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = (1290, 1301, 1279)
# a k-point's planes and residues at 16 atoms, lmax 10: 64 x 3904 x 1536 + 21 x 32 x 65536 bytes
ONE = 64 * 3904 * 1536 + 21 * 32 * 65536
REST = 16 * 3872 * sum(SIZES) + (32 << 20)           # the Y workspace, radial factors and lists


@pytest.fixture(scope="module")
def load():
    from exciting_amd import synth
    a = (215.0 * 16) ** (1.0 / 3.0)
    w = synth.make_small(natm_per_species=(8, 8), lmax=10, lorbl=(0, 1), n_target=1400, nk=1, seed=4,
                         cell=(0.95 * a, a, a / 0.95), rmt=(1.6, 1.5))
    rng = np.random.default_rng(4)
    kps = [synth.make_kpoint(w.crystal, rng, n, None) for n in SIZES]
    m = max(k.ngp for k in kps)
    return w.crystal, [synth.pad_kpoint(k, m) for k in kps]


def _leave(free):
    """Tensors that leave about `free` bytes of the device memory (what is reported as free settles
    once memory has been written, hence two steps)."""
    import torch
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    hog = []
    for rest in (free + (1 << 30), free):
        hog.append(torch.zeros(torch.cuda.mem_get_info()[0] - rest, dtype=torch.uint8, device="cuda"))
        torch.cuda.synchronize()
    return hog


def _flags():
    from exciting_amd import lapw
    return lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE | lapw.EXC_BATCH_GRAPH


def _run(ctx, b):
    import torch
    for t in b.H + b.O:
        t.fill_(float("nan"))
    torch.cuda.synchronize()
    ctx.setup_batched_dev(b, _flags())
    torch.cuda.synchronize()


def test_less_free_memory(load):
    import torch
    from exciting_amd import lapw
    cr, kps = load
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, kps)
    ref = {}
    for name, variant in (("exact", -1), ("tiles", 0)):
        ctx = lapw.Context(cr, stream=s)
        ctx.set_variant("bmt", variant)
        _run(ctx, b)
        assert ctx.exact_products() == (name == "exact")
        ref[name] = [t.clone() for t in b.H + b.O]
        ctx.close()
    assert not torch.equal(ref["exact"][0], ref["tiles"][0])
    # an eighth of what is free holds one k-point's or less; a half of it holds less than one's
    for name, free in (("exact", REST + 5 * ONE), ("tiles", REST + ONE + ONE // 2)):
        ctx = lapw.Context(cr, stream=s)
        hog = _leave(free)
        print(f"{torch.cuda.mem_get_info()[0] >> 20} MiB free of {free >> 20}: {name}", flush=True)
        _run(ctx, b)
        del hog
        torch.cuda.empty_cache()
        assert ctx.exact_products() == (name == "exact")
        for x, y in zip(b.H + b.O, ref[name]):
            assert torch.equal(x, y)
        ctx.status()
        ctx.close()


def test_workspace_given_back(load):
    import torch
    from exciting_amd import lapw
    cr, kps = load
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    n, nb, nev = 900, 8, 4
    g = torch.Generator(device="cuda").manual_seed(1)
    H = []
    for _ in range(nb):
        x = torch.randn(n, n, dtype=torch.complex128, device="cuda", generator=g)
        H.append((x + x.conj().T).contiguous())
    one = torch.eye(n, dtype=torch.complex128, device="cuda")
    ev = [torch.zeros(nev, dtype=torch.float64, device="cuda") for _ in H]
    vec = [torch.zeros((nev, n), dtype=torch.complex128, device="cuda") for _ in H]
    ref = [torch.linalg.eigvalsh(h.cpu())[:nev] for h in H]
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, kps)
    _run(ctx, b)
    first = [t.clone() for t in b.H + b.O]
    assert ctx.exact_products()
    batch = 3 * 16 * n * n * nb                       # the grouped solve's padded matrices
    hog = _leave(batch - (64 << 20))
    print("eigensolve with the exact products' workspace held", flush=True)
    ctx.eigen_batched_dev([n] * nb, H, [one] * nb, nev, ev, vec)
    torch.cuda.synchronize()
    for e, r in zip(ev, ref):
        assert (e.cpu() - r).abs().max() <= 1e-10 * max(1.0, r.abs().max())
    del hog
    torch.cuda.empty_cache()
    print("the batch again", flush=True)
    _run(ctx, b)
    assert ctx.exact_products()
    for x, y in zip(b.H + b.O, first):
        assert torch.equal(x, y)
    ctx.close()


def test_workspace_in_a_graph_of_the_callers(load):
    """A graph the caller records around an eager call holds the workspace's addresses: an allocation
    that does not fit then fails, and the graph's replays keep their bits."""
    import torch
    from exciting_amd import lapw
    cr, kps = load
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    flags = lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, kps)
        ctx.setup_batched_dev(b, flags)
        torch.cuda.synchronize()
        assert ctx.exact_products()
        first = [t.clone() for t in b.H + b.O]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        ctx.setup_batched_dev(b, flags)
    # the adjoint's workspace, 16 (2 nst natm naa + 3 nst ngp) bytes, is allocated at its first call
    d, nst = b.dks[0], 4000
    C = torch.zeros((nst, b.nmat[0]), dtype=torch.complex128, device="cuda")
    wt = torch.zeros(nst, dtype=torch.float64, device="cuda")
    dt = torch.zeros((cr.natm, 3), dtype=torch.float64, device="cuda")
    dv = torch.zeros(cr.ngvec, dtype=torch.complex128, device="cuda")
    hog = _leave(100 << 20)
    print("an adjoint that does not fit, beside a recorded graph", flush=True)
    with pytest.raises(lapw.ExcError) as ei:
        ctx.vjp_dev(d.ngp, d.ngkmax, b.apw[0], d.igpig, d.vgpc, d.sfacgp, C, b.nmat[0], nst, wt, wt, dt, dv)
    assert ei.value.code == lapw.EXC_ERR_HIP
    del hog
    torch.cuda.empty_cache()
    for i in range(3):
        for t in b.H + b.O:
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        print(f"replay {i}", flush=True)
        g.replay()
        torch.cuda.synchronize()
        for x, y in zip(b.H + b.O, first):
            assert torch.equal(x, y)
    ctx.close()
