"""The grouped setup's workspaces: what a batch that does not fit leaves behind."""
import pytest

from conftest import small

pytestmark = pytest.mark.gpu


def _too_large(b, nk=200, ngp=2_000_000):
    """nk descriptors of a basis whose Y workspace (16 natm naa ngp bytes each) is beyond the card's
    memory; refused while it is laid out, so its pointers (the small batch's) are never read."""
    from exciting_amd import lapw
    big = type("Batch", (), {})()
    big.nk, big.desc = nk, (lapw.KPointDev * nk)()
    for e in big.desc:
        for f, _ in lapw.KPointDev._fields_:
            setattr(e, f, getattr(b.desc[0], f))
        e.ngp = e.ngkmax = ngp
        e.ldh = ngp + 100
    return big


@pytest.mark.parametrize("graph", [False, True])
def test_batch_that_does_not_fit(graph):
    """It is refused, and the batch before it, whose Y workspace was given up for it, then gives
    the same bits as at first (its tables are laid out again)."""
    import torch
    from exciting_amd import lapw
    w = small("b")
    s = torch.cuda.Stream()
    ctx = lapw.Context(w.crystal, stream=s)
    flags = lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE | (lapw.EXC_BATCH_GRAPH if graph else 0)
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(w.crystal, w.kpoints)
        ctx.setup_batched_dev(b, flags)
        torch.cuda.synchronize()
        first = [t.clone() for t in b.H + b.O]
        for t in b.H + b.O:
            t.fill_(float("nan"))
        print(f"batch beyond the memory, graph {graph}", flush=True)
        with pytest.raises(lapw.ExcError) as ei:
            ctx.setup_batched_dev(_too_large(b), flags)
        assert ei.value.code == lapw.EXC_ERR_HIP
        print("the small batch again", flush=True)
        ctx.setup_batched_dev(b, flags)
        torch.cuda.synchronize()
    for x, y in zip(first, b.H + b.O):
        assert torch.equal(x, y)
    ctx.status()
    ctx.close()
