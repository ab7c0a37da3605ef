"""Which grouped FP64 batches take the exact integer products: the whole batch decides, not its largest
basis.  8 atoms, lmax 10 (K = 1936); H of either route within 1e-14 of the pinned FP64 MFMA tiles', the
bar between the FP64 summation orders (test_gpu_exact.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,exact", [((1400,), True), ((1400, 1390), True), ((1400, 1300, 60), True),
                                         ((1400,) + (300,) * 12, False), ((100,) * 5 + (1400,), False), ((700, 690), False)])
def test_route_by_the_whole_batch(sizes, exact):
    import torch
    from exciting_amd import lapw, synth
    a = (215.0 * 8) ** (1.0 / 3.0)
    w = synth.make_small(natm_per_species=(4, 4), lmax=10, lorbl=(0, 1), n_target=max(sizes) + 90, nk=1, seed=6,
                         cell=(0.95 * a, a, a / 0.95), rmt=(1.6, 1.5))
    cr, rng = w.crystal, np.random.default_rng(6)
    kps = [synth.make_kpoint(cr, rng, n, None) for n in sizes]
    m = max(k.ngp for k in kps)
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    out = []
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, [synth.pad_kpoint(k, m) for k in kps])
        for v in (-1, 0):
            ctx.set_variant("bmt", v)
            print(f"route of {sizes}, variant {v}", flush=True)
            ctx.setup_batched_dev(b, lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE)
            torch.cuda.synchronize()
            assert ctx.exact_products() == (exact and v < 0)
            out.append([h.clone() for h in b.H])
    for x, y in zip(*out):
        assert (torch.linalg.norm(x - y) / torch.linalg.norm(y)).item() <= 1e-14
    ctx.status()
    ctx.close()
