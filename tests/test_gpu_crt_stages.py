"""The register-pipelined residue GEMM (k_crt.hip, variants 8 to 10) at every remainder of its k loop: one to
nine LDS stages of 64 bytes of k, where two, three or four rotate; bases below and above a 256-wide
tile.  The products are exact integers: H of every variant equals variant 4's (128 x 128 tiles, another
k loop) bit for bit, and the oracle's within the split's own bar (1e-9 relative, as
test_gpu_crt.py holds it)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,natm,n", [(1, (1,), 20), (4, (1, 1), 60), (4, (1, 2), 40), (4, (2, 2), 70), (5, (2, 2), 90),
                                         (6, (1, 2), 270), (6, (2, 2), 60), (7, (2, 2), 257), (7, (2, 2), 64), (8, (1, 2), 100)])
def test_pipelined_stages(lmax, natm, n):
    import torch
    from exciting_amd import lapw, synth
    from oracle import lapw_ref as R
    w = synth.make_small(natm_per_species=natm, lmax=lmax, lorbl=(0, 1), n_target=n, nk=2, seed=40 + n)
    cr = w.crystal
    k = cr.natm * cr.maxaa
    s = torch.cuda.Stream()
    ctx = lapw.Context(cr, stream=s)
    out = {}
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(cr, w.kpoints)
        for v in (4, 8, 9, 10):
            ctx.set_variant("crtgemm", v)
            for t in b.H:
                t.fill_(float("nan"))
            print(f"residue GEMM variant {v}: K {k} ({(k + 63) // 64} stages), N {b.nmat}", flush=True)
            ctx.setup_batched_dev(b, lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_SPLIT_CRT | lapw.EXC_BATCH_OLP_LEGENDRE)
            torch.cuda.synchronize()
            out[v] = [h.clone() for h in b.H]
    for v in (8, 9, 10):
        for h, h4 in zip(out[v], out[4]):
            assert torch.equal(h, h4)
    H_ref, _, _ = R.setup(cr, w.kpoints[0])
    assert np.linalg.norm(out[4][0].cpu().numpy().T - H_ref) <= 1e-9 * np.linalg.norm(H_ref)
    ctx.close()
