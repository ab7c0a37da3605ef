"""The default overlap kernel of the addition theorem (k_olp.hip: 64 rows x 16 columns a wave, the
columns' factors by lane broadcast) against variant 2 over every l range it is compiled for, one
atom to several, and bases around the edges of its 64 x 64 tiles and 16-column slices; and at
those sizes against the oracle.

Bars: within 1e-14 of the largest element of variant 2, as test_gpu_olp.py holds its variants to each
other (the same recurrence, the same number of roundings, another order); 1e-12 relative
(Frobenius) of the oracle, as there; every element written, the lower triangle the conjugate."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,natm,n", [(1, 1, 9), (2, 2, 63), (3, 1, 64), (4, 3, 65), (5, 2, 79), (6, 1, 81), (7, 2, 127),
                                         (8, 5, 129), (9, 1, 145), (10, 4, 200), (11, 2, 96), (12, 1, 33)])
def test_olp_default_against_rows_and_oracle(lmax, natm, n):
    import torch
    from exciting_amd import lapw, synth
    from oracle import lapw_ref as R
    w = synth.make_small(natm_per_species=(natm,), lmax=lmax, lorbl=(0,), n_target=n, nk=2, seed=50 + lmax)
    s = torch.cuda.Stream()
    ctx = lapw.Context(w.crystal, stream=s)
    out = {}
    with torch.cuda.stream(s):
        b = lapw.DeviceBatch(w.crystal, w.kpoints)
        for v in (-1, 2):
            ctx.set_variant("olp", v)
            for t in b.O:
                t.fill_(float("nan"))
            print(f"overlap lmax {lmax}, {natm} atoms, N {b.nmat}, variant {v}", flush=True)
            ctx.setup_batched_dev(b, lapw.EXC_BATCH_MATCH | lapw.EXC_BATCH_OLP_LEGENDRE)
            torch.cuda.synchronize()
            out[v] = [t.cpu().numpy().T for t in b.O]
    for i, kp in enumerate(w.kpoints):
        o, ref = out[-1][i], out[2][i]
        assert np.isfinite(o).all()
        assert np.abs(o - ref).max() <= 1e-14 * np.abs(ref).max()
        il = np.tril_indices(o.shape[0], -1)
        assert np.array_equal(o[il], np.conj(o.T[il]))
        O_ref = R.setup(w.crystal, kp)[1]
        assert np.linalg.norm(o - O_ref) <= 1e-12 * np.linalg.norm(O_ref)
    ctx.close()
