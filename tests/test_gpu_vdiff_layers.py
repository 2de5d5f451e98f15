"""The vertical diffusion solve (csrc/column.hip) bit for bit against the oracle at the layer counts
around its rules: 9 and 10 (weights of the half levels divided in place, then in LDS), 45 to 63 (1 to
19 rows eliminated a second time: one to three chunks, partly filled), both forms, with and without
row interchanges.  The operations and their order are the oracle's, so the bits are equal."""
import numpy as np
import pytest

from test_gpu_column import _dev, _vdiff_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("km", [2, 5, 9, 10, 45, 46, 47, 52, 53, 59, 61, 63])
@pytest.mark.parametrize("pivot", [False, True])
@pytest.mark.parametrize("mom", [False, True])
def test_vdiff_layers(gpu, km, pivot, mom):
    import torch
    import dsht
    import oracle
    N, I, J = 10, 36, 16  # 576 points: a partly filled block
    p = dsht.Plan(N, I, J, radius=6.371e6)
    q0, rhs, kv, e3, cdk, fdk = _vdiff_case(km, J, I, km, pivot)
    bf = np.random.default_rng(km).uniform(0.0, 1e-3, (J, I)) if mom else None
    dev = [_dev(a, gpu) for a in (q0, rhs, kv, e3, cdk, fdk)]
    out = p.col_vdiff_d(*dev, 3600.0, 1.0, "N", "D", btm_frict=None if bf is None else _dev(bf, gpu))
    torch.cuda.synchronize()
    ref, swaps = oracle.col_vdiff(q0, rhs, kv, e3, cdk, fdk, 3600.0, 1.0, "N", "D", btm_frict=bf)
    assert swaps > 0 or not (pivot and km >= 20)
    assert np.array_equal(out.cpu().numpy(), ref)
