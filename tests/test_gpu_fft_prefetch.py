"""The register inverse FFTs of FP64 coefficients that fetch part of the next row group ahead
(M = I/2 = 192 and 256) against the LDS kernel (DSHT_TUNE_FFT = 1): truncations below, at and
above the two thirds of M that are fetched ahead, one row group a block and many.

Tolerance: either kernel's transform of 2 M <= 512 points rounds each output by at most a few
eps per stage times the root-mean-square coefficient sum; 9 stages of 4 eps on both sides is
2e-14 of the largest output; 1e-13 is used.
"""
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-13


@pytest.mark.parametrize("N,I,J", [(31, 384, 48), (127, 384, 192), (130, 384, 192), (190, 384, 256),
                                   (170, 512, 256), (173, 512, 256), (254, 512, 256)])
@pytest.mark.parametrize("nc", [1, 40])
def test_prefetch_equals_lds(gpu, N, I, J, nc):
    import torch
    import dsht
    p = dsht.Plan(N, I, J, radius=6.371e6)
    g = torch.Generator(device=gpu).manual_seed(N + nc)
    w = torch.randn((p.lm, nc), generator=g, device=gpu, dtype=torch.float64)
    v = torch.randn((p.lm, nc), generator=g, device=gpu, dtype=torch.float64)
    grid = lambda: torch.full((nc, J, I), float("nan"), dtype=torch.float64, device=gpu)

    def every():
        out = [p.inv_d(k, w, grid()) for k in (dsht.VAL, dsht.GRADLON)]
        out += p.vordiv2uv_d(w, v, grid(), grid())
        torch.cuda.synchronize()
        return out

    reg = every()
    p.set_tuning(dsht.TUNE_FFT, 1)
    for k, (a, b) in enumerate(zip(reg, every())):
        assert torch.isfinite(a).all(), k
        assert float((a - b).abs().max() / b.abs().max()) < TOL, k
