"""The whole-K staged FP64 contractions (csrc/legendre_f64w.hip, the default) against the
per-wave fragment-stream kernels (DSHT_TUNE_LEG = 2), which share nothing with them but the
tables: every operator, at truncations and grids with partly empty row tiles, K steps and
latitude tiles, and column counts around the 8- and 16-column blocks.

Tolerance: both sum the same at most 172 products per output in FP64, in the same order; the
factors i m, R and cos are rounded in other places.  172 eps = 2e-14 of the largest output
covers both; 1e-13 is used.
"""
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-13


@pytest.mark.parametrize("N,I,J", [(5, 16, 8), (31, 96, 48), (85, 270, 136), (170, 540, 270)])
@pytest.mark.parametrize("nc", [1, 8, 9, 17])
@pytest.mark.parametrize("layout", ["LC", "CL"])
def test_staged_equals_streamed(gpu, N, I, J, nc, layout):
    import torch
    import dsht
    p = dsht.Plan(N, I, J, radius=6.371e6)
    g = torch.Generator(device=gpu).manual_seed(N * 100 + nc)
    rnd = lambda *s: torch.randn(s, generator=g, device=gpu, dtype=torch.float64)
    shape = (p.lm, nc) if layout == "LC" else (nc, p.lm)
    wa, wb, ga, gb = rnd(*shape), rnd(*shape), rnd(nc, J, I), rnd(nc, J, I)
    diag = rnd(p.lm)
    spec = lambda: torch.empty(shape, dtype=torch.float64, device=gpu)
    grid = lambda: torch.empty((nc, J, I), dtype=torch.float64, device=gpu)

    def every():
        out = [p.fwd_d(k, ga, spec(), layout=layout, diag=d)
               for k in (dsht.VAL, dsht.DIVLAMBDA, dsht.DIVMU) for d in (None, diag)]
        out += [p.alpha_fwd_d(ga, gb, spec(), layout=layout, diag=diag)]
        out += p.uv2vordiv_d(ga, gb, spec(), spec(), layout=layout, diag=diag)
        out += [p.inv_d(k, wa, grid(), layout=layout)
                for k in (dsht.VAL, dsht.GRADLAMBDA, dsht.GRADMU, dsht.GRADLON, dsht.GRADLAT)]
        out += p.inv_vgrad_d(wa, grid(), grid(), grid(), layout=layout)
        out += [p.alpha_inv_d(wa, wb, grid(), layout=layout)]
        out += p.vordiv2uv_d(wa, wb, grid(), grid(), layout=layout)
        torch.cuda.synchronize()
        return out

    staged = {cb: None for cb in (0, 16, 32)}
    for cb in staged:
        p.set_tuning(dsht.TUNE_LEG_CB, cb)
        staged[cb] = every()
    p.set_tuning(dsht.TUNE_LEG_CB, 0)
    p.set_tuning(dsht.TUNE_LEG, 2)
    ref = every()
    for cb, out in staged.items():
        for k, (a, b) in enumerate(zip(out, ref)):
            err = float((a - b).abs().max() / b.abs().max())
            assert err < TOL, (cb, k, err)
