"""The LF-AM3 step where the spectral vertical solve stops: 1016 layers are the last that leave its
blocks their smallest number of systems (8) in LDS, and 1018 the first whose default form solves on
the grid.  Against the step with fragment-stream contractions (DSHT_TUNE_LEG = 2), whose solves are
on the grid and whose transforms are separate calls.

Tolerance as the step's other comparisons at these shapes: 1e-9 relative L2 a field (the rounding
noise of the constant geopotential's gradient; a wrong factor or layer shows at 1e-6 or more).
"""
import pytest

from test_gpu_lfam3 import OMEGA, _load, _pool, _read

pytestmark = pytest.mark.gpu
TOL = 1e-9


@pytest.mark.parametrize("km", [1016, 1018])
def test_most_layers(gpu, km):
    import torch
    import dsht
    import lfam3
    import oracle
    from conftest import rel_l2
    N, I, J = 10, 32, 16
    st = lfam3.initial_state(oracle.Oracle(N, I, J, 6.371e6), km, seed=km)
    got = []
    for kind in (0, 2):
        p, pool = _pool(N, I, J, km, 1, dt=1800.0)
        p.set_tuning(dsht.TUNE_LEG, kind)
        _load(pool, 0, st)
        pool.set_rotation(0, OMEGA)
        torch.cuda.synchronize()
        pool.step(1)
        torch.cuda.synchronize()
        got.append(_read(pool, 0))
    for f in ("U", "V", "T", "S", "P"):
        assert rel_l2(got[0][f], got[1][f]) < TOL, f
