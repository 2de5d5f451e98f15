"""The LF-AM3 step's fused transforms at the block shapes that the smaller tests do not reach,
against the separate passes of the same step: past 64 north latitudes the forward contractions run
eight waves a block and 16 columns (w += w_xy(x)), and at 512 longitudes the tracer updates are
epilogues of the M = 256 inverse FFT.  All three time levels are compared.

* DSHT_TUNE_FFT = 1: the LDS FFT, without cos(lat) in the transform and without epilogues.
* DSHT_TUNE_LEG = 2: fragment-stream contractions, w_xy(C) - w_AlphaOptr_xy(A, B) and w += w_xy(x)
  as calls and passes of their own, the vertical solves on the grid.

Ragged ends: T21's 22 and T42's 43 wavenumbers leave partly empty row tiles (whose lanes must not
add to, or read, another lane's coefficient), 3 runs of 6 layers partly empty column tiles.

Tolerance 1e-9 relative L2 a field, as the step's other comparisons: the horizontal gradient of the
constant geopotential is rounding noise of the transforms, below 1e-10 of the winds at T170 (n eps
geo over the winds' forcing); a wrong coefficient, column or update shows at 1e-6 or more.
"""
import pytest

from test_gpu_lfam3 import OMEGA, _load, _pool

pytestmark = pytest.mark.gpu
TOL = 1e-9


@pytest.mark.parametrize("N,I,J,km,runs,steps", [(21, 64, 32, 6, 3, 2), (42, 128, 64, 6, 3, 1), (85, 270, 136, 10, 1, 1),
                                                 (127, 384, 192, 10, 1, 1), (170, 512, 256, 10, 1, 1)])
@pytest.mark.parametrize("key,kind", [("TUNE_FFT", 1), ("TUNE_LEG", 2)])
def test_fused_equals_separate(gpu, N, I, J, km, runs, steps, key, kind):
    import torch
    import dsht
    import lfam3
    import oracle
    from conftest import rel_l2
    o = oracle.Oracle(N, I, J, 6.371e6)
    states = [lfam3.initial_state(o, km, seed=N + r) for r in range(runs)]
    got = []
    for value in (0, kind):
        p, pool = _pool(N, I, J, km, runs, dt=600.0)
        p.set_tuning(getattr(dsht, key), value)
        for r in range(runs):
            _load(pool, r, states[r])
            pool.set_rotation(r, (r + 1) * OMEGA)
        torch.cuda.synchronize()
        for _ in range(steps):
            pool.step(runs)
        torch.cuda.synchronize()
        got.append([(lev, f, r, pool.run_view(f, lev, r).cpu().numpy()) for lev in (dsht.LF_B, dsht.LF_N, dsht.LF_A)
                    for f in (dsht.LF_U, dsht.LF_V, dsht.LF_TRC, dsht.LF_SFCPRES) for r in range(runs)])
    for (lev, f, r, a), b in zip(*got):
        if f == dsht.LF_TRC:
            for t in range(2):
                assert rel_l2(b[3][t], a[t]) < TOL, (lev, f, r, t)
        else:
            assert rel_l2(b[3], a) < TOL, (lev, f, r)
