"""The LF-AM3 step's column walks and constant vertical solve (csrc/lfam3.hip) against the CPU
restatement at the layer counts where their code changes: the smallest (2 layers: no interior
QUICK half level; 4: one), partly filled rounds of layers, and the solve's register forms
(up to 32 and 64 layers) and memory form (more).  One step each; boundary conditions of either
kind; a large viscosity on the thin bottom layers makes the solve interchange rows.

Tolerance: a wrong factor, layer or boundary row changes a field by 1e-6 or more of its size
in one step.  Rounding: the horizontal gradient of the constant geopotential (5e4 m2/s2) is
rounding noise of the transforms, about n eps geo, times the density over the winds' forcing:
below 1e-11 of the winds at T21; the surface pressure cancels one more digit.  1e-9.
"""
import pytest

from test_gpu_lfam3 import OMEGA, _load, _pool, _read

pytestmark = pytest.mark.gpu
TOL = 1e-9


@pytest.mark.parametrize("km,cfg", [
    (2, {}), (4, {"trc_sfc_bc": "D"}), (10, {"mom_sfc_bc": "D", "mom_btm_bc": "N"}), (32, {"btm_frict": 1e-4}),
    (34, {"trc_btm_bc": "D"}), (64, {}), (66, {}),
    (20, {"vvisc": 50.0, "vdiff": 20.0}), (40, {"vvisc": 50.0, "vdiff": 20.0, "lam": 1.0}), (68, {"vvisc": 50.0})])
def test_layers_match_oracle(gpu, km, cfg):
    import numpy as np
    import torch
    import lfam3
    import oracle
    from conftest import rel_l2
    N, I, J = 21, 64, 32
    _, pool = _pool(N, I, J, km, 2, dt=1800.0, **cfg)
    o = oracle.Oracle(N, I, J, 6.371e6)
    ocfg = lfam3.Config(dt=1800.0, **cfg)
    states, steppers = [], []
    for r in range(2):
        st = lfam3.initial_state(o, km, seed=km + r)
        states.append(st)
        steppers.append(lfam3.Step(o, km, ocfg, (r + 1) * OMEGA))
        _load(pool, r, st)
        pool.set_rotation(r, (r + 1) * OMEGA)
    if cfg.get("vvisc", 0.0) > 1.0:  # the system of these cases does interchange rows
        s = steppers[0]
        one = np.ones((km, 1, 1))
        _, swaps = oracle.col_vdiff(one, one, cfg["vvisc"] * one, ocfg.depth * one, s.cdk, s.fdk, ocfg.dt, ocfg.lam,
                                    "N", "D", btm_frict=np.zeros((1, 1)))
        assert swaps > 0
    torch.cuda.synchronize()
    pool.step(2)
    torch.cuda.synchronize()
    for r in range(2):
        ref = steppers[r].advance(states[r])
        got = _read(pool, r)
        for f in ("U", "V", "T", "S", "P"):
            assert rel_l2(got[f], ref[f + "N"]) < TOL, (r, f)
        assert np.array_equal(got["UB"], ref["UB"])


@pytest.mark.parametrize("key", ["TUNE_FFT", "TUNE_LEG"])
def test_fused_equals_separate(gpu, key):
    """The step's fused transforms (cos(lat) inside the FFT, w_xy(C) - w_AlphaOptr_xy(A, B) and
    w += w_xy(x) in one contraction) against the separate passes it takes where the plan uses the
    LDS FFT (DSHT_TUNE_FFT = 1) or the fragment-stream contractions (DSHT_TUNE_LEG = 2)."""
    import torch
    import dsht
    import lfam3
    import oracle
    from conftest import rel_l2
    N, I, J, km = 21, 64, 32, 6
    o = oracle.Oracle(N, I, J, 6.371e6)
    st = lfam3.initial_state(o, km, seed=5)
    got = []
    for kind in (0, {"TUNE_FFT": 1, "TUNE_LEG": 2}[key]):
        p, pool = _pool(N, I, J, km, 1, dt=1800.0)
        p.set_tuning(getattr(dsht, key), kind)
        _load(pool, 0, st)
        pool.set_rotation(0, OMEGA)
        torch.cuda.synchronize()
        pool.step(1)
        torch.cuda.synchronize()
        got.append(_read(pool, 0))
    for f in ("U", "V", "T", "S", "P"):
        assert rel_l2(got[1][f], got[0][f]) < TOL, f


@pytest.mark.parametrize("km", [2, 8, 20, 64, 66, 120, 510, 960])
@pytest.mark.parametrize("cfg", [{}, {"vvisc": 50.0, "vdiff": 20.0, "trc_sfc_bc": "D"}])
def test_spectral_solve_equals_grid_solve(gpu, km, cfg):
    """The implicit vertical solves on spectra, with the loads of up to 64 layers at once, in rounds
    and with fewer systems a block where the layers fill the LDS (960: the grid form on both
    sides), against the solves on the grid (taken with DSHT_TUNE_LEG = 2), for two of three runs."""
    import torch
    import dsht
    import lfam3
    import oracle
    from conftest import rel_l2
    N, I, J = 10, 32, 16
    o = oracle.Oracle(N, I, J, 6.371e6)
    got = []
    for kind in (0, 2):
        p, pool = _pool(N, I, J, km, 3, dt=1800.0, **cfg)
        p.set_tuning(dsht.TUNE_LEG, kind)
        for r in range(2):
            _load(pool, r, lfam3.initial_state(o, km, seed=5 + r))
            pool.set_rotation(r, OMEGA)
        torch.cuda.synchronize()
        pool.step(2)
        torch.cuda.synchronize()
        got.append([_read(pool, r) for r in range(2)])
    for r in range(2):
        for f in ("U", "V", "T", "S", "P"):
            assert rel_l2(got[0][r][f], got[1][r][f]) < TOL, (r, f)
