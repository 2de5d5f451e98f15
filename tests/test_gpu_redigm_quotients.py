"""The quotients of the Redi/GM column part (csrc/redigm.hip), formed from a reciprocal, where a
quotient overflows: like the division they give an infinity there (the correction step alone gives
NaN, which v_div_fixup_f64 replaces).  Divisors inside the range in which the reciprocal is used: a layer thickness
of 1e-260 m, and a radius of 0.25 (a scaled sphere).

The fluxes' classes (NaN, +inf, -inf, finite) are the oracle's at every point.  Finite values agree
to 1e-13 of each column's largest value, as the column part's do elsewhere.
"""
import numpy as np
import pytest

from test_gpu_redigm import _cfg_pair, _dev, _fields
from test_gpu_redigm_segments import _device

pytestmark = pytest.mark.gpu


def thin_layers(p):
    """Columns of 1e-260 m with a gradient of 1e162 K in one layer: the flux divergence over the
    thickness passes the largest double there."""
    km = 6
    x = _fields(p, km, seed=3)
    rng = np.random.default_rng(3)
    x["gl"], x["ga"] = (rng.standard_normal((2 * km, p.jm, p.im)) for _ in range(2))
    for j, i in ((2, 3), (5, 7)):
        x["h"][:, j, i] = 1e-260
        x["gl"][2, j, i] = 1e162
    return x


def large_gradients(p):
    """GradLon of 1e308 K in one layer of a sphere of radius 0.25: an infinite slope, whose taper 0
    leaves the latitude flux finite."""
    km = 6
    x = _fields(p, km, seed=4)
    rng = np.random.default_rng(4)
    x["gl"], x["ga"] = (1e-8 * rng.standard_normal((2 * km, p.jm, p.im)) for _ in range(2))
    for j, i in ((2, 3), (5, 7)):
        x["gl"][2, j, i] = 1e308
    return x


def oracle_column(x, lat, radius, ocfg):
    import math
    import redigm as RG
    km = len(x["pt"])
    cs = np.array([math.cos(v) for v in lat])
    g = (x["gl"][:km], x["ga"][:km], x["gl"][km:], x["ga"][km:])
    with np.errstate(all="ignore"):
        r = RG.column_part(x["pt"], x["sa"], x["h"], x["z"], x["topo"], g, lat, cs, x["cdk"], x["rfdk"], ocfg, radius)
    return [np.asarray(a).reshape(x["gl"].shape) for a in r]


def kind(a):
    return np.where(np.isnan(a), 3, np.where(np.isinf(a), np.sign(a), 2))


@pytest.mark.parametrize("case,radius", [(thin_layers, 6.371e6), (large_gradients, 0.25)])
def test_overflowing_quotients(gpu, case, radius):
    import dsht
    p = dsht.Plan(10, 32, 16, radius=radius)
    x = case(p)
    ocfg, cfg = _cfg_pair()
    for name, g, ref in zip(("flx_lon", "flx_lat", "vdiv"), _device(p, x, gpu, cfg), oracle_column(x, p.y_Lat, radius, ocfg)):
        assert np.array_equal(kind(g), kind(ref)), name
        fin = np.isfinite(ref)
        d = np.abs(np.where(fin, g, 0.0) - np.where(fin, ref, 0.0))
        top = np.where(fin, np.abs(ref), 0.0).max(axis=0)
        assert (d <= 1e-13 * top).all(), name
