"""The segmented column walk of the Redi/GM mixing (csrc/redigm.hip) against the oracle: layer
counts around the 3-layer segments and their halos, tapers that reach over several segments, and
columns with infinities, NaN and a zero thickness, whose neighbours must not see them.

Tolerance: as the column part's (1e-13 of each output's largest value): no multiply-add is
contracted and the quotients round as the divisions do, so only tanh, exp and sin may differ in
the last bit.  Special values: the same class (NaN, +inf, -inf, finite) as the oracle's at every
point, and the columns without any are the same bits as without them elsewhere.
"""
import math

import numpy as np
import pytest

from test_gpu_redigm import R_EARTH, _cfg_pair, _dev, _fields

pytestmark = pytest.mark.gpu


def _inputs(p, km, tilt, shallow):
    x = _fields(p, km, seed=100 + km, tilt=tilt, shallow=shallow)
    rng = np.random.default_rng(km)
    x["gl"], x["ga"] = (rng.standard_normal((2 * km, p.jm, p.im)) * 1e-6 * R_EARTH for _ in range(2))
    return x


def _device(p, x, gpu, cfg):
    import torch
    d = _dev(x, gpu)
    out = p.col_redigm_d(d["pt"], d["sa"], d["h"], d["z"], d["topo"], d["cdk"], d["rfdk"], d["gl"], d["ga"], cfg=cfg)
    torch.cuda.synchronize()
    return [o.cpu().numpy().reshape(x["gl"].shape) for o in out]


def _oracle(p, x, ocfg):
    import redigm as RG
    km = len(x["pt"])
    lat = p.y_Lat
    cs = np.array([math.cos(v) for v in lat])
    g = (x["gl"][:km], x["ga"][:km], x["gl"][km:], x["ga"][km:])
    with np.errstate(all="ignore"):
        r = RG.column_part(x["pt"], x["sa"], x["h"], x["z"], x["topo"], g, lat, cs, x["cdk"], x["rfdk"], ocfg, R_EARTH)
    return [np.asarray(a).reshape(x["gl"].shape) for a in r]


@pytest.mark.parametrize("N,I,J", [(5, 16, 8), (31, 100, 48)])
@pytest.mark.parametrize("km", [2, 3, 4, 5, 7, 31])
@pytest.mark.parametrize("interior,tilt,shallow", [("DM95", 1.0, True), ("DM95", 40.0, False), ("GKW91", 40.0, True)])
def test_segments_match_oracle(gpu, N, I, J, km, interior, tilt, shallow):
    import dsht
    p = dsht.Plan(N, I, J, radius=R_EARTH)
    x = _inputs(p, km, tilt, shallow)
    ocfg, cfg = _cfg_pair(interior=interior)
    for name, g, ref in zip(("flx_lon", "flx_lat", "vdiv"), _device(p, x, gpu, cfg), _oracle(p, x, ocfg)):
        assert np.max(np.abs(g - ref)) < 1e-13 * np.max(np.abs(ref)), name


def test_special_values_stay_in_their_columns(gpu):
    import dsht
    p = dsht.Plan(10, 32, 16, radius=R_EARTH)
    km = 13
    x = _inputs(p, km, 5.0, False)
    ocfg, cfg = _cfg_pair()
    clean = _device(p, x, gpu, cfg)
    x["gl"][4, 2, 3] = np.inf
    x["ga"][km + 6, 3, 5] = -np.inf
    x["pt"][5, 4, 7] = np.nan
    x["h"][6, 5, 9] = 0.0
    x["gl"][2, 6, 11] = 1e300
    x["h"][3, 7, 13] = 1e-305
    bad = np.zeros((16, 32), bool)
    for j, i in ((2, 3), (3, 5), (4, 7), (5, 9), (6, 11), (7, 13)):
        bad[j, i] = True
    kind = lambda a: np.where(np.isnan(a), 3, np.where(np.isinf(a), np.sign(a), 2))
    for c, g, ref in zip(clean, _device(p, x, gpu, cfg), _oracle(p, x, ocfg)):
        assert np.array_equal(g[:, ~bad], c[:, ~bad])
        assert np.array_equal(kind(g[:, bad]), kind(ref[:, bad]))
