"""The Redi/GM column part (csrc/redigm.hip) on both sides of the rule that gives a thread its whole
column, scans and walk in one launch (up to 9 layers, 3 within the whole tendency; up to 14 from
65536 points on, up to 20 from 98304), or a segment of layers after a launch of the scans: layer counts and grids around each line,
against the oracle, with tapers that reach over most layers and with scans that find nothing.

Tolerance as the column part's elsewhere: 1e-13 of each output's largest value.
"""
import numpy as np
import pytest

from test_gpu_redigm import R_EARTH, _cfg_pair
from test_gpu_redigm_segments import _device, _inputs, _oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,I,J,km", [(5, 16, 8, 2), (10, 32, 16, 8), (10, 32, 16, 9), (10, 32, 16, 10), (31, 100, 48, 9),
                                      (127, 384, 170, 10),
                                      (127, 512, 128, 14), (127, 512, 128, 15), (127, 512, 192, 20),
                                      (127, 512, 192, 21)])
@pytest.mark.parametrize("interior,tilt,shallow", [("DM95", 40.0, True), ("GKW91", 1.0, False)])
def test_columns_match_oracle(gpu, N, I, J, km, interior, tilt, shallow):
    import dsht
    p = dsht.Plan(N, I, J, radius=R_EARTH)
    x = _inputs(p, km, tilt, shallow)
    ocfg, cfg = _cfg_pair(interior=interior)
    for name, g, ref in zip(("flx_lon", "flx_lat", "vdiv"), _device(p, x, gpu, cfg), _oracle(p, x, ocfg)):
        assert np.max(np.abs(g - ref)) < 1e-13 * np.max(np.abs(ref)), name


@pytest.mark.parametrize("km", [2, 9, 10])
def test_padded_layers(gpu, km):
    """Layers of a larger pitch (and 8 bytes off a 16-byte boundary) give the same bits."""
    import torch
    import dsht
    p = dsht.Plan(10, 32, 16, radius=R_EARTH)
    x = {k: torch.tensor(np.ascontiguousarray(v), device=gpu) for k, v in _inputs(p, km, 5.0, True).items()}
    pitch = p.im * p.jm + 7

    def padded(t):
        buf = torch.full((1 + t.shape[0] * pitch,), float("nan"), dtype=torch.float64, device=gpu)
        v = torch.as_strided(buf, t.shape, (pitch, p.im, 1), 1)
        v.copy_(t)
        return v

    def call(f):
        return p.col_redigm_d(f(x["pt"]), f(x["sa"]), f(x["h"]), f(x["z"]), x["topo"], x["cdk"], x["rfdk"], f(x["gl"]),
                              f(x["ga"]))
    for a, b in zip(call(padded), call(lambda t: t)):
        assert torch.equal(a, b)
