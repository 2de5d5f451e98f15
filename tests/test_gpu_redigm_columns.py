"""The Redi/GM column part (csrc/redigm.hip) on both sides of the rule that gives a thread its whole
column, scans and walk in one launch (up to 9 layers; up to 14 from 65536 points on, up to 20 from
98304), or a segment of layers after a launch of the scans: layer counts and grids around each line,
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
