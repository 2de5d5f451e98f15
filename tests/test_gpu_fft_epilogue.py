"""The inverse FFTs that finish a field as they store it (csrc/fft_reg.hip) against the same call
with the passes apart, at every register FFT length.

* Redi/GM: right-hand sides that cannot take 16-byte stores (odd pitch, or 8 bytes off) get a plain
  inverse and a pass; both evaluate (rhs + hdiv) + vdiv from the same FFT up to its rounding, a few
  eps of the largest tendency: 1e-13 of the largest value.  Also with the columns cut into chunks
  that straddle the two tracers.
* LF-AM3: the LDS FFT (DSHT_TUNE_FFT = 1) takes the passes apart; the tolerance is that of the
  step's other comparisons, 1e-9 (the geopotential gradient's rounding noise).
"""
import pytest

from test_gpu_lfam3 import OMEGA, _load, _pool, _read
from test_gpu_redigm import R_EARTH, _dev, _fields

pytestmark = pytest.mark.gpu
SIZES = [(5, 16, 8), (10, 32, 16), (21, 64, 32), (23, 72, 36), (31, 96, 48), (42, 128, 64), (47, 144, 72),
         (63, 192, 96), (85, 256, 128), (85, 270, 136), (127, 384, 192), (170, 512, 256), (170, 540, 270)]


@pytest.mark.parametrize("N,I,J", SIZES)
def test_redigm_rhs(gpu, N, I, J):
    import torch
    import dsht
    km = 5
    p = dsht.Plan(N, I, J, radius=R_EARTH)
    x = _dev(_fields(p, km, seed=N, tilt=5.0), gpu)
    g = torch.Generator(device=gpu).manual_seed(N)
    r0 = [1e-6 * torch.randn((km, J * I), generator=g, device=gpu, dtype=torch.float64) for _ in range(2)]

    def call(pitch, off):
        rhs = []
        for r in r0:
            buf = torch.zeros(km * pitch + off, dtype=torch.float64, device=gpu)
            v = torch.as_strided(buf, (km, J, I), (pitch, I, 1), off)
            v.copy_(r.view(km, J, I))
            rhs.append((buf, v))
        p.redigm_d(x["pt"], x["sa"], x["h"], x["z"], x["topo"], x["cdk"], x["rfdk"], rhs[0][1], rhs[1][1])
        torch.cuda.synchronize()
        for buf, v in rhs:  # nothing outside the columns
            pad = torch.as_strided(buf, (km - 1, pitch - I * J), (pitch, 1), off + I * J)
            assert not pad.any() and not buf[:off].any()
        return [v.clone() for _, v in rhs]

    ref = call(I * J + 1, 0)  # odd pitch: apart
    for pitch, off, chunk in ((I * J, 0, 0), (I * J + 6, 2, 0), (I * J, 0, 3), (I * J, 1, 0)):
        p.set_tuning(dsht.TUNE_CHUNK_COLS, chunk)
        for a, b in zip(call(pitch, off), ref):
            assert float((a - b).abs().max()) < 1e-13 * float(b.abs().max()), (pitch, off, chunk)
        p.set_tuning(dsht.TUNE_CHUNK_COLS, 0)


@pytest.mark.parametrize("N,I,J", SIZES[:-2])
def test_lfam3_tracers(gpu, N, I, J):
    import torch
    import dsht
    import lfam3
    import oracle
    from conftest import rel_l2
    km = 4
    st = lfam3.initial_state(oracle.Oracle(N, I, J, 6.371e6), km, seed=N)
    got = []
    for kind in (0, 1):
        p, pool = _pool(N, I, J, km, 1, dt=600.0)
        p.set_tuning(dsht.TUNE_FFT, kind)
        _load(pool, 0, st)
        pool.set_rotation(0, OMEGA)
        torch.cuda.synchronize()
        pool.step(1)
        pool.step(1)
        torch.cuda.synchronize()
        got.append(_read(pool, 0))
    for f in got[0]:
        if f[0] in "TS":
            assert rel_l2(got[1][f], got[0][f]) < 1e-9, f
