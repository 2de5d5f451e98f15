"""The device memory of an LF-AM3 pool: 34 grids per layer and run (12 of state, 22 of work), 19 per
run and 8 spectra per layer and run, and what a served run is counted for (41 grids) covers it with
the scratch of the step's transforms."""
import pytest

pytestmark = pytest.mark.gpu


def test_pool_memory(gpu):
    import gc
    import torch
    import dsht
    N, I, J, km, runs = 42, 128, 64, 60, 8
    grid, spec = 8 * I * J, 8 * (N + 1) ** 2
    p = dsht.Plan(N, I, J, radius=6.371e6)
    gc.collect()  # nothing of earlier tests is freed between the readings
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info(gpu)[0]
    pool = dsht.LfAm3(p, dsht.lfam3_config(km=km, max_runs=runs))
    took = free - torch.cuda.mem_get_info(gpu)[0]
    fields = runs * ((34 * km + 19) * grid + 8 * km * spec)
    assert 0.98 * fields < took < 1.02 * fields  # allocations are rounded up to pages
    pool.step(runs)
    torch.cuda.synchronize()
    stepped = free - torch.cuda.mem_get_info(gpu)[0]
    assert stepped < 1.02 * runs * (41 * km * grid + 12 * km * spec)
