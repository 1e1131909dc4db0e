"""Records staged per wave and moved to the phase-space and singles lists 64 at a time: nothing is
lost, doubled or written past a list's capacity."""
import numpy as np
import pytest

import mcpet
from harness import psf_sorted, water_cube_scenario


def _rows(p):
    return {r.tobytes() for r in psf_sorted(p)}


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [{}, dict(block_size=64, blocks_per_cu=1)])
def test_phase_space_list_at_its_capacity(kw):
    print(f"staged phase-space records, {kw}", flush=True)
    o = water_cube_scenario(n_decays=5e4, tpb=16, tally_psf_sinogram=0, psf_size=100_000).run_oracle("fmath")
    n = int(o["psf_requested"])
    full = _rows(o["psf"])
    assert n > 1000 and len(full) == n
    for size in (1, 2, 63, 64, 65, 130, n - 1, n, n + 1):
        g = water_cube_scenario(n_decays=5e4, tpb=16, tally_psf_sinogram=0, psf_size=size).run_gpu(
            kernel=mcpet.KERNEL_PERSISTENT, count_events=False, **kw)
        k = min(size, n)
        assert g["psf_requested"] == n and g["psf_count"] == k and len(g["psf"]) == k
        rows = _rows(g["psf"])
        assert len(rows) == k and rows <= full


@pytest.mark.gpu
def test_singles_list_at_its_capacity():
    kw = dict(n_decays=5e4, tpb=16, tally_psf_sinogram=mcpet.TALLY_SINGLES, coincidence_window_ps=4500)
    print("staged singles", flush=True)
    full = water_cube_scenario(singles_capacity=200_000, **kw).run_gpu(count_events=False)
    n = int(full["singles_requested"])
    rows = {r.tobytes() for r in full["singles"]}
    assert n > 1000 and full["singles_count"] == n and len(rows) == n
    for cap in (1, 63, 65, n - 1, n):
        g = water_cube_scenario(singles_capacity=cap, **kw).run_gpu(count_events=False)
        assert g["singles_requested"] == n and g["singles_count"] == cap
        kept = {r.tobytes() for r in g["singles"]}
        assert len(kept) == cap and kept <= rows
        assert np.all(np.diff(g["singles"]["time_ps"].astype(np.int64)) >= 0)
