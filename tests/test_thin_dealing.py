"""Streams dealt thinly to the persistent kernel's waves (few streams for the device): the same
tallies as the oracle's at the edges of the dealing."""
import pytest

import mcpet
from harness import assert_tallies_equal, water_cube_scenario


@pytest.mark.gpu
@pytest.mark.parametrize("tpb,kw", [
    (1, {}),                                          # 729 streams: one lane per wave, fewer waves than resident
    (9, {}),                                          # 6561 streams: two lanes, a short last row
    (7, dict(block_size=64, blocks_per_cu=1)),        # 5103 streams on 256 waves: 20 lanes
    (449, {}),                                        # 327321 streams: 64 lanes, still dealt
    (450, {}),                                        # 328050 streams: full waves, in queue order
    (539, {}),
    (540, {}),
    (540, dict(blocks_per_cu=12)),                    # more waves than are resident: no chunk by number
])
def test_thinly_dealt_streams_give_the_oracles_tallies(tpb, kw):
    print(f"thin dealing: water cube, tpb {tpb}, {kw}", flush=True)
    sc = water_cube_scenario(n_decays=3e4, tpb=tpb, material_dose=True)
    o = sc.run_oracle("fmath")
    assert_tallies_equal(sc.run_gpu(kernel=mcpet.KERNEL_PERSISTENT, count_events=False, **kw), o, counters="lite")


@pytest.mark.gpu
@pytest.mark.parametrize("decays,tpb,kw", [
    (3, 540, {}),                                     # waves whose streams are all without a decay
    (200, 540, dict(blocks_per_cu=1)),                # first chunks of 96 (393660 streams on 1024 waves)
    (3e4, 259, dict(blocks_per_cu=1)),                # 188811 streams: fewer than 192 a wave
    (3e4, 270, dict(block_size=64, blocks_per_cu=4)),   # 196830: a few more
    (4e5, 450, {}),                                   # about one decay a stream, lanes that ask again and again
])
def test_streams_made_ready_together_give_the_oracles_tallies(decays, tpb, kw):
    print(f"ready streams: water cube, {decays} decays, tpb {tpb}, {kw}", flush=True)
    sc = water_cube_scenario(n_decays=decays, tpb=tpb, material_dose=True)
    o = sc.run_oracle("fmath")
    assert_tallies_equal(sc.run_gpu(kernel=mcpet.KERNEL_PERSISTENT, count_events=False, **kw), o, counters="lite")
