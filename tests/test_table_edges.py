"""Interaction tables and detector settings at the edge of what the loader accepts: the kernels follow
the oracle there too, stream by stream."""
import gzip

import numpy as np
import pytest

import mcpet
from conftest import AIR, WATER
from harness import Scenario, assert_tallies_equal
from mcpet import phantoms

KERNELS = [mcpet.KERNEL_PLAIN, mcpet.KERNEL_PERSISTENT]


def _water_file(tmp_path, section, edit):
    """The water file with `edit` applied to the fields of every row of the table below `section`."""
    lines = gzip.open(WATER, "rt").read().split("\n")
    at = next(i for i, l in enumerate(lines) if section in l) + 1
    n = int(lines[at].lstrip("# "))
    for i in range(n):
        lines[at + 2 + i] = "  " + "  ".join(edit(i, lines[at + 2 + i].split()))
    path = tmp_path / "water.mcgpu"
    path.write_text("\n".join(lines))
    return str(path)


def _scenario(water, **cfgkw):
    mat, dens, act, vs = phantoms.water_cube(n_decays=5e4)
    cfg = phantoms.make_config(seed=2026, threads_per_block=8, materials=[AIR, water], tally_psf_sinogram=0,
                               psf_size=100_000, material_dose=True, **cfgkw)
    return Scenario(cfg, mat, dens, act, vs, [AIR, water])


def _profile(shell, value):
    return lambda i, f: f[:2] + [value if i == shell else f[2]] + f[3:]


# a momentum profile that is not a number leaves the Compton energy undefined (absorbed, as below the
# tables); a resolution that is not a number every detected energy (in no bin of the spectrum)
@pytest.mark.gpu
@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("j0,e_resol", [("nan", 0.12), (None, float("nan"))])
def test_undefined_energies_follow_the_oracle(tmp_path, kernel, j0, e_resol):
    water = _water_file(tmp_path, "[NUMBER OF SHELLS", _profile(2, j0)) if j0 else WATER
    sc = _scenario(water, e_resol=e_resol)
    o = sc.run_oracle()
    assert o["counters"]["compton"] > 1000 and o["spectrum"].sum() == (0 if np.isnan(e_resol) else 2 * o["counters"]["pairs_tallied"])
    assert_tallies_equal(sc.run_gpu(kernel=kernel), o)


# a profile of no, hardly any, negative and (beyond what a product in binary32 holds) unbounded width
@pytest.mark.gpu
@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("shell,j0", [(0, "0"), (2, "0"), (1, "-0.0"), (0, "1e-40"), (0, "3e-25"), (1, "-20.0"), (0, "1e30"), (1, "inf")])
def test_momentum_profiles_of_any_width_follow_the_oracle(tmp_path, kernel, shell, j0):
    sc = _scenario(_water_file(tmp_path, "[NUMBER OF SHELLS", _profile(shell, j0)))
    o = sc.run_oracle()
    assert o["counters"]["compton"] > 1000
    assert_tallies_equal(sc.run_gpu(kernel=kernel), o)


# negative squared momentum transfers: Rayleigh cosines above 1, whose direction is undefined (the photon leaves)
@pytest.mark.gpu
@pytest.mark.parametrize("kernel", KERNELS)
def test_rayleigh_cosines_above_one_follow_the_oracle(tmp_path, kernel):
    sc = _scenario(_water_file(tmp_path, "[DATA VALUES TO SAMPLE SQUARED",
                               lambda i, f: [f"{-1.0 + 0.01 * i:.3f}"] + f[1:] if i < 64 else f))
    o = sc.run_oracle()
    assert o["counters"]["rayleigh"] > 100
    assert_tallies_equal(sc.run_gpu(kernel=kernel), o)
