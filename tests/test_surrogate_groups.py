"""Samples of a batch go through the network together, in equal groups: every sample's output has
the same bits as alone, and the gradients are the mean of the samples' own ones."""
import ctypes as C

import numpy as np
import pytest

import mcpet
from harness import head_scenario
from test_surrogate import _layer_rel, integer_network, unet_reference


def _network(grid, cin, c, rng):
    net = mcpet.Surrogate(grid, in_channels=cin, width=c, seed=11)
    p = net.params()
    p[-(c + 1):] = rng.normal(0, 0.1, c + 1)   # a residual that is not zero
    net.set_params(p.astype(np.float32))
    return net


# one group, a full one, two unequal ones of 64 at most (35 + 34); widths with and without whole
# 32-channel slices; volumes below and above one tile; one whose group is bounded by its voxels; one whose
# sample does not fit half of the input staging (2 MB)
@pytest.mark.gpu
@pytest.mark.parametrize("grid,cin,c,batch", [((4, 4, 4), 1, 3, 69), ((4, 8, 20), 2, 16, 5), ((8, 12, 16), 4, 32, 3),
                                              ((12, 36, 36), 2, 32, 7), ((32, 68, 64), 2, 8, 5), ((16, 48, 48), 16, 4, 3)])
def test_batch_equals_its_samples(grid, cin, c, batch):
    rng = np.random.default_rng(5)
    net = _network(grid, cin, c, rng)
    x = rng.random((batch, cin) + grid).astype(np.float32)
    y = rng.random((batch,) + grid).astype(np.float32)
    together = net.forward(x)
    alone = np.concatenate([net.forward(x[i:i + 1]) for i in range(batch)])
    assert np.array_equal(together, alone)
    loss, grad = net.gradients(x, y)
    each = [net.gradients(x[i:i + 1], y[i:i + 1]) for i in range(batch)]
    mean = np.mean([g.astype(np.float64) for _, g in each], axis=0)
    # the loss gradient of a sample is scaled by 1 / batch before its BF16 rounding, which moves each
    # product's operands by up to 2^-9: the norm of the difference is bounded by that of the parts
    size = np.mean([np.linalg.norm(g.astype(np.float64)) for _, g in each])
    assert np.linalg.norm(grad - mean) <= 2.0 ** -8 * size
    assert abs(loss - np.mean([l for l, _ in each])) <= 1e-5 * abs(loss)


# three groups, staged in one piece each; in five, five and four pieces of one sample each; in three pieces of
# a sample's voxels each
@pytest.mark.gpu
@pytest.mark.parametrize("grid,cin,c,batch", [((4, 4, 4), 1, 3, 150), ((32, 56, 56), 4, 8, 14), ((32, 68, 132), 4, 4, 5)])
def test_groups_behind_a_transport_run_keep_their_samples(grid, cin, c, batch):
    """While a run (some 50 ms) holds the device, the kernels that read a group's input wait behind it, and the
    host must not fill the staging with the next group's until they have."""
    rng = np.random.default_rng(batch)
    net = _network(grid, cin, c, rng)
    x = rng.random((batch, cin) + grid).astype(np.float32)
    alone = np.concatenate([net.forward(x[i:i + 1]) for i in range(batch)])
    sc = head_scenario(n_decays=1e8)
    with mcpet.Simulation(sc.cfg, sc.phantom, sc.tables) as sim:
        for _ in range(2):
            sim.run()
            together = net.forward(x)
            sim.sync()
            assert np.array_equal(together, alone)


@pytest.mark.gpu
def test_gradient_tensors_of_a_group_wait_for_its_first_gradients():
    """Width 32 on 32 x 56 x 56 in groups of six: the forward's tensors are 285 bytes a voxel and sample, the
    gradients' 1084; beside them the weight gradients' partial sums (57 MB), parameters and optimiser state (27 MB)."""
    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert mcpet.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    grid, vox = (32, 56, 56), 32 * 56 * 56
    x = np.random.default_rng(2).random((6, 4) + grid).astype(np.float32)
    warm = mcpet.Surrogate(grid, in_channels=4, width=32, seed=1)   # the kernels' code and scratch
    warm.gradients(x, x[:, 0])
    free = [free_bytes()]
    net = mcpet.Surrogate(grid, in_channels=4, width=32, seed=1)
    for call in (lambda: net.forward(x), lambda: net.gradients(x, x[:, 0])):
        call()
        free.append(free_bytes())
    held = free[0] - np.array(free[1:], float)
    slack = 40e6                                                    # the allocations' granularity
    assert held[0] < (6 * 285 + 1084) * vox + 84e6 + slack
    assert abs(held[1] - held[0] - 5 * 1084 * vox) < slack


# 20 x 44 x 68 takes the tiles of 16 x 8 x 2 (1100 four-row tiles) with a remainder in x and y, its
# half resolution the plane-wise products with one in x and y; 36 x 28 x 84 a remainder of every kind
@pytest.mark.gpu
@pytest.mark.parametrize("grid,batch", [((20, 44, 68), 2), ((36, 28, 84), 1)])
def test_ragged_tiles_are_exact_on_integer_networks(grid, batch):
    """Sums of small integers: equal to the float64 reference bit for bit."""
    cin, c = 2, 32
    rng = np.random.default_rng(sum(grid))
    p = integer_network(cin, c, rng)
    x = rng.integers(0, 4, (batch, cin) + grid).astype(np.float32)
    net = mcpet.Surrogate(grid, in_channels=cin, width=c, seed=3)
    net.set_params(p.astype(np.float32))
    _, _, yr = unet_reference(p, x.astype(np.float64), np.zeros((batch,) + grid), cin, c, "bf16", grad=False)
    assert np.abs(yr).max() < 2.0 ** 24 and np.all(yr == np.round(yr))
    assert np.array_equal(net.forward(x).astype(np.float64), yr)


# width 160: the weight gradient of 960 -> 320 channels goes in two passes of output channels, the
# others in one; remainders of the tiles of both strides in x, y and z
@pytest.mark.gpu
@pytest.mark.parametrize("grid,c,batch", [((4, 4, 4), 160, 1), ((12, 20, 36), 8, 2)])
def test_weight_gradients_match_the_reference(grid, c, batch):
    """The bounds of test_surrogate's comparison: 2e-3 a layer, or four times what float32 sums in
    another order change."""
    cin = 2
    rng = np.random.default_rng(c)
    net = _network(grid, cin, c, rng)
    p = net.params().astype(np.float64)
    x, t = rng.random((batch, cin) + grid), rng.random((batch,) + grid)
    x, t = x.astype(np.float32), t.astype(np.float32)
    _, g = net.gradients(x, t)
    gr, g32 = (unet_reference(p, x.astype(np.float64), t.astype(np.float64), cin, c, m)[1] for m in ("bf16", "bf16f32"))
    rel, rel32 = _layer_rel(g.astype(np.float64), gr, cin, c), _layer_rel(g32, gr, cin, c)
    assert all(r <= max(2e-3, 4 * r32) for r, r32 in zip(rel, rel32)), (rel, rel32)
