"""The dense-F~ entry's total is held in as many bits as the order loop's: a
compensated pair, rounded once.

Run on the same entries in the same order the two give the same bits.
"""
import numpy as np
import pytest

from conftest import make_oracle
from sparrowpy_amd import testing
from test_gpu_parity import _np, _oracle_directional, ops  # noqa: F401

pytestmark = pytest.mark.gpu

C, DT = 343., 1 / 2000
SOURCE = np.array([1.1, .8, .6])


def _args(r, T, K):
    return (T, r.energy_init_source, r.distance_patches_to_source,
            r.pair_distances(), r.fft, r.p2o, C, DT, K, r.visible_patches)


def _vis(r):
    vis = np.zeros((r.n_patches,) * 2, np.uint8)
    a, b = np.asarray(r.visible_patches).T
    vis[a, b] = 1
    return vis


@pytest.mark.parametrize("n_points,K", [((2, 4), 1), ((2, 4), 7),
                                        ((4, 8), 6), ((8, 16), 5)])
def test_per_pair_bits_are_the_order_loops(ops, n_points, K):
    r = _oracle_directional(testing.shoebox_room_stub(2.5, 2., 1.5), .5,
                            n_points=n_points, seed=3)
    r.init_source_energy(SOURCE)
    r.fft = r.fft * (1 + .05 * np.random.default_rng(7).random(r.fft.shape))
    out = _np(ops.energy_exchange(*_args(r, 301, K)))
    assert ops.energy_exchange_groups() == 0
    plan = ops.ExchangePlan.from_dense(_vis(r), r.pair_distances(), r.p2o,
                                       r.fft, C, DT)
    want = _np(ops.exchange_orders(plan, r.energy_init_source,
                                   r.distance_patches_to_source, C, DT, 301,
                                   K))
    np.testing.assert_array_equal(out, want)


@pytest.mark.parametrize("K", [1, 10, 201])
@pytest.mark.parametrize("size,patch", [((1., 1.2, .9), .9),
                                        ((2.5, 2., 1.5), .5)])
def test_grouped_bits_are_the_order_loops(ops, size, patch, K):
    """One direction: a destination's rows are multiples of its first entry's,
    one group, whose plan can be written down."""
    import torch
    r = make_oracle(testing.shoebox_room_stub(*size), patch)
    r.set_air_attenuation(np.array([1e-4]), np.array([1000.]))
    r.bake_geometry()
    r.init_source_energy(np.array([.6, .5, .4]))
    out = _np(ops.energy_exchange(*_args(r, 301, K)))
    assert ops.energy_exchange_groups() == r.n_patches
    base = ops.ExchangePlan.from_dense(_vis(r), r.pair_distances(), r.p2o,
                                       r.fft, C, DT)
    first = base.row_ptr[:-1]
    n = base.row_ptr[1:] - first
    weight = base.coef[:, 0, 0]
    lag = base.lag.clone()
    lag[base.row_ptr[1:] - 1] |= ops.GroupedPlan.LAST_IN_GROUP
    count = torch.arange(r.n_patches + 1, device=lag.device)
    plan = ops.GroupedPlan(
        base.P, 1, 1, base.row_ptr, count, base.row_ptr,
        count[:-1].to(torch.int32), base.src, lag,
        (weight / weight[first].repeat_interleave(n))[None].contiguous(),
        base.coef[first].contiguous())
    want = _np(ops.exchange_orders(plan, r.energy_init_source,
                                   r.distance_patches_to_source, C, DT, 301,
                                   K))
    np.testing.assert_array_equal(out, want)
