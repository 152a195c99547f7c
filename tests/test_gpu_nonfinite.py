"""Infinite and NaN factors and gradients: orders limited to the bins that
energy can have reached give what whole orders give.  Such a factor times the
zero of a bin beyond is NaN, in the reference's loop from the pair's delay on.
"""
import numpy as np
import pytest

import oracle as orc
from sparrowpy_amd import testing
from sparrowpy_amd.coordinates import Coordinates
from test_gpu_adjoint_reach import _room
from test_gpu_parity import _np, _oracle_directional, ops  # noqa: F401
from test_gpu_sums import ROOM, SRC, _plan

pytestmark = pytest.mark.gpu

C, DT, T = 343., 1 / 2000, 301
INF, NAN = float("inf"), float("nan")


@pytest.fixture(scope="module")
def room():
    r = _oracle_directional(testing.shoebox_room_stub(*ROOM), .5,
                            n_points=(4, 8), seed=3)
    r.init_source_energy(SRC)
    return r


@pytest.mark.parametrize("value", [INF, -INF, NAN])
@pytest.mark.parametrize("form,array", [
    ("pairs", "coef"), ("grouped", "scal"), ("grouped", "rtab"),
    ("grouped-16-8", "rtab"), ("grouped-row-4", "scal"),
    ("grouped-row-2", "rtab"), ("ds", "dscal"), ("ds-16", "scal"),
    ("ds-row-4", "dscal"), ("ds-row-2", "scal")])
def test_factors(ops, room, form, array, value):
    plan = _plan(ops, room, form, DT)
    a = getattr(plan, array)
    if a.dim() == 2:            # a band's weight of the first entry
        a[1, 0] = value
    else:                       # a direction's factor: an entry's, or a row's
        a[int(plan.grp_key[0]) if array == "rtab" else 0, 1, 2] = value
    if getattr(plan, "tiles", None):        # they hold the weights as they were
        plan.tiles = ops.tile_plan(plan, 16, min_merge=0)
        plan.tiles.R = 8
    args = (plan, room.energy_init_source, room.distance_patches_to_source,
            C, DT, T)
    far = int(room.distance_patches_to_source.max() / C / DT) + 1
    for f in (ops.exchange_orders, ops.exchange_sum):
        for K in (1, 4):
            short, whole = (_np(f(*args, K, reach)) for reach in (far, None))
            assert np.isnan(whole[..., -1]).any()
            np.testing.assert_array_equal(short, whole)


@pytest.mark.parametrize("value", [INF, NAN])
def test_dense_entry(ops, room, value):
    fft = room.fft.copy()
    i, j = room.visible_patches[7]
    fft[i, j, 2, 1] = value
    args = (T, room.energy_init_source, room.distance_patches_to_source,
            room.pair_distances(), fft, room.p2o, C, DT, 3,
            room.visible_patches)
    out, ref = _np(ops.energy_exchange(*args)), orc.exchange(*args,
                                                             nthreads=8)
    assert np.isnan(ref[..., -1]).any()
    assert np.isnan(out[np.isnan(ref)]).all()


@pytest.mark.parametrize("directional", [False, True])
@pytest.mark.parametrize("where", ["table", "early gradient",
                                   "late gradient"])
@pytest.mark.parametrize("every", [1, 3])
def test_adjoint(directional, where, every):
    import torch
    from sparrowpy_amd import adjoint
    make = adjoint.BRDFExchangeAdjoint if directional else \
        adjoint.ExchangeAdjoint
    adj = make(_room(directional, 1), Coordinates(*SRC),
               Coordinates([1.9, .7], [1.2, .9], [1., .4]), C, DT,
               (T + .5) * DT, 4, checkpoint_every=every)
    assert adj.reach < 40
    tables = [adj.table0.clone()] if directional else \
        [adj.A0.clone(), adj.C0.clone()]
    grad = torch.rand(2, 2, T, generator=torch.Generator().manual_seed(0),
                      dtype=torch.float64).cuda()
    if where == "table":
        tables[0].view(-1)[0] = NAN
    else:
        grad[1, 0, 20 if where == "early gradient" else T - 1] = INF
    out = []
    for reach in (adj.reach, T):
        adj.reach = reach
        h = adj.forward(*tables)
        g = adj.backward(grad)
        out.append([_np(x) for x in (h, *([g] if directional else g))])
    assert any(np.isnan(x).any() for x in out[1])
    np.testing.assert_array_equal(out[0][0], out[1][0])
    for a, b in zip(out[0][1:], out[1][1:]):
        np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
        m = np.isfinite(b)
        np.testing.assert_array_equal(m, np.isfinite(a))
        assert not m.any() or np.abs(a[m] - b[m]).max() <= \
            1e-12 * np.abs(b[m]).max()
