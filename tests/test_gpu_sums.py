"""The sum of all orders, order by order (spr_exchange_orders) and by the recurrence x_{k+1} = x_0 + A x_k
(spr_exchange_sum), on every plan form, against the oracle's FP64 loop.

Tolerance: every term of an order is non-negative, so a sum's relative
error is at most that of its terms; an order rounds to float32 at most twice
(group sums, histogram), x_0 once: after K orders (2 K + 1) * 2^-24, plus
one more for float64 rounding.  Bins within 60 dB of their histogram's peak
(float32 denormals carry no relative error).
"""
import numpy as np
import pytest

import oracle as orc
from conftest import rel_err_within_db
from sparrowpy_amd import testing
from test_gpu_parity import (_ds_plan, _grouped_and_generic, _np,
                             _oracle_directional, ops)  # noqa: F401

pytestmark = pytest.mark.gpu

SRC = np.array([1.1, .8, .6])
ROOM = (2.5, 2., 1.5)


@pytest.fixture(scope="module")
def rooms():
    out = {}
    for n in ((2, 4), (4, 8), (6, 8), (8, 16)):
        r = _oracle_directional(testing.shoebox_room_stub(*ROOM), .5,
                                n_points=n, seed=3)
        r.init_source_energy(SRC)
        out[r.brdf_out.shape[1]] = r
    return out


def _plan(ops, r, form, dt):
    grouped, pairs = _grouped_and_generic(ops, r, 343., dt)
    if form == "pairs":
        return pairs
    plan = _ds_plan(ops, r, 343., dt) if form.startswith("ds") else grouped
    tiles = form.split("-")[1:]
    plan.order_shape = -1
    if tiles and tiles[0] == "row":
        plan.order_shape = int(tiles[1])
    elif tiles:
        plan.tiles = ops.tile_plan(plan, int(tiles[0]), min_merge=0)
        plan.tiles.R = int(tiles[1]) if len(tiles) > 1 else 8
    return plan


def _check(ops, r, plan, T, dt, K):
    args = (plan, r.energy_init_source, r.distance_patches_to_source, 343.,
            dt, T, K)
    ref = orc.exchange(T, r.energy_init_source, r.distance_patches_to_source,
                       r.pair_distances(), r.fft, r.p2o, 343., dt, K,
                       r.visible_patches, nthreads=8)
    # with the tightest reach, and with none
    far = int(np.max(r.distance_patches_to_source) / 343. / dt) + 1
    outs = [_np(f(*args, far)) for f in (ops.exchange_orders,
                                         ops.exchange_sum)]
    for f, out in zip((ops.exchange_orders, ops.exchange_sum), outs):
        np.testing.assert_array_equal(_np(f(*args)), out)
    for out in outs:
        assert np.isfinite(out).all()
        assert (out[ref == 0] == 0).all()
        err = rel_err_within_db(out, ref)
        print(f"[sum] T={T} K={K}: max rel err {err:.3e}")
        assert err <= (2 * K + 2) * 2.0 ** -24
    return outs[0]


@pytest.mark.parametrize("form", ["pairs", "grouped", "grouped-4",
                                  "grouped-8", "grouped-16-8",
                                  "grouped-16-16", "grouped-row-2",
                                  "grouped-row-4", "ds", "ds-16", "ds-row-2",
                                  "ds-row-4"])
@pytest.mark.parametrize("D", [4, 16, 24, 64])
def test_sum_matches_oracle(ops, rooms, form, D):
    """Every plan form and padded direction count; 301 bins (no whole
    number of time blocks), an odd and an even number of orders."""
    r = rooms[D]
    dt = 1 / 2000
    plan = _plan(ops, r, form, dt)
    for K in (5, 6):
        _check(ops, r, plan, 301, dt, K)


@pytest.mark.parametrize("form", ["pairs", "grouped-16-8", "grouped-row-2",
                                  "grouped-row-4", "ds"])
@pytest.mark.parametrize("K", [1, 2, 7])
def test_orders_give_the_stepped_total(ops, rooms, form, K):
    """One call gives the bits of stepping an ExchangeState."""
    r = rooms[16]
    plan = _plan(ops, r, form, 1 / 2000)
    T = 301
    out = _check(ops, r, plan, T, 1 / 2000, K)
    st = ops.ExchangeState(*r.energy_init_source.shape, T)
    st.init(r.energy_init_source, r.distance_patches_to_source, 343.,
            1 / 2000)
    for _ in range(K):
        st.step(plan)   # always two passes
    np.testing.assert_array_equal(out, _np(st.finalize()))


@pytest.mark.parametrize("form", ["pairs", "grouped", "grouped-16-8",
                                  "grouped-row-2", "grouped-row-4", "ds",
                                  "ds-row-2", "ds-row-4"])
@pytest.mark.parametrize("T,K", [(1, 0), (75, 1), (1500, 2), (4099, 3),
                                 (2049, 6)])
def test_sum_lengths_and_orders(ops, rooms, form, T, K):
    """One bin and no order, one order, delays of hundreds of bins beyond
    the kernels' lane strides (48 kHz), many time blocks."""
    r = rooms[16]
    dt = 1. if T == 1 else 1 / 2000 if T == 75 else 1 / 48000
    _check(ops, r, _plan(ops, r, form, dt), T, dt, K)


@pytest.mark.parametrize("shape", [-1, 0, 2, 4])
@pytest.mark.parametrize("walls", [[0], [0, 1], [0, 2], [0, 1, 2, 3]])
def test_rows_without_brdf(ops, walls, shape):
    """One direction and one group per destination (the waves share it), and
    destinations with no source at all (walls in one plane, or facing away)."""
    from conftest import make_oracle
    room = testing.shoebox_room_stub(*ROOM)
    r = make_oracle([room[w] for w in walls], .25)
    r.set_air_attenuation(np.array([1e-3]), np.array([1000.]))
    r.bake_geometry()
    r.init_source_energy(SRC)
    args = (r.visibility_matrix, r.patches_center, r.patches_area,
            r.form_factors, r.p2o, r.air, r.patch_to_wall_ids, None, None,
            None, 1, 1, 343., 1 / 2000)
    plan = ops.GroupedPlan.from_geometry(*args)
    plan.order_shape = shape
    _check(ops, r, plan, 200, 1 / 2000, 4)


def test_sum_reports_delay_beyond_histogram(ops, rooms):
    r = rooms[16]
    plan = _plan(ops, r, "grouped", 1 / 2000)
    args = (plan, r.energy_init_source, r.distance_patches_to_source, 343.,
            1 / 2000)
    for f in (ops.exchange_orders, ops.exchange_sum):
        with pytest.raises(IndexError):
            f(*args, 3, 2)
        with pytest.raises(ValueError):
            f(*args, 100, 2, reach=3)


def test_split_walls_give_the_rows_orders(ops):
    """A BRDF per patch (one wall each): tiles across the walls of a plane,
    the bits of the row-by-row plan."""
    from sparrowpy_amd import DirectionalRadiosityFast, samplings
    from sparrowpy_amd import brdf as B
    from sparrowpy_amd.coordinates import Coordinates, FrequencyData
    from sparrowpy_amd.geometry import Polygon, create_patches
    rng = np.random.default_rng(0)
    dirs = samplings.hemisphere(samplings.sph_gaussian(sh_order=3))
    f = np.array([500.])
    walls = [Polygon(p, w.up_vector, w.normal)
             for w in testing.shoebox_room_stub(3, 2.5, 2)
             for p in create_patches(w.pts, .5)]
    r = DirectionalRadiosityFast.from_polygon(walls, .5)
    for i in range(len(walls)):
        r.set_wall_brdf([i], B.create_from_scattering(
            dirs, dirs, FrequencyData(rng.uniform(.2, .8, (1, 1)), f),
            FrequencyData(rng.uniform(.1, .3, (1, 1)), f)), dirs, dirs)
    r.bake_geometry()
    r.init_source_energy(Coordinates(*SRC))
    plan = r._exchange_plan(343., 1 / 2000)
    assert plan.diffuse_specular and plan.tiles is not None
    plan.order_shape = -1
    outs = []
    for tiles in (plan.tiles, None):
        plan.tiles = tiles
        outs.append(_np(ops.exchange_orders(
            plan, r._energy_init_source, r._distance_patches_to_source, 343.,
            1 / 2000, 333, 5)))
    np.testing.assert_array_equal(*outs)
