"""Order loops whose waves share a sum, formed in parts: the diffuse sums of a
diffuse + specular plan and the group of a plan with one group per destination
in the one-launch order.  They give the stepped total to float32 rounding, not
bit for bit: each is within (2 K + 2) 2^-24 of the exact sum."""
import numpy as np
import pytest

from conftest import make_oracle, rel_err_within_db
from sparrowpy_amd import testing
from test_gpu_parity import _np, ops  # noqa: F401
from test_gpu_sums import ROOM, SRC, _plan, rooms  # noqa: F401

pytestmark = pytest.mark.gpu

DT, T = 1 / 2000, 301


def _compare(ops, r, plan, K):
    args = (r.energy_init_source, r.distance_patches_to_source, 343., DT)
    st = ops.ExchangeState(*r.energy_init_source.shape, T)
    st.init(*args)
    for _ in range(K):
        st.step(plan)
    want = _np(st.finalize())
    far = int(r.distance_patches_to_source.max() / 343. / DT) + 1
    for reach in (far, None):
        out = _np(ops.exchange_orders(plan, *args, T, K, reach))
        assert (out[want == 0] == 0).all()
        assert rel_err_within_db(out, want) <= 2 * (2 * K + 2) * 2.0 ** -24


@pytest.mark.parametrize("shape", [0, 2, 4])
@pytest.mark.parametrize("D", [4, 16, 64])
@pytest.mark.parametrize("K", [1, 6])
def test_diffuse_sums(ops, rooms, D, shape, K):
    plan = _plan(ops, rooms[D], "ds", DT)
    plan.order_shape = shape
    _compare(ops, rooms[D], plan, K)


@pytest.mark.parametrize("shape", [0, 2, 4])
@pytest.mark.parametrize("K", [1, 6])
def test_the_only_group(ops, shape, K):
    r = make_oracle(testing.shoebox_room_stub(*ROOM), .5)
    r.set_air_attenuation(np.array([1e-3]), np.array([1000.]))
    r.bake_geometry()
    r.init_source_energy(SRC)
    plan = ops.GroupedPlan.from_geometry(
        r.visibility_matrix, r.patches_center, r.patches_area, r.form_factors,
        r.p2o, r.air, r.patch_to_wall_ids, None, None, None, 1, 1, 343., DT)
    plan.order_shape = shape
    _compare(ops, r, plan, K)
