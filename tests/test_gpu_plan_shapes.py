"""Source energies that do not fit the plan are refused: its kernels take the
sizes from the plan, the buffers theirs from the energy."""
import numpy as np
import pytest

from sparrowpy_amd import testing
from test_gpu_parity import (_grouped_and_generic, _oracle_directional,
                             ops)  # noqa: F401

pytestmark = pytest.mark.gpu


def test_energies_that_do_not_fit(ops):
    r = _oracle_directional(testing.shoebox_room_stub(2.5, 2., 1.5), .5,
                            n_points=(2, 4))
    r.init_source_energy(np.array([1.1, .8, .6]))
    e0, d0 = r.energy_init_source, r.distance_patches_to_source
    tail = (343., 1 / 2000, 100, 2)
    for plan in _grouped_and_generic(ops, r, 343., 1 / 2000):
        for f in (ops.exchange_orders, ops.exchange_sum):
            for e in (e0[:-1], e0[:, :-1], e0[..., :-1]):
                with pytest.raises(ValueError, match="the plan has"):
                    f(plan, e, d0, *tail)
            with pytest.raises(ValueError, match="distance_0"):
                f(plan, e0, d0[:-1], *tail)
            with pytest.raises(ValueError, match="need a plan"):
                f(None, e0, d0, *tail)
            f(None, e0, d0, *tail[:-1], 0)
