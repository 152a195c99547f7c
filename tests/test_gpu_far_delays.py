"""Delays of more bins than a number holds are reported as those beyond the
histogram are."""
import pytest

from sparrowpy_amd import testing
from sparrowpy_amd.coordinates import Coordinates, FrequencyData

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("speed", [1., 1e-300, 5e-324])
@pytest.mark.parametrize("orders", [0, 2])
def test_slow_sound(speed, orders):
    from sparrowpy_amd import DirectionalRadiosityFast
    r = DirectionalRadiosityFast.from_polygon(
        testing.shoebox_room_stub(2., 2., 2.), 1.)
    r.set_air_attenuation(FrequencyData([0.], [1000.]))
    r.bake_geometry()
    r.init_source_energy(Coordinates(.6, .5, .4))
    with pytest.raises(IndexError):
        r.calculate_energy_exchange(speed, 1e-3, .1, orders)
