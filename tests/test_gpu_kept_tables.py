"""The device's copies of BRDF tables and air attenuation, uploaded with the
first source, follow the object's own arrays."""
import numpy as np
import pytest

from sparrowpy_amd import brdf as B
from sparrowpy_amd import samplings, testing
from sparrowpy_amd.coordinates import Coordinates, FrequencyData

pytestmark = pytest.mark.gpu

FREQS = np.array([500., 1000.])
SRC, RCV = Coordinates(1.1, .8, .6), Coordinates(1.9, 1.2, 1.)
DIRS = samplings.hemisphere(samplings.sph_gaussian(sh_order=1))
TURN = np.array([[.8, .6, 0.], [-.6, .8, 0.], [0., 0., 1.]])   # 37 degrees
TURNED = Coordinates(*(DIRS.cartesian @ TURN).T)


def _brdf(s, alpha):
    return B.create_from_scattering(
        DIRS, DIRS, FrequencyData(np.full((1, 2), s), FREQS),
        FrequencyData(np.full((1, 2), alpha), FREQS))


def _room():
    from sparrowpy_amd import DirectionalRadiosityFast
    r = DirectionalRadiosityFast.from_polygon(
        testing.shoebox_room_stub(2.5, 2., 1.5), .5)
    r.set_wall_brdf(np.arange(6), _brdf(.4, .2), DIRS, DIRS)
    r.set_air_attenuation(FrequencyData(np.array([1e-3, 2e-3]), FREQS))
    return r


def _histogram(r):
    r.bake_geometry()
    r.init_source_energy(SRC)
    r.calculate_energy_exchange(343., 1 / 2000, .1, 3, recalculate=True)
    return r.collect_energy_receiver_mono(RCV).time


def _change(r, what):
    if what == "brdf":
        r.set_wall_brdf([1, 4], _brdf(.7, .5), DIRS, DIRS)
    elif what == "air":
        r.set_air_attenuation(FrequencyData(np.array([.2, .3]), FREQS))
    else:
        with pytest.raises(IndexError):     # wall 0 is changed before wall 99
            r.set_wall_brdf([0, 99], _brdf(.7, .5), TURNED, TURNED)


@pytest.mark.parametrize("what", ["brdf", "air", "brdf of a missing wall"])
def test_a_later_change_reaches_the_next_source(what):
    r = _room()
    before = _histogram(r)
    _change(r, what)
    after = _histogram(r)
    assert not np.array_equal(before, after)
    fresh = _room()
    _change(fresh, what)
    np.testing.assert_array_equal(after, _histogram(fresh))
