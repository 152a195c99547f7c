"""Diffuse + specular plans with destinations that no entry reaches in a
specular direction: fully diffuse walls (scattering 1), all of them or all
but one, and one direction.  Such a destination has the diffuse group alone,
which starts at its row's end.

Histograms against the oracle's FP64 loop: the tolerance of a sum of orders,
each rounded to float32 twice.  Gradients of float32 histograms: 1e-4 of the
largest component.
"""
import numpy as np
import pytest

from conftest import make_oracle, rel_err_within_db
from oracle import adjoint as oadj
from sparrowpy_amd import brdf as B
from sparrowpy_amd import samplings, testing
from sparrowpy_amd.coordinates import Coordinates, FrequencyData
from test_gpu_parity import _ds_plan, _np, ops  # noqa: F401
from test_gpu_sums import _check

pytestmark = pytest.mark.gpu

FREQS = np.array([500., 1000.])
SRC = np.array([1.1, .8, .6])
RCV = np.array([[1.9, 1.2, 1.], [.7, .9, .4]])
C, DT = 343., 1 / 2000


def _walls_and_brdfs(D, specular):
    """A room whose walls scatter everything but those of ``specular``."""
    rng = np.random.default_rng(5)
    walls = testing.shoebox_room_stub(2.5, 2., 1.5)
    dirs = samplings.hemisphere(samplings.sph_gaussian(
        n_points={8: (2, 8), 32: (4, 16)}[D])) if D > 1 \
        else Coordinates(np.zeros(1), np.zeros(1), np.ones(1))
    brdfs = []
    for w in range(len(walls)):
        alpha = rng.uniform(.05, .3, (1, 2))
        if D == 1:
            freq = np.ones((1, 1, 2)) * (1 - alpha) / np.pi
            brdfs.append(FrequencyData(freq, FREQS))
            continue
        s = rng.uniform(.2, .8, (1, 2)) if w in specular else np.ones((1, 2))
        brdfs.append(B.create_from_scattering(
            dirs, dirs, FrequencyData(s, FREQS), FrequencyData(alpha, FREQS)))
    return walls, dirs, brdfs


def _oracle(walls, dirs, brdfs):
    r = make_oracle(walls, .5)
    for w, br in enumerate(brdfs):
        r.set_wall_brdf([w], br.freq, dirs.cartesian, dirs.cartesian, FREQS)
    r.set_air_attenuation(np.array([1e-3, 3e-3]), FREQS)
    r.bake_geometry()
    r.init_source_energy(SRC)
    return r


@pytest.mark.parametrize("shape", [-1, 0, 2, 4])
@pytest.mark.parametrize("D,specular", [(1, ()), (8, ()), (8, (0,)),
                                        (32, ()), (32, (4,))])
def test_rows_without_a_specular_direction(ops, D, specular, shape):
    r = _oracle(*_walls_and_brdfs(D, specular))
    plan = _ds_plan(ops, r, C, DT)
    groups = np.diff(_np(plan.grp_ptr))
    entries = np.diff(_np(plan.row_ptr))
    assert ((groups == 1) & (entries > 8)).any()
    assert specular == () or groups.max() > 1
    plan.order_shape = shape
    for K in (1, 6):
        _check(ops, r, plan, 301, DT, K)


@pytest.mark.parametrize("D,specular", [(1, ()), (8, ()), (8, (0,))])
@pytest.mark.parametrize("shape", [-1, 0, 2, 4])
def test_adjoint_without_a_specular_direction(ops, D, specular, shape):
    import torch
    from sparrowpy_amd import DirectionalRadiosityFast, adjoint
    walls, dirs, brdfs = _walls_and_brdfs(D, specular)
    T, K = 200, 4
    o = _oracle(walls, dirs, brdfs)
    o.calculate_energy_exchange(C, DT, T * DT, K)
    want = o.collect_energy_receiver_mono(RCV)
    grad = np.random.default_rng(2).uniform(-1., 1., want.shape)
    gt = oadj.gradient(o, RCV, grad, K)
    r = DirectionalRadiosityFast.from_polygon(walls, .5)
    for w, br in enumerate(brdfs):
        r.set_wall_brdf([w], br, dirs, dirs)
    r.set_air_attenuation(FrequencyData(np.array([1e-3, 3e-3]), FREQS))
    r.bake_geometry()
    adj = adjoint.ExchangeAdjoint(r, Coordinates(*SRC), Coordinates(*RCV.T),
                                  C, DT, (T + .5) * DT, K, checkpoint_every=2)
    adj.plan.order_shape = shape
    H = _np(adj.forward(adj.A0, adj.C0))
    assert rel_err_within_db(H, want) <= (2 * K + 4) * 2.0 ** -24
    gA, _ = adj.backward(torch.tensor(grad, device="cuda"))
    ref = gt.sum(1)     # a diffuse constant feeds every direction
    assert np.abs(_np(gA) - ref).max() <= 1e-4 * np.abs(ref).max()
