"""Calls whose blocks hold 2^32 work items or more, beyond one launch: small
arrays with one bin, so that every receiver, source or destination takes a
block of its own."""
import pytest

pytestmark = pytest.mark.gpu


def test_mono_collection_of_many_receivers():
    """1,024 work items a receiver; etc * factor * exp(-air * distance) in
    float64, rounded to float32 once."""
    import torch
    from sparrowpy_amd import ops
    n = (1 << 22) + 5
    gen = torch.Generator("cuda").manual_seed(0)
    f64 = dict(dtype=torch.float64, device="cuda", generator=gen)
    points = torch.rand(n, 3, **f64)
    factor = torch.rand(n, 1, **f64)
    idx = torch.zeros(n, 1, dtype=torch.int64, device="cuda")
    etc = torch.full((1, 1, 1, 1), .75, dtype=torch.float32, device="cuda")
    centers = torch.tensor([[2., 3., 4.]], dtype=torch.float64, device="cuda")
    air = torch.tensor([.01], dtype=torch.float64, device="cuda")
    out = ops.collect(etc, points, centers, idx, factor, air, 343., 1.,
                      patchwise=False)
    dist = (points - centers).norm(dim=1, keepdim=True)
    want = .75 * factor * torch.exp(-.01 * dist)
    assert float((out.double().reshape(n, 1) / want - 1).abs().max()) \
        <= 2 ** -23


@pytest.mark.parametrize("shape", [-1, 0, 2, 4])
def test_orders_of_many_destinations_and_bands(shape):
    """512 work items a destination and band in the one-launch order, which
    the two passes take over.  Each destination hears the next patch at once:
    every bin of the sum is a product chain, two roundings an order."""
    import torch
    from sparrowpy_amd import ops
    P, B, K = 8200, 1024, 2
    gen = torch.Generator("cuda").manual_seed(1)
    f64 = dict(dtype=torch.float64, device="cuda")
    n = torch.arange(P + 1, device="cuda")
    rowid = ((n[:-1] + 1) % P).to(torch.int32)
    lag = torch.full((P,), ops.GroupedPlan.LAST_IN_GROUP, dtype=torch.int32,
                     device="cuda")
    scal = torch.rand(B, P, generator=gen, **f64) + .5
    rtab = torch.rand(1, B, 1, generator=gen, **f64) + .5
    plan = ops.GroupedPlan(P, 1, B, n, n, n, torch.zeros_like(rowid), rowid,
                           lag, scal, rtab)
    plan.order_shape = shape
    e0 = torch.rand(P, 1, B, generator=gen, **f64) + .5
    out = ops.exchange_orders(plan, e0, torch.zeros(P, **f64), 343., 1., 1,
                              K)
    term, want = e0[:, 0], e0[:, 0].clone()
    for _ in range(K):
        term = term.roll(-1, 0) * scal.T * rtab[0, :, 0]
        want += term
    err = float((out.double().reshape(P, B) / want - 1).abs().max())
    assert err <= (2 * K + 2) * 2.0 ** -24


def test_adjoint_of_many_sources_and_bands():
    """512 work items a source and band: one entry each, so mu is lambda plus
    two products, rounded to float32 and added to it."""
    import torch
    from sparrowpy_amd import _hip
    P, B = 8200, 1024
    gen = torch.Generator("cuda").manual_seed(2)

    def rand(*shape, dtype=torch.float32):
        return torch.rand(*shape, dtype=dtype, generator=gen,
                          device="cuda") + .5
    lam, mu, ek = (rand(P, B) for _ in range(3))
    wa, wc = (rand(B, P, dtype=torch.float64) for _ in range(2))
    n = torch.arange(P + 1, device="cuda")
    i32 = dict(dtype=torch.int32, device="cuda")
    tkey = ((n[:-1] + 1) % P).to(torch.int32)
    tlag = torch.full((P,), 0x40000000, **i32)
    out = torch.full((P, B), float("nan"), device="cuda")
    ga = torch.zeros(2, B, P, dtype=torch.float64, device="cuda")
    _hip.call("spr_exchange_adjoint_ds", P, 1, B, 1, P,
              *(_hip.ptr(t) for t in (n, tkey, tlag, torch.zeros(P, **i32),
                                      wa, wc, lam, mu, mu, ek, out, ga)),
              _hip.stream_ptr())
    heard = mu.double().roll(-1, 0)
    want = lam.double() + heard * (wa + wc).T
    assert float((out.double() / want - 1).abs().max()) <= 2 ** -23
    want = heard * ek.double()
    assert float((ga.transpose(1, 2) / want - 1).abs().max()) <= 1e-12


def test_gather_on_many_diffuse_specular_tiles():
    """1,024 work items a tile, band and 256 bins: a scene's tiles behind half
    a million empty ones give the sums they give by themselves."""
    import dataclasses

    import torch
    from sparrowpy_amd import ops, testing
    from test_gpu_parity import _ds_plan, _oracle_directional
    r = _oracle_directional(testing.shoebox_room_stub(2.5, 2., 1.5), .5,
                            n_bands=4, seed=3)
    plan = _ds_plan(ops, r, 343., 1 / 2000)
    tiles = ops.tile_plan(plan, 16, min_merge=0)
    empty, T = 1 << 19, 300
    before = torch.zeros(empty, dtype=torch.int64, device="cuda")
    many = dataclasses.replace(
        tiles, P=tiles.P + 16 * empty, tptr=torch.cat([before, tiles.tptr]),
        **{k: torch.cat([before.repeat(16), getattr(tiles, k)])
           for k in ("gstart", "gdiff")})
    shape = (plan.P, plan.D, plan.B, T)
    gen = torch.Generator("cuda").manual_seed(4)
    prev = torch.rand(shape, device="cuda", generator=gen)
    sums = []
    for plan.tiles in (tiles, many):
        out = torch.zeros(plan.n_groups, plan.B, T, device="cuda")
        ops.gather_groups(plan, shape, prev, out)
        sums.append(out)
    assert float(sums[0].max()) > 0
    assert torch.equal(*sums)
