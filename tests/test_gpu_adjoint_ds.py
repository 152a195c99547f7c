"""One backward order of the diffuse + specular plan at the edges of its
tiling (8 waves of whole directions, 64 entries to a block, two at a time, 128
or 256 bins) against float64 torch, on random transposed entries.

Tolerances: mu_out is lambda plus a float64 sum rounded to float32, added in
float32 -- two roundings, 2^-24 of the sum of the magnitudes each; the table
gradients are float64 sums of products in another order, at most 4,000 terms:
4,000 * 2^-53 < 1e-12 of the sum of the magnitudes.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,entries", [(1, 1), (1, 300), (3, 17), (16, 130),
                                       (64, 61), (64, 700)])
@pytest.mark.parametrize("T", [1, 64, 127, 128, 129, 256, 257, 700])
def test_adjoint_ds_edges(D, entries, T):
    import torch
    from sparrowpy_amd import _hip
    P, B = 3, 2
    gen = torch.Generator().manual_seed(1000 * D + entries + T)

    def rand(*shape):
        return torch.rand(*shape, generator=gen, dtype=torch.float64) - .5

    def ints(n, *shape):
        return torch.randint(n, shape, generator=gen)
    # source 1 has no entry, and of the others not every direction has one
    src = ints(2, entries).sort().values * 2
    order = (src * D + ints(D, entries)).sort().values
    src, d = order // D, order % D
    j, m = ints(P, entries), ints(D, entries)
    lag = ints(T + 40, entries)
    last = torch.ones(entries, dtype=torch.bool)
    last[:-1] = order[1:] != order[:-1]
    tgptr = torch.searchsorted(order, torch.arange(P * D + 1))
    wa, wc = rand(B, entries), rand(B, entries)
    lam, mu, ek = (rand(P, D, B, T).float() for _ in range(3))
    musum = mu.double().sum(1).float()

    def ahead(x):       # x [..., T] of each entry, moved ahead by its delay
        t = torch.arange(T) + lag[:, None, None]
        y = torch.gather(x, 2, t.clamp(max=T - 1).expand(entries, B, T))
        return torch.where(t < T, y, 0.)
    x, y = ahead(musum.double()[j]), ahead(mu.double()[j, m])
    e = ek.double()[src, d]
    terms = wa.T[..., None] * x + wc.T[..., None] * y
    size = (wa.T[..., None] * x).abs() + (wc.T[..., None] * y).abs()
    want = lam.double().reshape(P * D, B, T).index_add(0, order, terms)
    bound = lam.double().abs().reshape(P * D, B, T).index_add(0, order, size)
    g = torch.stack([(e * x).sum(2).T, (e * y).sum(2).T])
    g_size = torch.stack([(e * x).abs().sum(2).T, (e * y).abs().sum(2).T])

    def dev(t, dtype):
        return t.to(dtype).contiguous().cuda()
    i32, f64 = torch.int32, torch.float64
    out = torch.full((P, D, B, T), float("nan"), device="cuda")
    ga = torch.ones(2, B, entries, dtype=f64, device="cuda")
    a = [dev(tgptr, torch.int64), dev(d << 25 | j, i32),
         dev(lag | torch.where(last, 0x40000000, 0), i32), dev(m, i32),
         dev(wa, f64), dev(wc, f64)] + [dev(t, torch.float32)
                                        for t in (lam, musum, mu, ek)]
    _hip.call("spr_exchange_adjoint_ds", P, D, B, T, entries,
              *(_hip.ptr(t) for t in a), _hip.ptr(out), _hip.ptr(ga),
              _hip.stream_ptr())
    err = (out.cpu().double().reshape(P * D, B, T) - want).abs()
    assert (err <= 2 ** -23 * bound).all()
    err = (ga.cpu() - 1 - g).abs()
    assert (err <= 1e-12 * (1 + g_size)).all()
