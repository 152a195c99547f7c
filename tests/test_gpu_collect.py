"""Mono collection at the edges of its tiling (16 waves of patches, 64 terms
at a time, 256 bins) against float64 torch.

Tolerance: the float64 sums are rounded to float32 once (2^-24), non-negative
terms; twice that for the sums' own rounding.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 15, 17, 1023, 1025, 1100])
@pytest.mark.parametrize("T", [1, 255, 257, 700])
def test_collect_mono_edges(P, T):
    import torch
    from sparrowpy_amd import ops
    gen = torch.Generator().manual_seed(P * 1000 + T)

    def rand(*shape):
        return torch.rand(*shape, generator=gen, dtype=torch.float64).cuda()
    R, D, B, c, dt = 2, 3, 2, 343., 1 / 4000
    etc = rand(P, D, B, T).float()
    pts, ctr = 9 * rand(R, 3), 9 * rand(P, 3)
    idx = (rand(R, P) * D).long().clamp(max=D - 1)
    # a third of the patches unseen; receiver 1 sees none
    factor = rand(R, P) * (rand(R, P) > 1 / 3)
    factor[1] = 0
    air = rand(B) * .01
    out = ops.collect(etc, pts, ctr, idx, factor, air, c, dt)
    d = ctr[None] - pts[:, None]
    dist = torch.sqrt((d[..., 0] ** 2 + d[..., 1] ** 2) + d[..., 2] ** 2)
    n = torch.ceil(dist / c / dt).long()
    ref = torch.zeros(R, B, T, dtype=torch.float64, device="cuda")
    t = torch.arange(T, device="cuda")
    for r in range(R):
        rows = etc[torch.arange(P, device="cuda"), idx[r]].double()
        ts = ((t - n[r][:, None]) % T)[:, None].expand(P, B, T)
        w = factor[r][:, None] * torch.exp(-air * dist[r][:, None])
        ref[r] = (rows.gather(2, ts) * w[..., None]).sum(0)
    torch.testing.assert_close(out.double(), ref, rtol=2 ** -23, atol=0)
