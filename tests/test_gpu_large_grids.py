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
