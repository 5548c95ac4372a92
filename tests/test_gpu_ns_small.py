"""The one-launch Newton-Schulz kernel for small matrices (reference dion/muon.py:620-647) against the product-by-product
launches (option "ns_flow" = 0): the tiles compute the same values in the same order of k, so every result must be the same
bits -- on shapes around the 32 / 64 tile edges, off every alignment grid, with fewer and more matrices than queues."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


@pytest.fixture
def flow_option():
    from dion_amd import _lib

    yield lambda mode: _lib.set_option("ns_flow", mode)
    _lib.set_option("ns_flow", -1)


@pytest.mark.parametrize("batch,m,n,steps", [
    (1, 1, 1, 5), (1, 64, 64, 5), (3, 65, 63, 5), (2, 64, 129, 3), (1, 256, 768, 5), (9, 192, 320, 5), (17, 128, 96, 8),
    (1, 448, 512, 2), (1, 33, 1000, 1), (2, 301, 100, 5),
])
def test_newton_schulz_small_kernel_equals_product_launches(dev, flow_option, batch, m, n, steps):
    from dion_amd.newton_schulz import newton_schulz

    torch.manual_seed(3)
    G = torch.randn(batch, m, n, device=dev)
    coeffs = [(3.4445, -4.7750, 2.0315)] * steps
    for src in (G, G.to(BF)):
        flow_option(0)
        ref = newton_schulz(src, coeffs=coeffs)
        flow_option(-1)
        got = newton_schulz(src, coeffs=coeffs)
        torch.cuda.synchronize()
        assert torch.isfinite(got.float()).all() and torch.equal(ref, got)


@pytest.mark.parametrize("dtype", [BF, torch.float32])
@pytest.mark.parametrize("shapes", [
    [(64, 27), (27, 64), (77, 77), (301, 100), (100, 301), (301, 100)],     # five buckets: a second round of one
    [(128, 128)] * 12,
    [(256, 256)] * 16 + [(1024, 256)] * 4 + [(256, 1024)] * 4,
    [(8, 200)] * 90 + [(200, 8)],                                           # more matrices than one staging launch takes
])
def test_muon_step_small_kernel_equals_product_launches(dev, flow_option, shapes, dtype):
    from dion_amd import Muon

    runs = []
    for mode in (0, -1):
        flow_option(mode)
        gen = torch.Generator(device=dev).manual_seed(5)
        params = [torch.nn.Parameter((torch.randn(s, generator=gen, device=dev) * 0.02).to(dtype)) for s in shapes]
        opt = Muon(params, lr=0.02, mu=0.95, weight_decay=0.01, nesterov=True)
        for _ in range(2):
            for p in params:
                p.grad = (torch.randn(p.shape, generator=gen, device=dev) * 1e-3).to(dtype)
            opt.step()
        torch.cuda.synchronize()
        runs.append([(p.detach().clone(), opt.state[p]["momentum"].clone()) for p in params])
    for i, ((xa, ma), (xb, mb)) in enumerate(zip(*runs)):
        assert torch.isfinite(xb.float()).all() and torch.equal(xa, xb), f"weights differ, matrix {i} {shapes[i]}"
        assert torch.equal(ma, mb), f"momentum differs, matrix {i}"


def test_a_small_launch_that_gave_up_poisons_the_result(dev, flow_option):
    """The status word set before the launch (as by a wait beyond its limit): every result is NaN, the next call is clean."""
    from dion_amd import _lib
    from dion_amd.newton_schulz import newton_schulz

    G = torch.randn(3, 96, 160, device=dev)
    try:
        _lib.set_option("ns_flow_fail", 1)
        out = newton_schulz(G)
        torch.cuda.synchronize()
        assert torch.isnan(out.float()).all()
    finally:
        _lib.set_option("ns_flow_fail", 0)
    assert torch.isfinite(newton_schulz(G).float()).all()
