"""The one-launch fp64 pass over the matrices that the orthonormaliser's fp32 pass could not do (reference dion/dion.py:1267-1308),
against Householder QR in fp64: ill-conditioned factors among ordinary ones, at the edges of its 32 / 64 tiles and of its eight
queues."""
import pytest
import torch

from conftest import rel_fro

pytestmark = pytest.mark.gpu


def _factors(batch, rows, r, cond):
    """Every third factor ill-conditioned (singular values over a range of `cond`), the others Gaussian."""
    gen = torch.Generator().manual_seed(5)
    P = torch.randn(batch, rows, r, generator=gen, dtype=torch.float64)
    for b in range(0, batch, 3):
        U, _ = torch.linalg.qr(P[b])
        V, _ = torch.linalg.qr(torch.randn(r, r, generator=gen, dtype=torch.float64))
        P[b] = (U * torch.logspace(0, -torch.log10(torch.tensor(float(cond))).item(), r, dtype=torch.float64)) @ V.T
    return P


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch,rows,r", [(1, 300, 27), (4, 512, 64), (10, 1001, 65), (3, 1100, 200), (17, 264, 33), (2, 1500, 260)])
def test_flagged_factors_match_householder(dev, dtype, batch, rows, r):
    from dion_amd import _lib
    from dion_amd.newton_schulz import orthonormalize

    P = _factors(batch, rows, r, 1e6 if dtype == torch.float32 else 3e3).to(dtype)
    try:
        _lib.set_option("ns_flow_fail", 1)      # (a launch that gave up: NaN in what it works on)
        poisoned = torch.isnan(orthonormalize(P.to(dev)).float()).flatten(1).any(1).cpu()
    finally:
        _lib.set_option("ns_flow_fail", 0)
    assert poisoned.tolist() == [b % 3 == 0 for b in range(batch)]
    Q, info = orthonormalize(P.to(dev), return_info=True)
    assert Q.dtype == dtype and bool((info == 0).all())
    eye = torch.eye(r, dtype=torch.float64)
    for b in range(batch):
        q = Q[b].double().cpu()
        Qh, Rh = torch.linalg.qr(P[b].double())
        Qh = Qh * torch.sign(torch.diagonal(Rh))
        assert (q.T @ q - eye).norm().item() <= (1e-4 if dtype == torch.float32 else 4e-2) * max(1.0, (r / 64) ** 0.5)
        assert rel_fro(q, Qh) <= (1e-5 if b % 3 == 0 else 1e-4) + (0 if dtype == torch.float32 else 5e-3), b


def test_flagged_rank_deficient_factor_drops_columns(dev):
    """Columns that depend on earlier ones come out as zero and are reported; the others are orthonormal."""
    from dion_amd.newton_schulz import orthonormalize

    torch.manual_seed(1)
    P = torch.randn(2, 640, 72)
    P[1, :, 40:50] = P[1, :, 10:20] + P[1, :, 20:30]
    Q, info = orthonormalize(P.to(dev), return_info=True)
    assert int(info[0]) == 0 and 41 <= int(info[1]) <= 50
    q = Q[1].double().cpu()
    live = q.norm(dim=0) > 0.5
    assert live[:40].all() and torch.isfinite(q).all() and int(live.sum()) >= 62 - 10
    q = q[:, live]
    assert (q.T @ q - torch.eye(q.size(1), dtype=torch.float64)).norm().item() <= 5e-3   # (fp64 noise of the dependent columns, squared)
