"""The 64 x 64 diagonal block of the blocked Cholesky factorisations (csrc/diag64.h) and the triangular solve behind them
(csrc/gemm_f64.hip), through the orthonormaliser: ranks at the edges of the block's panels of 16 columns, columns of zeros, whose
pivots fail, at their first and last columns, whole and ragged rows, one and several matrices to an XCD; and the bf16 products
with the triangular factors (csrc/gemm_bf16.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS32 = 2.0**-24


def _factor(m, r, seed):
    """Columns of a random orthonormal basis with scales between 1 and 4 and a mixing that keeps the condition below 20."""
    g = torch.Generator().manual_seed(seed)
    U = torch.linalg.qr(torch.randn(m, r, generator=g, dtype=torch.float64))[0]
    V = torch.linalg.qr(torch.randn(r, r, generator=g, dtype=torch.float64))[0]
    return (U * torch.linspace(1, 4, r, dtype=torch.float64)) @ V


def _q64(P):
    """Thin-QR factor with a positive diagonal of R, in 64 bits."""
    Q, R = torch.linalg.qr(P.double())
    return Q * torch.sign(torch.diagonal(R))


@pytest.mark.parametrize("r", [1, 8, 15, 16, 17, 24, 40, 48, 63, 64, 65, 80, 127, 128, 200])
@pytest.mark.parametrize("qr_method", ["qr", "cqr"])
def test_ranks_at_the_edges_of_the_panels(r, qr_method):
    from dion_amd.newton_schulz import orthonormalize

    m = 4 * r + 24
    P = torch.stack([_factor(m, r, s) for s in range(3)]).float()
    # fp64 pass: the result is rounded once, 2^-24 of an entry, which is at most 1; and the pass works in fp64.
    # fp32 pass alone: sums of m products of fp32 numbers, and the condition (4) squared: 16 eps sqrt(m) a column and a
    # hundred times that as the safe side.
    passes = 1 if qr_method == "qr" else 2
    tol = 4 * EPS32 if qr_method == "qr" else 100 * 16 * EPS32 * m**0.5
    Q, info = orthonormalize(P.cuda(), passes=passes, qr_method=qr_method, return_info=True)
    assert not info.any()
    for b in range(3):
        assert (Q[b].cpu().double() - _q64(P[b])).norm() <= tol * r**0.5


@pytest.mark.parametrize("col", [0, 5, 15, 16, 31, 32, 47, 48, 63, 64, 79])
def test_a_column_of_zeros_is_dropped_and_reported(col):
    from dion_amd.newton_schulz import orthonormalize

    m, r = 300, 80
    P = torch.stack([_factor(m, r, s) for s in range(2)]).float()
    P[1, :, col] = 0
    Q, info = orthonormalize(P.cuda(), passes=1, qr_method="qr", return_info=True)
    assert info.tolist() == [0, col + 1]
    assert not Q[1, :, col].any()
    keep = [j for j in range(r) if j != col]
    assert (Q[1].cpu().double()[:, keep] - _q64(P[1][:, keep])).norm() <= 4 * EPS32 * r**0.5
    assert (Q[0].cpu().double() - _q64(P[0])).norm() <= 4 * EPS32 * r**0.5


@pytest.mark.parametrize("batch, m, r", [(1, 64, 64), (3, 352, 192), (8, 64, 64), (9, 100, 64), (11, 288, 128), (17, 129, 65), (2, 1000, 320)])
@pytest.mark.parametrize("qr_method", ["qr", "cqr"])
def test_solve_over_batches_and_ragged_rows(batch, m, r, qr_method):
    from dion_amd.newton_schulz import orthonormalize

    P = torch.stack([_factor(m, r, s) for s in range(batch)]).float()
    passes = 1 if qr_method == "qr" else 2
    tol = 4 * EPS32 if qr_method == "qr" else 100 * 16 * EPS32 * m**0.5   # (as above)
    Q = orthonormalize(P.cuda(), passes=passes, qr_method=qr_method).cpu().double()
    for b in range(batch):
        assert (Q[b] - _q64(P[b])).norm() <= tol * r**0.5


@pytest.mark.parametrize("batch, r", [(1, 128), (2, 136), (1, 320), (1, 520), (2, 768)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_products_with_triangular_factors(batch, r, dtype):
    """P T and the correction, whose column tiles stop their sums at the triangle's edge (one, whole and ragged tiles)."""
    from dion_amd.newton_schulz import orthonormalize

    m = 4 * r
    P = torch.stack([_factor(m, r, s) for s in range(batch)]).to(dtype)
    one = orthonormalize(P.cuda(), qr_method="cqr").cpu().double()
    two = orthonormalize(P.cuda(), qr_method="rcqr").cpu().double()
    # Storing: half an ulp of every entry.  cqr: fp32 sums of m products, the condition squared (as above).  rcqr: the
    # defect D that cqr leaves, squared, and the two bf16 operands of its correction; the fp32 product P T, condition 4.
    ulp = (2.0**-9 if dtype == torch.bfloat16 else EPS32) * r**0.5
    for b in range(batch):
        q = _q64(P[b])
        assert (one[b] - q).norm() <= ulp + 100 * 16 * EPS32 * m**0.5 * r**0.5
        D = 0.0 if dtype == torch.bfloat16 else float((one[b].T @ one[b] - torch.eye(r, dtype=torch.float64)).norm())
        assert (two[b] - q).norm() <= ulp + D * D + 2.0**-8 * D + 16 * 4 * EPS32 * r**0.5
