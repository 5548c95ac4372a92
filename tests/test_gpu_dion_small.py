"""The one-launch Dion kernel for small matrices (reference dion/dion.py:742-875) against the bucket-by-bucket launches (option
"dion_small" = 0), which the oracle checks: shapes around the 32 / 64 tile edges, ranks around the blocks of the factorisation,
rows off every alignment, more and fewer matrices than queues, zero and rank-deficient gradients."""
import pytest
import torch

from conftest import rel_fro

pytestmark = pytest.mark.gpu

BF, F32 = torch.bfloat16, torch.float32


@pytest.fixture
def option():
    from dion_amd import _lib

    yield _lib.set_option
    _lib.set_option("dion_small", -1)
    _lib.set_option("ns_flow_fail", 0)


def _run(dev, shapes, dtype, fraction, multiple, steps, mu=0.95, kind="random"):
    from dion_amd import Dion

    gen = torch.Generator(device=dev).manual_seed(7)
    torch.manual_seed(7)
    params = [torch.nn.Parameter((torch.randn(s, generator=gen, device=dev) * 0.02).to(dtype)) for s in shapes]
    opt = Dion(params, lr=0.02, mu=mu, weight_decay=0.01, rank_fraction=fraction, rank_multiple_of=multiple)
    for _ in range(steps):
        for p in params:
            g = torch.randn(p.shape, generator=gen, device=dev) * 1e-2
            if kind == "zero":
                g.zero_()
            elif kind == "deficient":
                g[:, g.size(1) // 4:] = 0
                g[g.size(0) // 4:, :] = 0
            p.grad = g.to(dtype)
        opt.step()
    torch.cuda.synchronize()
    return [(p.detach(), opt.state[p]["momentum"], opt.state[p]["Q"]) for p in params], opt


@pytest.mark.parametrize("dtype", [F32, BF])
@pytest.mark.parametrize("shapes,fraction,multiple", [
    ([(1, 1), (3, 2), (8, 8)], 1.0, 1),
    ([(64, 64), (65, 63), (63, 65), (128, 192), (192, 128)], 0.5, 1),
    ([(33, 1000), (1000, 33), (301, 100)], 1.0, 1),
    ([(256, 256)] * 9 + [(1024, 256)] * 2 + [(256, 1024)], 0.5, 8),
    ([(341, 127), (127, 341), (257, 520)], 0.25, 1),
    ([(256, 300)] * 2, 1.0, 1),                         # four blocks of the factorisation
    ([(2048, 400)], 0.5, 1),                            # eight K slices of the Gram product, the last one ragged
])
def test_small_dion_kernel_agrees_with_bucket_launches(dev, option, dtype, shapes, fraction, multiple):
    runs = []
    for mode in (0, 1):
        option("dion_small", mode)
        runs.append(_run(dev, shapes, dtype, fraction, multiple, 2)[0])
    tol = 2e-5 if dtype == F32 else 1e-2
    for i, (a, b) in enumerate(zip(*runs)):
        for name, x, y in zip(("X", "M", "Q"), a, b):
            e = rel_fro(y, x)
            assert torch.isfinite(y.float()).all() and e <= tol * (100 if name == "Q" and min(shapes[i]) == max(shapes[i]) else 1), \
                (i, shapes[i], name, e)


@pytest.mark.parametrize("dtype", [F32, BF])
def test_small_dion_kernel_zero_and_deficient_gradients(dev, option, dtype):
    """A zero gradient keeps Q (up to its normalisation) and decays the weights; a rank-deficient one takes the second pass of
    the orthonormaliser (the noise columns differ between the two roads, the update of the weights' range does not)."""
    shapes = [(96, 200), (200, 96), (256, 160)]
    for kind in ("zero", "deficient"):
        runs, infos = [], []
        for mode in (0, 1):
            option("dion_small", mode)
            out, opt = _run(dev, shapes, dtype, 0.5, 1, 1, kind=kind)
            runs.append(out)
            infos.append([int(v.max()) > 0 for v in opt._info.values()])
        assert infos[0] == infos[1]
        for i, (a, b) in enumerate(zip(*runs)):
            assert all(torch.isfinite(t.float()).all() for t in b)
            if kind == "zero":
                assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
                assert rel_fro(b[2], a[2]) <= (1e-6 if dtype == F32 else 5e-3)
            else:
                assert rel_fro(b[1], a[1]) <= (1e-4 if dtype == F32 else 1e-2), (i, rel_fro(b[1], a[1]))


def test_a_small_dion_launch_that_gave_up_poisons_the_result(dev, option):
    """The status word set before the launch (as by a wait beyond its limit): weights, momentum and Q are NaN."""
    option("dion_small", 1)
    option("ns_flow_fail", 1)
    out, _ = _run(dev, [(96, 160), (160, 96)], F32, 0.5, 1, 1)
    assert all(torch.isnan(t).all() for tri in out for t in tri)
    option("ns_flow_fail", 0)
    out, _ = _run(dev, [(96, 160), (160, 96)], F32, 0.5, 1, 1)
    assert all(torch.isfinite(t).all() for tri in out for t in tri)


def test_the_profile_books_the_one_launch_step_as_itself(dev, option):
    """A step of small matrices is one kind of its own with the step's flops: no update pass, no orthonormaliser ran."""
    from dion_amd import _lib

    lib, shapes = _lib.load(), [(96, 160), (160, 96)]
    option("dion_small", 1)
    try:
        _lib.check(lib.dion_amd_profile_reset(), "reset")
        _lib.check(lib.dion_amd_profile_enable(1), "enable")
        _run(dev, shapes, F32, 0.5, 1, 3)
        prof = _lib.profile_read()
    finally:
        lib.dion_amd_profile_enable(0)
        lib.dion_amd_profile_reset()
    assert set(prof) == {"dion_small"}
    launches, ms, work = prof["dion_small"]
    assert launches == 3 and ms > 0 and work == 3 * 2 * 8.0 * 96 * 160 * 48
