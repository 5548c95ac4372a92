"""The Dion step of small matrices taken together, ten launches over all of them (reference dion/dion.py:742-875), against the bucket-by-bucket launches (option
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
            elif isinstance(kind, int):     # zeros but for one element
                v = g.flatten()[kind].item()
                g.zero_().view(-1)[kind] = v
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


@pytest.mark.parametrize("dtype", [F32, BF])
@pytest.mark.parametrize("at", [0, 8191, 8192, 100 * 161 - 3, -1])
def test_one_element_is_found_wherever_it_is(dev, option, dtype, at):
    """B is not zero if one element is (the chunks of the pass that adds the gradient hold 8192): Q is not kept."""
    shapes, runs = [(100, 161), (161, 100)], []
    for mode, kind in ((0, at), (1, at), (1, "zero")):
        option("dion_small", mode)
        runs.append(_run(dev, shapes, dtype, 0.5, 1, 1, kind=kind)[0])
    for a, b, zero in zip(*runs):
        assert rel_fro(b[1], a[1]) <= (1e-4 if dtype == F32 else 1e-2)
        assert rel_fro(b[2], zero[2]) > 0.5


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


def _agree(shapes, runs, tol):
    for i, (a, b) in enumerate(zip(*runs)):
        for name, x, y in zip(("X", "M", "Q"), a, b):
            e = rel_fro(y, x)
            assert torch.isfinite(y.float()).all() and e <= tol, (i, shapes[i], name, e)


@pytest.mark.parametrize("shapes", [
    [(64, 96)] * 60 + [(96, 64)] * 36,                                  # the most matrices one launch takes
    [(64, 96)] * 60 + [(96, 64)] * 37,                                  # one more: bucket by bucket
    [(32 + 8 * i, 64 + 8 * i) for i in range(8)],                       # the most buckets
    [(32 + 8 * i, 64 + 8 * i) for i in range(9)],                       # one more
    [(64, 96)] * 200 + [(40, 72)],
])
def test_groups_around_the_limits_of_one_launch(dev, option, shapes):
    runs = []
    for mode in (0, 1):
        option("dion_small", mode)
        out, opt = _run(dev, shapes, F32, 0.5, 8, 2)
        runs.append(out)
        assert all(opt.state[p]["Q"].abs().sum() > 0 for p in opt.param_groups[0]["params"])
    _agree(shapes, runs, 2e-5)
    if len(shapes) > 96 or len(set(shapes)) > 8:                        # both took the same road
        for a, b in zip(*runs):
            assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_a_group_split_between_both_roads(dev, option):
    """Matrices of two dtypes in one group: the few fp32 ones go out in one launch, the many bf16 ones bucket by bucket, and every
    parameter is stepped exactly once."""
    from dion_amd import Dion

    shapes = [(64, 96)] * 5 + [(96, 64)] * 60 + [(128, 64)] * 50 + [(64, 64)] * 3
    dtypes = [F32] * 5 + [BF] * 110 + [F32] * 3
    runs = []
    for mode in (0, -1):
        option("dion_small", mode)
        gen = torch.Generator(device=dev).manual_seed(8)
        torch.manual_seed(8)
        params = [torch.nn.Parameter((torch.randn(s, generator=gen, device=dev) * 0.02).to(d)) for s, d in zip(shapes, dtypes)]
        opt = Dion(params, lr=0.02, rank_fraction=0.5)
        for p in params:      # (in one order, whichever road creates them)
            opt._get_or_initialize_state(p, opt.param_groups[0])
        for _ in range(2):
            for p in params:
                p.grad = (torch.randn(p.shape, generator=gen, device=dev) * 1e-2).to(p.dtype)
            opt.step()
        torch.cuda.synchronize()
        runs.append([(p.detach(), opt.state[p]["momentum"], opt.state[p]["Q"]) for p in params])
        assert len(opt.cholesky_info()) == 4 and all(int(v.max()) == 0 for v in opt.cholesky_info().values())
    fp32 = [i for i, d in enumerate(dtypes) if d == F32 and shapes[i][0] != shapes[i][1]]
    _agree([shapes[i] for i in fp32], [[r[i] for i in fp32] for r in runs], 2e-5)
    for i, (a, b) in enumerate(zip(*runs)):
        if dtypes[i] == BF:
            assert all(torch.equal(x, y) for x, y in zip(a, b)), i
        else:
            assert rel_fro(b[0], a[0]) <= 2e-5 and rel_fro(b[1], a[1]) <= 2e-5, i


@pytest.mark.parametrize("shape,shift", [((96, 160), 8), ((160, 96), 24), ((33, 64), 1), ((77, 53), 3)])
def test_dion_weights_off_the_128_byte_grid(dev, option, shape, shift):
    """Views of flat buffers that are only 16-byte aligned (off the 8-grid: aligned to their elements) are left to the bucket
    launches: the bits of aligned copies on that road, and nothing around the views is touched."""
    from dion_amd import Dion

    option("dion_small", 0)
    runs, numel = [], shape[0] * shape[1]
    for moved in (False, True):
        gen = torch.Generator(device=dev).manual_seed(9)
        torch.manual_seed(9)
        flats, params = [], []
        for _ in range(3):
            x = torch.randn(shape, generator=gen, device=dev) * 0.02
            if moved:
                flat = torch.full((numel + shift + 40,), 7.0, device=dev)
                flat[shift:shift + numel] = x.flatten()
                x = flat[shift:shift + numel].view(shape)
                assert x.data_ptr() % 128
                flats.append(flat)
            params.append(torch.nn.Parameter(x))
        opt = Dion(params, lr=0.02, rank_fraction=0.5)
        for p in params:
            p.grad = torch.randn(shape, generator=gen, device=dev) * 1e-2
        opt.step()
        torch.cuda.synchronize()
        runs.append([(p.detach().clone(), opt.state[p]["momentum"], opt.state[p]["Q"]) for p in params])
        for flat in flats:
            assert (flat[:shift] == 7).all() and (flat[shift + numel:] == 7).all()
        option("dion_small", 1)
    for a, b in zip(*runs):
        assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("dtype", [F32, BF])
@pytest.mark.parametrize("ms", [(127, 128, 129, 200), (191, 192, 193, 264), (255, 256, 257, 264), (319, 320, 321, 449)])
def test_numbers_of_stages_and_ragged_ends(dev, option, dtype, ms):
    """K loops of two to eight stages whose last one is whole, one element deep or ragged, B by rows and by columns."""
    shapes, runs = [(m, 72) for m in ms] + [(77, m) for m in ms], []
    for mode in (0, 1):
        option("dion_small", mode)
        runs.append(_run(dev, shapes, dtype, 0.5, 1, 2)[0])
    _agree(shapes, runs, 2e-5 if dtype == F32 else 1e-2)   # (as above)


@pytest.mark.parametrize("dtype", [F32, BF])
@pytest.mark.parametrize("shapes, fraction", [
    ([(768, 768)] * 4 + [(768, 3072), (3072, 768)], 0.25), ([(1024, 1024), (4096, 1024)], 0.25), ([(2048, 2048), (2048, 520)], 1 / 32)])
def test_medium_matrices(dev, option, dtype, shapes, fraction):
    """Widths and ranks up to where the rule takes all buckets together."""
    runs = []
    for mode in (0, -1):
        option("dion_small", mode)
        runs.append(_run(dev, shapes, dtype, fraction, 8, 2)[0])
    _agree(shapes, runs, 2e-5 if dtype == F32 else 1e-2)   # (as above)


@pytest.mark.parametrize("dtype", [F32, BF])
@pytest.mark.parametrize("n, rank, ms", [
    (3, 2, (65, 97, 129, 193, 257)),                    # (in bf16 stages of 64 k, in fp32 of 32)
    (2, 1, (65, 66, 97, 98, 129, 130)),
    (1, 1, (33, 39, 65, 71, 72, 135)),
    (5, 3, (65, 129)), (7, 4, (97, 193)), (9, 5, (65, 129)),
])
def test_tall_matrices_of_a_few_columns(dev, option, dtype, n, rank, ms):
    """B'^T P of matrices whose rows are shorter than the eight elements of a load: the loads of the last rows are moved back, also
    where the last stage of the K loop is shorter than they are many."""
    shapes, runs = [(m, n) for m in ms], []
    for mode in (0, 1):
        option("dion_small", mode)
        runs.append(_run(dev, shapes, dtype, rank / n, 1, 1, mu=0.5)[0])
        assert all(q.shape == (n, rank) for _, _, q in runs[-1])
    _agree(shapes, runs, 2e-5 if dtype == F32 else 1e-2)   # (as above)


def _step64(X, G, M, Q, mu):
    """Error feedback and Q of one step in 64 bits, on the CPU, from the states as they are held (X stands for the shape only)."""
    B, Q = M.cpu().double() + G.cpu().double(), Q.cpu().double()
    wide = X.size(0) < X.size(1)
    B = B.mT if wide else B
    P, U = torch.linalg.qr(B @ Q)
    P = P * U.diagonal().sign()
    R = B.mT @ P
    M = B - (1 - mu) * P @ R.mT
    return M.mT if wide else M, R / R.norm(dim=0)


@pytest.mark.parametrize("shape", [(200, 200), (256, 256), (256, 512)])
def test_full_rank_bf16_factors_are_as_exact_together_as_by_buckets(dev, option, shape):
    """Rank beyond 192 columns: P's rounding to bf16, which both roads share, times the factor's condition decides the error of a
    step against 64 bits (1e-2 to 1e-1 of Q); the order of operations of the factorisation does not show in it."""
    from dion_amd import Dion, DionMixedPrecisionConfig

    gen = torch.Generator(device=dev).manual_seed(11)
    torch.manual_seed(11)
    params = [torch.nn.Parameter((torch.randn(shape, generator=gen, device=dev) * 0.02).to(BF)) for _ in range(4)]
    opt = Dion(params, lr=0.02, mu=0.95, rank_fraction=1.0,
               mixed_precision_config=DionMixedPrecisionConfig(momentum_dtype=BF, Q_dtype=F32))
    for p in params:
        opt._get_or_initialize_state(p, opt.param_groups[0])
    for _ in range(3):
        grads = [(torch.randn(shape, generator=gen, device=dev) * 1e-2).to(BF) for _ in params]
        before = [(p.detach().clone(), opt.state[p]["momentum"].clone(), opt.state[p]["Q"].clone()) for p in params]
        errors = []
        for mode in (0, 1):
            option("dion_small", mode)
            for p, g, (x, m, q) in zip(params, grads, before):
                p.grad = g
                p.data.copy_(x)
                opt.state[p]["momentum"].copy_(m)
                opt.state[p]["Q"].copy_(q)
            opt.step()
            torch.cuda.synchronize()
            errors.append([])
            for p, g, (x, m, q) in zip(params, grads, before):
                m64, q64 = _step64(x, g, m, q, 0.95)
                errors[-1].append((rel_fro(opt.state[p]["momentum"], m64), rel_fro(opt.state[p]["Q"], q64)))
        for buckets, together in zip(*errors):
            assert all(t <= 1.01 * b for b, t in zip(buckets, together)), errors   # (measured: equal to four digits)
