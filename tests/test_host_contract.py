"""CPU-side contract of the entry points and of the host module: what they accept, what they refuse, and how often they run what
a user registered.  Nothing is launched: library calls end at a workspace of no bytes, steps at a missing GPU."""
import ctypes

import pytest
import torch

ALIGN, WORKSPACE = -2, -3
BASE = 0x7F0000000000     # addresses that are looked at, never followed


def _pointers(offset, count=2):
    return (ctypes.c_void_p * count)(*[BASE + i * (1 << 24) + offset for i in range(count)])


@pytest.mark.parametrize("m,n", [(33, 64), (64, 33), (33, 65), (1, 8), (4095, 4096)])
def test_matrices_off_the_8_grid_need_only_the_alignment_of_their_elements(m, n):
    """A view into a flat buffer may start anywhere when a dimension is no multiple of 8 (reference dion/muon.py:525-573 takes
    any tensor): the check behind the addresses, that of the workspace's size, is the one that answers."""
    from dion_amd import _lib

    lib = _lib.load()
    coeffs = _lib.float_array([1.0, 1.0, 1.0])
    for code, size in ((_lib.BF16, 2), (_lib.F32, 4)):
        for offset, want in ((0, WORKSPACE), (size, WORKSPACE), (8, WORKSPACE), (size // 2, ALIGN)):
            ptrs = _pointers(offset)
            rc = lib.dion_amd_newton_schulz(BASE + offset, code, m * n, n, BASE, m * n, n, 1, m, n, coeffs, 1, 1e-7, _lib.BF16, 1,
                                            BASE, 0, None)
            assert rc == want, (m, n, code, offset)
            assert lib.dion_amd_muon_step(ptrs, ptrs, ptrs, 2, m, n, code, code, 0.9, 0, 1.0, 0.1, coeffs, 1, 1e-7, 1,
                                          BASE, 0, None) == want
            k = _lib.MuonBucket()
            k.X = k.G = k.M = ctypes.cast(ptrs, ctypes.POINTER(ctypes.c_void_p))
            k.batch, k.m, k.n, k.decay, k.adjusted_lr = 2, m, n, 1.0, 0.1
            assert lib.dion_amd_muon_step_buckets(ctypes.byref(k), 1, code, code, 0.9, 0, coeffs, 1, 1e-7, 1, BASE, 0, None) == want


def test_matrices_on_the_8_grid_need_16_byte_alignment():
    from dion_amd import _lib

    lib = _lib.load()
    coeffs = _lib.float_array([1.0, 1.0, 1.0])
    for offset, want in ((0, WORKSPACE), (16, WORKSPACE), (8, ALIGN)):
        ptrs = _pointers(offset)
        assert lib.dion_amd_newton_schulz(BASE + offset, _lib.BF16, 0, 64, BASE, 0, 64, 1, 32, 64, coeffs, 1, 1e-7, _lib.BF16, 1,
                                          BASE, 0, None) == want
        assert lib.dion_amd_muon_step(ptrs, ptrs, ptrs, 2, 32, 64, _lib.F32, _lib.F32, 0.9, 0, 1.0, 0.1, coeffs, 1, 1e-7, 1,
                                      BASE, 0, None) == want


def _buckets(spec):
    from dion_amd import _lib

    arr = (_lib.MuonBucket * len(spec))()
    for k, (batch, m, n) in zip(arr, spec):
        k.batch, k.m, k.n = batch, m, n
    return arr


def _unpadded(batch, m, n):
    """Two iterates and two Gram-sized matrices in bf16 with every dimension and pitch on the 8-grid (and off multiples of 4 KiB),
    the partial sums and control words: what the iteration cannot do without, per bucket."""
    m, n = sorted((-(-m // 8) * 8, -(-n // 8) * 8))
    pitch = lambda k: k + (64 if k * 2 % 4096 == 0 else 0)
    return batch * (2 * 2 * m * pitch(n) + 2 * 2 * m * pitch(m) + 4 * (m // 32 + 1) * (n // 64 + 2) + 4096)


@pytest.mark.parametrize("spec", [
    [(224, 16, 4096), (224, 4096, 16)],             # the factors of a low-rank adapter: 115 MiB, padded to tiles 939
    [(224, 64, 4096), (224, 4096, 64)],
    [(128, 136, 4096)], [(1600, 72, 72)], [(32, 24, 50000)], [(256, 8, 8192)],
    [(48, 768, 768), (96, 16, 768)],                # beside a bucket on the tile grid
    [(256, 300, 300)], [(24, 1096, 1096)], [(4, 648, 10000)], [(14, 341, 1021)],
])
def test_workspace_of_thin_matrices_is_not_a_multiple_of_their_own_size(spec):
    """Padding to whole tiles may add 70 per cent to the working matrices, not a factor of eight (a call of more work than the
    one-launch kernel takes)."""
    from dion_amd import _lib

    lib = _lib.load()
    got = lib.dion_amd_muon_buckets_workspace_bytes(_buckets(spec), len(spec))
    assert 0 < got <= 1.75 * sum(_unpadded(*k) for k in spec)


def test_workspace_holds_either_layout():
    """Few thin matrices go to the one-launch kernel, whose tiles are 64 wide: the queries make room for that."""
    from dion_amd import _lib

    lib = _lib.load()
    tiles = 3 * 2 * (2 * 64 * 4096 + 2 * 64 * 64)
    assert lib.dion_amd_muon_buckets_workspace_bytes(_buckets([(3, 16, 4096)]), 1) >= tiles
    assert lib.dion_amd_ns_workspace_bytes(3, 16, 4096, _lib.BF16) >= tiles
    assert lib.dion_amd_muon_workspace_bytes(3, 4096, 16) >= tiles
    # one matrix of a batch that goes through in chunks
    assert lib.dion_amd_ns_workspace_bytes(1, 16, 4096, _lib.F32) < 4 * 4 * 16 * 4096


@pytest.mark.parametrize("m,n", [
    (648, 10000), (10000, 648), (640, 10000),
    # working sets without padding within a kilobyte of the array
    (200, 41736), (232, 35920), (400, 20568), (536, 15112), (616, 13000), (1072, 6752), (1232, 5576), (1304, 5128),
])
def test_static_newton_schulz_takes_what_fits_without_padding(m, n):
    """The working set that has to fit the array is the one on the 8-grid: 26.3 MiB for 648 x 10000, which padding makes 32.4.
    (A misaligned source: the call ends at that check, or here at the missing GPU, and nothing is launched.)"""
    from dion_amd import _lib

    coeffs = _lib.float_array([1.0, 1.0, 1.0])
    args = (BASE + 1, _lib.BF16, m * n, n, BASE, m * n, n, 1, m, n, coeffs, 1, 1e-7, _lib.BF16, 1, None)
    rc = _lib.load().dion_amd_newton_schulz_static(*args)
    assert rc == ALIGN or rc > 0, rc


@pytest.mark.parametrize("m,n", [(4096, 4096), (648, 13000), (64, 200000)])
def test_static_newton_schulz_refuses_what_does_not_fit(m, n):
    from dion_amd import _lib

    coeffs = _lib.float_array([1.0, 1.0, 1.0])
    args = (BASE + 1, _lib.BF16, m * n, n, BASE, m * n, n, 1, m, n, coeffs, 1, 1e-7, _lib.BF16, 1, None)
    assert _lib.load().dion_amd_newton_schulz_static(*args) == -5


# ------------------------------------------------------------------ step hooks
def _optimizers():
    from dion_amd import Dion, DionReference, Muon

    return [Muon, Dion, DionReference]


def _record(opt):
    seen = []
    opt.register_step_pre_hook(lambda o, args, kwargs: seen.append(("pre", args, kwargs)))
    opt.register_step_post_hook(lambda o, args, kwargs: seen.append(("post", args, kwargs)))
    return seen


def _parameters():
    return [torch.nn.Parameter(torch.zeros(8, 8))]     # without gradients: a step has nothing to do


@pytest.mark.parametrize("cls", _optimizers())
@pytest.mark.parametrize("plain_first", [False, True])
def test_step_hooks_run_once_in_a_subclass(cls, plain_first):
    """A subclass whose step() calls super().step(): hooks act once per step, whether or not the class itself has been
    instantiated before, and through as many levels as there are."""
    class Mine(cls):
        def step(self, closure=None):
            return super().step(closure)

    class Deeper(Mine):
        def step(self, closure=None):
            return super().step(closure=closure)

    class Inherits(Deeper):
        pass

    if plain_first:
        cls(_parameters()).step()
    for kind in (Mine, Deeper, Inherits, cls):
        opt = kind(_parameters())
        seen = _record(opt)
        for n in (1, 2):
            assert opt.step() is None
            assert [s[0] for s in seen] == ["pre", "post"] * n, kind
        assert opt.param_groups[0]["step"] == 2
        with pytest.raises(ZeroDivisionError):
            opt.step(lambda: 1 / 0)
        del seen[:]
        assert opt.step(lambda: 7) == 7                 # an exception leaves nothing behind
        assert [s[0] for s in seen] == ["pre", "post"], kind


@pytest.mark.parametrize("cls", _optimizers())
def test_step_hooks_get_the_arguments_of_the_call(cls):
    """As torch's own optimizers hand them on."""
    closure = lambda: None
    calls = [lambda o: o.step(), lambda o: o.step(closure), lambda o: o.step(closure=closure)]
    want, got = [], []
    for kind, out in ((torch.optim.SGD, want), (cls, got)):
        opt = kind(_parameters(), lr=0.1)
        seen = _record(opt)
        for call in calls:
            call(opt)
        out += [(when, len(args), args[1:], kwargs, args[0] is opt) for when, args, kwargs in seen]
    assert got == want


@pytest.mark.parametrize("cls", _optimizers())
def test_global_hooks_and_the_profiler_see_every_step(cls):
    from torch.optim.optimizer import register_optimizer_step_post_hook, register_optimizer_step_pre_hook

    opt, seen = cls(_parameters()), []
    handles = [register_optimizer_step_pre_hook(lambda o, a, k: seen.append("pre")),
               register_optimizer_step_post_hook(lambda o, a, k: seen.append("post"))]
    opt.step()
    for h in handles:
        h.remove()
    opt.step()
    assert seen == ["pre", "post"]
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        opt.step()
    assert [e.name for e in prof.events()].count(f"Optimizer.step#{cls.__name__}.step") == 1
    scheduler = torch.optim.lr_scheduler.LambdaLR(opt, lambda epoch: 1.0)     # (it wraps the bound method)
    opt.step()
    scheduler.step()
    assert opt.param_groups[0]["step"] == 4


# ------------------------------------------------------------------ what the native module is handed
def _groups():
    """One optimizer for every road through the native module: Muon, Dion and both element-wise algorithms."""
    from dion_amd import Dion, Muon

    return [(Muon, "muon"), (Muon, "lion"), (Muon, "adamw"), (Dion, "dion"), (Dion, "lion"), (Dion, "adamw")]


@pytest.mark.parametrize("cls,algorithm", _groups())
@pytest.mark.parametrize("kind", [tuple, list, lambda ps: dict.fromkeys(ps)])
def test_parameters_of_a_group_may_be_any_collection(cls, algorithm, kind):
    """`group["params"]` is walked, not assumed to be a list."""
    from dion_amd import _lib

    params = [torch.nn.Parameter(torch.zeros(8, 8)) for _ in range(5)]
    opt = cls([dict(params=params, algorithm=algorithm)])
    opt.param_groups[0]["params"] = kind(params)
    opt.step()                                    # no gradients: nothing to do
    params[3].grad = torch.zeros(8, 8)
    with pytest.raises(_lib.DionAmdError, match="tensor is on cpu"):
        opt.step()
    assert list(opt.state) == [params[3]]
    opt.param_groups[0]["params"] = kind([])
    opt.step()
    opt.param_groups[0]["params"] = 3
    with pytest.raises(TypeError):
        opt.step()


@pytest.mark.parametrize("cls,algorithm", _groups())
def test_a_state_that_stays_missing_is_an_error(cls, algorithm):
    """A parameter whose state is not there after it was asked for is not skipped in silence."""
    from dion_amd import _lib

    class Forgets(cls):
        def _get_or_initialize_state(self, param, algo):
            return {}

    p = torch.nn.Parameter(torch.zeros(8, 8))
    p.grad = torch.zeros(8, 8)
    opt = Forgets([dict(params=[p], algorithm=algorithm)])
    with pytest.raises(_lib.DionAmdError, match="state"):
        opt.step()


@pytest.mark.parametrize("cls,algorithm", _groups())
def test_a_state_may_be_any_mapping(cls, algorithm):
    """What is not a dict is asked for its tensors like one; one that lacks a tensor is a KeyError."""
    from collections import UserDict

    from dion_amd import _lib

    p = torch.nn.Parameter(torch.zeros(8, 8))
    p.grad = torch.zeros(8, 8)
    opt = cls([dict(params=[p], algorithm=algorithm)])
    for state in (UserDict, dict):
        opt.state[p] = state(momentum=torch.zeros(8, 8), variance=torch.zeros(8, 8), Q=torch.zeros(8, 8))
        with pytest.raises(_lib.DionAmdError, match="tensor is on cpu"):
            opt.step()
        opt.state[p] = state(other=torch.zeros(8, 8))
        with pytest.raises(KeyError, match="momentum"):
            opt.step()
    opt.state = UserDict({p: dict(momentum=torch.zeros(8, 8), variance=torch.zeros(8, 8), Q=torch.zeros(8, 8))})
    with pytest.raises(_lib.DionAmdError, match="tensor is on cpu"):
        opt.step()


@pytest.mark.parametrize("shape,flatten,momentum", [
    ((8, 16), False, (8, 8)), ((8, 16), False, (8, 32)), ((3, 8, 16), False, (2, 8, 16)), ((3, 8, 16), True, (3, 8)),
    ((4, 8), False, (0, 8)),
])
def test_muon_refuses_a_momentum_of_another_size(shape, flatten, momentum):
    """A buffer that is not as large as its parameter would be read and written out of its bounds."""
    from dion_amd import Muon, _lib

    p = torch.nn.Parameter(torch.zeros(shape))
    p.grad = torch.zeros(shape)
    opt = Muon([p], flatten=flatten)
    opt.state[p]["momentum"] = torch.zeros(momentum)
    with pytest.raises(_lib.DionAmdError, match="do not fit"):
        opt.step()
    opt.state[p]["momentum"] = torch.zeros(shape, dtype=torch.bfloat16)      # half the bytes
    with pytest.raises(_lib.DionAmdError, match="do not fit"):
        opt.step()
    opt.state[p]["momentum"] = torch.zeros(p.numel()).view(shape)
    with pytest.raises(_lib.DionAmdError, match="tensor is on cpu"):
        opt.step()
    p.data = torch.zeros((2 * shape[0],) + shape[1:])                        # the gradient is the old one's
    opt.state[p]["momentum"] = torch.zeros(p.shape)
    with pytest.raises(_lib.DionAmdError, match="do not fit"):
        opt.step()


def test_profile_kinds_have_the_names_of_the_header():
    import os
    import re

    from dion_amd import _lib

    header = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "dion_amd.h")).read()
    kinds = {int(v): k for k, v in re.findall(r"#define DION_AMD_PROF_([A-Z_]+) (\d+)", header) if k != "KINDS"}
    assert sorted(kinds) == list(range(len(_lib.PROF_KINDS)))
    assert int(re.search(r"DION_AMD_PROF_KINDS (\d+)", header).group(1)) == len(kinds)
    assert [kinds[i].lower().replace("_", "") for i in sorted(kinds)] == [n.replace("_", "") for n in _lib.PROF_KINDS]
    lib = _lib.load()
    out = (ctypes.c_longlong(), ctypes.c_double(), ctypes.c_double())
    assert [lib.dion_amd_profile_read(k, *(ctypes.byref(o) for o in out)) for k in (len(kinds) - 1, len(kinds))] == [0, -1]


def test_what_the_one_launch_dion_step_takes():
    """Up to 96 matrices in 8 buckets, weights and momentum on the 128-byte grid, gradients and Q on the 16-byte one."""
    from dion_amd import _lib

    lib = _lib.load()

    def need(spec, x=0, m=0, g=0, q=0):
        arr, keep = (_lib.DionBucket * len(spec))(), []
        for k, (count, rows, cols) in zip(arr, spec):
            tables = [_pointers(off, count) for off in (x, g, m, q)]
            keep.append(tables)
            k.X, k.G, k.M, k.Q = (ctypes.cast(t, ctypes.POINTER(ctypes.c_void_p)) for t in tables)
            k.batch, k.m, k.n, k.r, k.scaled_lr = count, rows, cols, min(rows, cols) // 2, 0.1
        return lib.dion_amd_dion_buckets_workspace_bytes(arr, len(spec), _lib.F32, _lib.F32, _lib.F32, _lib.F32)

    buckets = [(2, 32 + 8 * i, 64 + 8 * i) for i in range(9)]
    try:
        _lib.set_option("dion_small", 1)
        assert need([(96, 64, 96)]) > 0 and need([(60, 64, 96), (36, 96, 64)]) > 0 and need(buckets[:8]) > 0
        assert need([(97, 64, 96)]) == 0 and need([(60, 64, 96), (37, 96, 64)]) == 0 and need(buckets) == 0
        assert need([(2, 64, 96)], g=16, q=16, x=128, m=256) > 0
        for kw in (dict(x=64), dict(m=16), dict(g=8), dict(q=4)):
            assert need([(2, 64, 96)], **kw) == 0, kw
        _lib.set_option("dion_small", 0)
        assert need([(2, 64, 96)]) == 0
    finally:
        _lib.set_option("dion_small", -1)
