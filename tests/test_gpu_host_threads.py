"""The native host module and other threads of the program: the interpreter lock is free while the library is called, and
optimizers that step in threads of their own get the results of stepping one after the other."""
import ctypes
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _params(dev, seed, shapes=((64, 96), (96, 64), (128, 128))):
    gen = torch.Generator(device=dev).manual_seed(seed)
    params = [torch.nn.Parameter(torch.randn(s, generator=gen, device=dev) * 0.02) for s in shapes]
    for p in params:
        p.grad = torch.randn(p.shape, generator=gen, device=dev) * 1e-3
    return params


def _optimizers(dev, seed):
    from dion_amd import Dion, Muon

    torch.manual_seed(seed)
    return [Muon(_params(dev, seed)), Dion(_params(dev, seed), rank_fraction=0.5),
            Muon([dict(params=_params(dev, seed), algorithm="lion", lr=1e-3)]),
            Muon([dict(params=_params(dev, seed), algorithm="adamw", lr=1e-3)])]


def test_the_interpreter_lock_is_free_during_library_calls(dev):
    """In the place of the library's step functions: the interpreter's own question whether this thread holds the lock.  Yes is 1,
    which a step reports as an error."""
    from dion_amd import _lib

    lib, host = _lib.load(), _lib.host()
    address = lambda f: ctypes.cast(f, ctypes.c_void_p).value
    asks = address(ctypes.pythonapi.PyGILState_Check)
    opts = _optimizers(dev, 0)
    for opt in opts:
        opt.step()
    real = [address(getattr(lib, "dion_amd_" + n)) for n in ("muon_buckets_workspace_bytes", "muon_step_buckets", "lion_step",
                                                             "adamw_step", "dion_buckets_workspace_bytes", "dion_step_buckets")]
    calls = list(real)
    for i in (1, 2, 3, 5):
        calls[i] = asks
    try:
        host.bind(_lib.DionAmdError, _lib.check, *calls)
        for opt in opts:
            opt.step()
    finally:
        host.bind(_lib.DionAmdError, _lib.check, *real)


def test_optimizers_stepping_in_threads(dev):
    """Four optimizers, a thread and a stream each, 20 steps: the bits of the same steps one after the other."""
    def run(threaded):
        opts = _optimizers(dev, 3)
        torch.cuda.synchronize()
        errors = []

        def work(opt):
            try:
                with torch.cuda.stream(torch.cuda.Stream(device=dev)):
                    for _ in range(20):
                        opt.step()
                    torch.cuda.current_stream().synchronize()
            except Exception as e:   # noqa: BLE001 (handed to the main thread)
                errors.append(e)

        threads = [threading.Thread(target=work, args=(o,)) for o in opts]
        for t in threads:
            t.start()
            if not threaded:
                t.join()
        for t in threads:
            t.join()
        assert not errors, errors
        return [p.detach().clone() for o in opts for g in o.param_groups for p in g["params"]]

    for a, b in zip(run(False), run(True)):
        assert torch.isfinite(b).all() and torch.equal(a, b)
