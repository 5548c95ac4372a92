"""Lion / AdamW updates for the non-matrix parameter groups (embeddings, lm_head, norms, biases).

Same signatures as the reference's `lion_update_foreach` / `adamw_update_foreach`
(dion/scalar_opts.py:152-187, 89-149); the work is one fused HIP pass per call
(`dion_amd_lion_step`, `dion_amd_adamw_step`) that reproduces the rounding of each of the
reference's tensor ops.  GPU tensors only: there is no CPU or PyTorch fallback.
"""
from typing import List

from torch import Tensor

from . import _lib


def lion_update_foreach(X: List[Tensor], G: List[Tensor], M: List[Tensor],
                        lr: Tensor, beta1: Tensor, beta2: Tensor, weight_decay: Tensor):
    """reference dion/scalar_opts.py:152-187."""
    assert len(X) == len(G) == len(M)
    _lib.host().element_lists(False, list(X), list(G), list(M), None, float(lr), float(beta1), float(beta2),
                              float(weight_decay), 0, 0.0)


def adamw_update_foreach(X: List[Tensor], G: List[Tensor], M: List[Tensor], V: List[Tensor],
                         lr: Tensor, beta1: Tensor, beta2: Tensor, weight_decay: Tensor, step, epsilon):
    """reference dion/scalar_opts.py:89-149."""
    assert len(X) == len(G) == len(M) == len(V)
    _lib.host().element_lists(True, list(X), list(G), list(M), list(V), float(lr), float(beta1), float(beta2),
                              float(weight_decay), float(step), float(epsilon))


def element_groups_step(opt, groups, adamw):
    """Lion or AdamW step of parameter groups of an optimizer (states are created where they are missing).

    Groups with equal hyper-parameters go out together, in one launch: the updates are element by element, and a launch
    over a few small tensors is mostly its own latency (24 fp32 matrices with two Lion and two AdamW groups: 255 -> 247 us)."""
    host = _lib.host()
    calls = {}
    for group in groups:
        key = (float(group["lr"]), float(group["beta1"]), float(group["beta2"]), float(group["weight_decay"]))
        key += (float(group["step"]), float(group["epsilon"])) if adamw else (0.0, 0.0)
        calls.setdefault(key, []).append(group)
    for key, members in calls.items():
        params = members[0]["params"] if len(members) == 1 else [p for g in members for p in g["params"]]
        args = (adamw, params, opt.state, *key)
        missing = host.element_group(*args)
        if missing is not None:
            for p in missing:
                opt._new_state(p, members[0])
            _lib.require_states(host.element_group(*args), f"{type(opt).__name__}.step")
