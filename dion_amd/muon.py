"""`Muon` optimizer whose matrix path runs on the MI355X kernels.

Signature-compatible with the reference class (dion/muon.py:25-131): same constructor
arguments and defaults, same param-group keys, same `self.state` layout
(`state[p]["momentum"]`, plus `"variance"` for AdamW groups), same exceptions.  One GPU
only: `distributed_mesh` must be None.

Per `step()` the matrices of every "muon" group are bucketed by (shape, dtype) -- the
grouping rule of `create_param_batches` (reference dion/opt_utils.py:48-65) -- by the native host
module (`csrc/host.cpp`) and handed, as arrays of device pointers, to `dion_amd_muon_step_buckets`,
which runs the fused momentum pass, the batched Newton-Schulz GEMMs and the fused weight update on
the current stream.
"""
import ctypes
import math
from collections import defaultdict
from typing import Callable, Optional, Tuple

import torch
from torch import Tensor
from torch.optim.optimizer import ParamsT

from . import _lib
from .elementwise_opts import element_groups_step
from .newton_schulz import NS_SCHEDULE_COEFFS, flat_coeffs, zeropower_via_newtonschulz5


def adjust_lr_rms_norm(lr, param_shape):
    """reference dion/muon.py:596-602"""
    A, B = param_shape[-2:]
    return lr * (0.2 * math.sqrt(max(A, B)))


def adjust_lr_spectral_norm(lr, param_shape):
    """reference dion/muon.py:605-610"""
    fan_out, fan_in = param_shape[-2:]
    return lr * math.sqrt(fan_out / fan_in)


def adjust_lr_keller_muon(lr, param_shape):
    """reference dion/muon.py:612-617"""
    fan_out, fan_in = param_shape[-2:]
    return lr * max(1, fan_out / fan_in) ** 0.5


_ADJUST = {
    "spectral_norm": adjust_lr_spectral_norm,
    "rms_norm": adjust_lr_rms_norm,
    "keller_muon": adjust_lr_keller_muon,
}
_ADJUST_CODE = {None: 0, "spectral_norm": 1, "rms_norm": 2, "keller_muon": 3}   # of _host.muon_group


class Muon(_lib.HookedOptimizer):
    """
    Muon for a single MI355X.

    Args (identical to the reference, dion/muon.py:55-69):
        params: parameters or param-group dicts. A group may override any default and
            selects its update rule with `algorithm` in {"muon", "lion", "adamw"}.
        distributed_mesh: must be None (one GPU).
        lr, mu, betas, weight_decay, epsilon, nesterov, adjust_lr, flatten: as in the reference.
        use_triton: accepted and ignored; the HIP kernels are always used.
        newton_schulz_func: optional custom `func(input: Tensor, epsilon) -> Tensor`; when
            given, the momentum pass and the weight update run as separate kernels around that function.
    """

    def __init__(
        self,
        params: ParamsT,
        distributed_mesh=None,
        lr: float = 0.01,
        mu: float = 0.95,
        betas: Tuple[float, float] = (0.9, 0.95),
        weight_decay: float = 0.01,
        epsilon: float = 1e-8,
        nesterov: bool = False,
        adjust_lr: Optional[str] = "spectral_norm",
        flatten: bool = False,
        use_triton: bool = False,
        newton_schulz_func: Optional[Callable] = None,
    ):
        if lr < 0.0:
            raise ValueError(f"Invalid learning rate: {lr}")
        if mu < 0.0:
            raise ValueError(f"Invalid momentum factor (mu): {mu}")
        if len(betas) != 2 or betas[0] < 0.0 or betas[1] < 0.0:
            raise ValueError(f"Invalid betas: {betas}")
        if adjust_lr not in ("spectral_norm", "rms_norm", "keller_muon", None):
            raise ValueError(
                f"Invalid adjust_lr value: {adjust_lr}. Must be 'spectral_norm', 'rms_norm', 'keller_muon', or None."
            )
        defaults = dict(
            lr=lr, mu=mu, beta1=betas[0], beta2=betas[1], weight_decay=weight_decay, algorithm="muon",
            step=0, epsilon=epsilon, nesterov=nesterov, flatten=flatten, adjust_lr=adjust_lr,
        )
        super().__init__(params, defaults)

        if distributed_mesh is not None:
            raise NotImplementedError(
                "dion_amd.Muon runs on one GPU: distributed_mesh must be None "
                f"(got {type(distributed_mesh).__name__})."
            )
        self._device_rank = 0
        self._world_size = 1
        self._process_group = None
        self._distributed_mesh = None

        if newton_schulz_func is not None:
            if not callable(newton_schulz_func):
                raise TypeError(f"newton_schulz_func must be a callable function, got {type(newton_schulz_func)}")
            self._newton_schulz_func = newton_schulz_func
            self._fused = False
        else:
            self._newton_schulz_func = zeropower_via_newtonschulz5
            self._fused = True
        self._workspace = _lib.Workspace()
        self._coeffs = flat_coeffs(NS_SCHEDULE_COEFFS)

    def step(self, closure=None):
        loss = None
        if closure is not None:
            with torch.enable_grad():
                loss = closure()

        muon_groups, lion_groups, adamw_groups = [], [], []
        for group in self.param_groups:
            group["step"] += 1
            algo = group["algorithm"]
            if algo == "muon":
                muon_groups.append(group)
            elif algo == "lion":
                lion_groups.append(group)
            elif algo == "adamw":
                adamw_groups.append(group)
            else:
                raise ValueError(f"Unknown algorithm: {algo}")

        for group in muon_groups:
            self._muon_group_step(group)
        element_groups_step(self, lion_groups, False)
        element_groups_step(self, adamw_groups, True)
        return loss

    # ------------------------------------------------------------------ state
    def _get_or_initialize_state(self, param: Tensor, algo: str) -> dict:
        state = self.state[param]
        if not state:
            state["momentum"] = torch.zeros_like(param)
            if algo == "adamw":
                state["variance"] = torch.zeros_like(param)
        return state

    def _new_state(self, param: Tensor, group: dict):
        with torch.no_grad():
            self._get_or_initialize_state(param, group["algorithm"])

    # ------------------------------------------------------------------ muon
    def _muon_group_step(self, group: dict):
        assert all(p.ndim >= 2 for p in group["params"]), "Muon optimizer only supports matrix parameters."
        adjust = group["adjust_lr"]
        if adjust not in _ADJUST_CODE:
            raise ValueError(f"Unknown adjust_lr value: {adjust}")
        if not self._fused:
            with torch.no_grad():
                self._muon_group_unfused(group)
            return
        # Buckets of one (dtype, grad dtype, device) go to the library together: their Newton-Schulz
        # products are grouped launches, so small buckets share the GPU instead of queueing
        # (the reference overlaps them as async tasks, dion/muon.py:185-270).
        args = (group["params"], self.state, float(group["lr"]), float(group["mu"]), float(group["weight_decay"]),
                float(group["epsilon"]), group["nesterov"], _ADJUST_CODE[adjust], group["flatten"],
                ctypes.addressof(self._coeffs), len(NS_SCHEDULE_COEFFS), self._workspace)
        host = _lib.host()
        missing = host.muon_group(*args)
        if missing is not None:
            for p in missing:
                self._new_state(p, group)
            _lib.require_states(host.muon_group(*args), "Muon.step")

    def _muon_group_unfused(self, group: dict):
        # hyper-parameters as 0-dim fp32 tensors, evaluated like reference dion/muon.py:205-208
        lr = torch.tensor(group["lr"])
        mu = torch.tensor(group["mu"])
        weight_decay = torch.tensor(group["weight_decay"])
        epsilon = torch.tensor(group["epsilon"])
        adjust = group["adjust_lr"]
        buckets = defaultdict(list)
        for p in group["params"]:
            if p.grad is not None:
                buckets[(p.shape, p.dtype, p.grad.dtype, p.device)].append(p)
        for (shape, *_), plist in buckets.items():
            states = [self._get_or_initialize_state(p, "muon") for p in plist]
            adjusted_lr = lr if adjust is None else _ADJUST[adjust](lr, shape)
            self._muon_bucket_unfused(plist, states, lr, adjusted_lr, mu, weight_decay, epsilon, group)

    def _muon_bucket_unfused(self, plist, states, lr, adjusted_lr, mu, weight_decay, epsilon, group):
        """Custom `newton_schulz_func` (the reference's plug-in hook, dion/muon.py:48-49, 122-131): the momentum pass
        and the weight update run as the library's stand-alone stages (`dion_amd_muon_pre` / `dion_amd_muon_post`,
        reference dion/muon.py:536-552 and 568-573) around the user's function, which is called per parameter with
        the reference's flatten rules (585-593) and a 0-dim fp32 `epsilon` tensor."""
        lib = _lib.load()
        p0 = plist[0]
        _lib.require_gpu(p0, "Muon.step")
        device = p0.device
        cols = p0.size(-1)
        rows = p0.numel() // cols
        Ms = [st["momentum"] for st in states]
        for t in (*plist, *Ms):
            if not t.is_contiguous():
                raise _lib.DionAmdError("Muon.step: parameters and momentum buffers must be contiguous")
        X = [p.view(rows, cols) for p in plist]
        G = [(p.grad if p.grad.is_contiguous() else p.grad.contiguous()).view(rows, cols) for p in plist]
        M = [m.view(rows, cols) for m in Ms]
        Us = [torch.empty((rows, cols), dtype=torch.bfloat16, device=device) for _ in plist]
        with torch.cuda.device(device):
            rc = lib.dion_amd_muon_pre(
                _lib.ptr_array(G), _lib.ptr_array(M), _lib.ptr_array(Us), len(plist), rows, cols,
                _lib.dtype_code(G[0].dtype), _lib.dtype_code(M[0].dtype), mu.item(), int(bool(group["nesterov"])),
                _lib.stream_ptr(device))
        _lib.check(rc, "dion_amd_muon_pre")
        O = []
        for p, u in zip(plist, Us):
            u = u.view(p.shape)
            if group["flatten"] and u.ndim >= 3:
                v = u.flatten(start_dim=1)
            elif u.ndim >= 4:
                v = u.flatten(end_dim=-3)
            else:
                v = u
            o = self._newton_schulz_func(v, epsilon=epsilon).reshape(p.shape)
            # the update is scaled and subtracted in the dtype the function returned (reference dion/muon.py:569-573):
            # bf16 and fp32 go to the library as they are, anything else as fp32
            if o.dtype not in (torch.bfloat16, torch.float32):
                o = o.to(dtype=torch.float32)
            o = o.reshape(rows, cols).contiguous()
            if o.data_ptr() % 16:   # (a contiguous view at an odd offset: the kernels move 16-byte segments)
                o = o.clone()
            O.append(o)
        o_dtypes = {o.dtype for o in O}
        if len(o_dtypes) > 1:
            O = [o.to(dtype=torch.float32) for o in O]
        alr = adjusted_lr.item() if isinstance(adjusted_lr, Tensor) else float(torch.tensor(adjusted_lr).item())
        with torch.cuda.device(device):
            rc = lib.dion_amd_muon_post(
                _lib.ptr_array(X), _lib.ptr_array(O), len(plist), rows, cols, _lib.dtype_code(X[0].dtype),
                _lib.dtype_code(O[0].dtype), (1 - lr * weight_decay).item(), alr, _lib.stream_ptr(device))
        _lib.check(rc, "dion_amd_muon_post")

    # ------------------------------------------------------------------ element-wise groups
