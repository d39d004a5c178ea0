"""LoRA side branches of the attention module's linear layers.

The reference patches the forward of every Linear a LoRA file names (longcat_video_dit.py:211-249):
``org_forward(x) + sum_i lora_up_i(lora_down_i(x)) * multiplier_i * alpha_scale_i``.  ``lora_up`` is either one
Linear or, for fused projections such as qkv, one Linear per equal slice of the output features, each fed its own
slice of the rank axis (lora_utils.py:12-21, 47-53).  Here the layer and the down projection go to hipBLASLt through the C ABI; the
up-projection of a single branch, its scaling and the sum are one pass over the layer's output (bsa_lora_up_add), or, where the caller
takes one rounding for the eager expression's, a part of the layer's product (bsa_linear_lora_bf16, bsa_linear_gated_bf16).  Several branches, whose scaled terms are summed before the
layer's output is added, take their up-projections from hipBLASLt too (the sliced one with row strides, in place) and one
elementwise pass, with the eager roundings.
"""
import ctypes as C
from typing import List, Optional, Sequence

import torch

from .. import _capi
from .attention import _bf16, _gemm_workspace, _on_device, _ptr, _stream, gated_residual, linear_bf16, linear_gated

MAX_BRANCHES = 4


class LoRABranch:
    """The tensors of one LoRAModule (lora_utils.py:23-66): ``lora_down.weight`` [n_sep * rank, in],
    ``lora_up`` weights (one [out, rank] matrix, or n_sep matrices [out / n_sep, rank]), the multiplier and
    ``alpha_scale = alpha / rank`` (a buffer the reference casts to the model dtype, longcat_video_dit.py:221)."""

    def __init__(self, lora_down: torch.Tensor, lora_up: Sequence[torch.Tensor], multiplier: float = 1.0,
                 alpha: Optional[float] = None):
        lora_up = list(lora_up) if isinstance(lora_up, (list, tuple)) else [lora_up]
        n = len(lora_up)
        assert n >= 1 and lora_down.shape[0] % n == 0
        self.rank = lora_down.shape[0] // n
        assert all(u.shape == lora_up[0].shape and u.shape[1] == self.rank for u in lora_up)
        self.lora_down = lora_down
        self.lora_up = lora_up
        self.multiplier = multiplier
        alpha = self.rank if alpha is None or alpha == 0 else alpha                 # lora_utils.py:56
        self.alpha_scale = float(alpha) / self.rank
        self.use_lora = True

    @property
    def out_features(self) -> int:
        return self.lora_up[0].shape[0] * len(self.lora_up)

    def to(self, device=None, dtype=None):
        self.lora_down = self.lora_down.to(device=device, dtype=dtype)
        self.lora_up = [u.to(device=device, dtype=dtype) for u in self.lora_up]
        return self


def _up_projection(lx: torch.Tensor, branch: LoRABranch, workspace: torch.Tensor) -> torch.Tensor:
    """lora_up(lx): one GEMM, or one per output slice writing its columns of the result in place."""
    n = len(branch.lora_up)
    if n == 1:
        return linear_bf16(lx, branch.lora_up[0], None, workspace=workspace)
    M, r = lx.shape[0], branch.rank
    per = branch.lora_up[0].shape[0]
    out = torch.empty(M, n * per, dtype=torch.bfloat16, device=lx.device)
    lib = _capi.load()
    with _on_device(lx):
        for i, w in enumerate(branch.lora_up):
            w = w.contiguous()
            _capi.check(lib.bsa_linear_bf16_ld(lx.data_ptr() + 2 * i * r, n * r, _ptr(w), r, None, None,
                                               out.data_ptr() + 2 * i * per, n * per, M, per, r,
                                               _ptr(workspace), workspace.numel(), _stream(lx)), "lora up projection")
    return out


def _one_pass(b: LoRABranch) -> bool:
    """What bsa_lora_up_add is built for, and faster at from 1 to 32 760 tokens, rank 16 to 128 and 64 to 12 288 columns (figures at the
    kernel); other branches, and sums over several, take the up-projection as a tensor."""
    per = b.lora_up[0].shape[0]
    return (b.rank % 16 == 0 and b.rank <= 128 and len(b.lora_up) <= 8 and per % 64 == 0
            and all(u.dtype == torch.bfloat16 and (not u.is_contiguous() or u.data_ptr() % 16 == 0) for u in b.lora_up))


def _with_one_branch(x, x2, weight, bias, b: LoRABranch, alpha: float, workspace, one_rounding, residual, gate) -> torch.Tensor:
    """The down projection, then the layer with its side branch, and with a gate residual + gate * that."""
    M, K, N = x2.shape[0], x2.shape[1], weight.shape[0]
    assert weight.shape[1] == K and b.out_features == N and b.lora_down.shape[1] == K
    if b.lora_down.dtype != torch.bfloat16:
        raise NotImplementedError("LoRA weights must be bf16 (the reference moves them to the model dtype)")
    x2 = x2.contiguous()
    lx = linear_bf16(x2, b.lora_down, None, workspace=workspace)                  # [M, n_sep * rank]
    w, bw = _bf16(weight), None if bias is None else _bf16(bias)
    ups = [u.contiguous() for u in b.lora_up]
    ptrs = (C.c_void_p * len(ups))(*[u.data_ptr() for u in ups])
    side = (_ptr(lx), lx.shape[1], ptrs, len(ups), b.rank, float(b.multiplier), alpha)
    if gate is not None:
        return linear_gated(x2, w, bw, residual, gate, workspace, side)
    if not one_rounding:
        out = linear_bf16(x, weight, bias, workspace=workspace)
        with _on_device(x):
            _capi.check(_capi.load().bsa_lora_up_add(_ptr(out), *side, _ptr(out), M, N, _stream(x)), "lora_up_add")
        return out
    out = torch.empty(*x.shape[:-1], N, dtype=torch.bfloat16, device=x.device)
    with _on_device(x):
        _capi.check(_capi.load().bsa_linear_lora_bf16(_ptr(x2), _ptr(w), _ptr(bw), *side, _ptr(out), M, N, K, _ptr(workspace),
                                                      workspace.numel(), _stream(x)), "linear with a LoRA branch")
    return out


@torch.no_grad()
def lora_linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor],
                loras: Optional[List[LoRABranch]] = None, workspace: Optional[torch.Tensor] = None,
                one_rounding: bool = False, residual: Optional[torch.Tensor] = None, gate: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The patched forward of longcat_video_dit.py:234-249 for a bf16 Linear, with the eager expression's roundings; one_rounding: a
    single branch may go into the layer's sum instead.  With a gate, residual + gate * that, as gated_residual."""
    active = [b for b in (loras or []) if b.use_lora]
    if gate is not None and not (one_rounding and len(active) == 1 and _one_pass(active[0])):
        return gated_residual(residual, gate, lora_linear(x, weight, bias, loras, workspace, one_rounding))
    if not active:
        return linear_bf16(x, weight, bias, workspace=workspace)                    # `org_output + 0`
    if len(active) > MAX_BRANCHES:
        raise NotImplementedError("at most %d LoRA branches per Linear are built" % MAX_BRANCHES)
    if not x.is_cuda:
        raise RuntimeError("the engine runs on the GPU only")
    if workspace is None:
        workspace = _gemm_workspace(x.device)
    N = weight.shape[0]
    x2 = x.reshape(-1, x.shape[-1])
    # alpha_scale lives in a bf16 buffer in the reference
    alphas = [float(torch.tensor(b.alpha_scale, dtype=torch.bfloat16)) for b in active]
    if len(active) == 1 and _one_pass(active[0]):
        return _with_one_branch(x, x2, weight, bias, active[0], alphas[0], workspace, one_rounding, residual, gate)
    org = linear_bf16(x, weight, bias, workspace=workspace)
    ups = []
    for b, a in zip(active, alphas):
        assert b.out_features == N and b.lora_down.shape[1] == x.shape[-1]
        if b.lora_down.dtype != torch.bfloat16:
            raise NotImplementedError("LoRA weights must be bf16 (the reference moves them to the model dtype)")
        lx = linear_bf16(x2, b.lora_down, None, workspace=workspace)              # [M, n_sep * rank]
        ups.append(_up_projection(lx, b, workspace))
    n = len(ups)
    up_ptrs = (C.c_void_p * n)(*[u.data_ptr() for u in ups])
    mult = (C.c_float * n)(*[float(b.multiplier) for b in active])
    alpha = (C.c_float * n)(*alphas)
    out2 = org.view(-1, N)
    with _on_device(x):
        _capi.check(_capi.load().bsa_lora_add(_ptr(out2), up_ptrs, mult, alpha, n, _ptr(out2), out2.numel(),
                                              _capi.BSA_BF16, _stream(x)), "lora_add")
    return org
