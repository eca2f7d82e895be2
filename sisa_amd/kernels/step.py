"""Generation on the HIP kernels of csrc/step.hip and csrc/prefill.hip: one new token of every row through a whole
decoder layer with a filled cache (``sisa_step``, seven launches behind one C call), a prompt through a layer with an empty
one (``sisa_prefill``, thirteen), and the filling of a layer's cache after a prefill on the fused route
(``sisa_cache_fill``). The module path these stand in for is src/sisa/modeling.py:171-199, 224-238,
288-291; there a layer's step is about seventy torch kernels, whose launches cost four times what they compute.

Both write into the cache's slabs in place and are for inference: the callers check that no gradient is wanted and
that nothing observes the modules they pass by (:func:`unobserved`, :func:`step_weights`).
"""
from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import Tensor, nn
from torch.nn.modules import module as _nn_module

from ..config import HIP_D_HEAD, HIP_D_STATE
from . import _lib
from . import attention as A
from . import fused_prep as P

__all__ = ["unobserved", "plain", "plain_linears", "rows_ok", "whole", "prefill_takes", "step_weights",
           "layer_step", "layer_prefill", "prefill", "MAX_ROWS", "MAX_WIDTH", "PREFILL_ROWS", "PREFILL_WORK"]

MAX_ROWS, MAX_WIDTH = 64, 1024          # SISA_STEP_MAX_ROWS, SISA_STEP_MAX_D
#: Prompts of at most this many tokens (all rows together) take ``sisa_prefill``, and at most PREFILL_WORK / width of them
#: in a model wider than 1,024: as far as it was measured no slower than the launch-by-launch route, whose library GEMMs
#: gain on it with size. Two layers of hidden width 2.7 D, us, native against launch by launch: width 768 318 and 990 for
#: 1,024 tokens, 664 and 1,015 for 8 x 1,024; 1,024 976 and 1,095; 1,536 647 and 982 for 2,048 tokens, 1,711 and 1,625 for
#: 8,192; 2,048 1,042 and 1,072, 2,865 and 2,477; 4,096 1,821 and 1,895 for 1,024, 4,017 and 3,656 for 3,072, 10,307 and
#: 8,009 for 8,192.
PREFILL_ROWS, PREFILL_WORK = 8192, 1 << 22


def prefill_takes(rows: int, width: int, d_ff: int) -> bool:
    """Whether a prompt is for ``sisa_prefill``: small enough (above), and its activations and weights, which the kernels
    read by 32-bit offsets, each ending below 2 GiB."""
    return (rows <= PREFILL_ROWS and (width <= 1024 or rows * width <= PREFILL_WORK)
            and max(rows, width) * (-(-d_ff // 64) * 64) * 2 < 1 << 31)


def unobserved(x: Tensor) -> bool:
    """Whether nothing follows the torch operations on ``x``: a plain tensor, no gradient or forward-mode level, no
    compile trace, function transform, dispatch or function mode, and no global module hooks."""
    return (type(x) is Tensor and not torch.is_grad_enabled() and not torch.compiler.is_compiling()
            and torch.autograd.forward_ad._current_level < 0
            and torch._C._functorch.peek_interpreter_stack() is None
            and not torch._C._len_torch_dispatch_stack() and not torch._C._len_torch_function_stack()
            and not _nn_module._global_forward_hooks and not _nn_module._global_forward_pre_hooks)


def plain(module: nn.Module, kind: type) -> bool:
    """A module of exactly this class whose call is its class's ``forward``: no hooks, no patched method."""
    return (type(module) is kind and not module._forward_hooks and not module._forward_pre_hooks
            and "forward" not in module.__dict__)


_ATTN_LINEARS = ("W_Q", "W_K", "W_V", "W_B", "W_C", "theta_proj", "alpha_proj", "forget_proj", "W_O")
_FFN_LINEARS = ("w_gate", "w_up", "w_down")


def plain_linears(attn: dict, ffn: dict) -> list[dict] | None:
    """The parameter dicts of a block's twelve linear modules (attention in the order of ``sisa_step_args`` with W_O
    last, then gate, up, down), or None unless every one is a :func:`plain` ``nn.Linear``."""
    out = []
    for mods, names in ((attn, _ATTN_LINEARS), (ffn, _FFN_LINEARS)):
        for name in names:
            m = mods.get(name)
            if type(m) is not nn.Linear or m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__:
                return None
            out.append(m._parameters)
    return out


def whole(x: Tensor | None) -> bool:
    """``x`` is contiguous and 16-byte aligned (or None)."""
    return x is None or (x.is_contiguous() and x.data_ptr() % 16 == 0)


def rows_ok(x: Tensor) -> bool:
    """``x`` (B, 1, D) has rows that 16-byte loads can read."""
    sb, _, sd = x.stride()
    return sd == 1 and sb % 8 == 0 and x.data_ptr() % 16 == 0


def step_weights(linears: list[dict], attn_norm, ffn_norm, H: int, x: Tensor) -> tuple[list[int], int] | None:
    """Addresses of the parameters in the order of ``sisa_step_args`` (attn_norm .. w_down) and the FFN's width, or
    None unless each is a plain contiguous parameter of the block's shape in ``x``'s dtype on its device, 16-byte
    aligned where the kernels load it in vectors, with biases on the two gates only."""
    D, s, dtype, device = x.shape[-1], HIP_D_STATE, x.dtype, x.get_device()
    q, k, v, b, c, theta, alpha, forget, o, gate, up, down = (p.get("weight") for p in linears)
    biases = [p.get("bias") for p in linears]
    if gate is None or any(t is not None for i, t in enumerate(biases) if i not in (6, 7)):
        return None
    ff = gate.shape[0]
    out = []
    for p, shape in ((attn_norm, (D,)), (q, (D, D)), (k, (D, D)), (v, (D, D)), (b, (H * s, D)), (c, (H * s, D)),
                     (theta, (H * s // 2, D)), (alpha, (H, D)), (biases[6], (H,)), (forget, (H, D)), (biases[7], (H,)),
                     (o, (D, D)), (ffn_norm, (D,)), (gate, (ff, D)), (up, (ff, D)), (down, (D, ff))):
        if type(p) is not nn.Parameter or p.dtype is not dtype or p.shape != shape or p.get_device() != device \
                or not p.is_contiguous():
            return None
        address = p.data_ptr()
        if address % 16 and shape != (H,):
            return None
        out.append(address)
    return out, ff


def layer_step(x: Tensor, res: Tensor | None, weights: list[int], d_ff: int, lambda_raw: Tensor,
               eps: tuple[float, float], slab, phi: Tensor) -> tuple[Tensor, Tensor, Tensor]:
    """The new position of ``x`` ``(B, 1, D)`` (plus ``res``, added first) through a layer; ``weights`` in the order of
    ``sisa_step_args`` (attn_norm .. w_down). Writes the position into ``slab`` (room for it is the caller's care) and
    returns ``(h, ffn, phi)``: the residual stream after the attention, the FFN output still to be added to it, and
    the phase at the new position."""
    B, _, D = x.shape
    H, pos = D // HIP_D_HEAD, slab.filled
    h, ffn = torch.empty((2, B, 1, D), device=x.device, dtype=x.dtype).unbind(0)
    phi_out = torch.empty((B, H, HIP_D_STATE // 2), device=x.device, dtype=torch.float32)
    lib = _lib.load()
    ws = torch.empty((lib.sisa_step_workspace_bytes(B, H, D, d_ff, pos + 1),), device=x.device, dtype=torch.uint8)
    buf = slab.buffers
    args = _lib.StepArgs(B, H, D, d_ff, _lib.dtype_code(x.dtype), pos, *eps, x.data_ptr(), x.stride(0),
                         None if res is None else res.data_ptr(), *weights, lambda_raw.data_ptr(),
                         *(_lib.view(buf[n]) for n in ("k", "v", "b", "g", "fgate")), phi.data_ptr(),
                         phi_out.data_ptr(), h.data_ptr(), ffn.data_ptr(), ws.data_ptr())
    _lib.call("sisa_step", args, x)
    return h, ffn, phi_out


def _fill(cache, layer_idx: int, name: str, args, x: Tensor) -> None:
    """The call that fills a layer's new cache entry; if it fails there is no entry again, not one of no positions."""
    try:
        _lib.call(name, args, x)
    except Exception:
        cache._slabs.pop(layer_idx, None)
        raise


def layer_prefill(x: Tensor, res: Tensor | None, weights: list[int], d_ff: int, lambda_raw: Tensor, w_down: Tensor,
                  eps: tuple[float, float], cache, layer_idx: int, checked: bool) -> tuple[Tensor, Tensor]:
    """A prompt ``x`` ``(B, L, D)`` (contiguous; plus ``res``, added first) through a layer whose cache entry is empty,
    filling it; ``weights`` as for :func:`layer_step`. Returns ``(h, f)``: the residual stream after the attention and the
    FFN output still to be added to it. ``checked``: assert on the device that ``g`` does not rise."""
    B, L, D = x.shape
    H, dev = D // HIP_D_HEAD, x.device
    ld = -(-d_ff // 64) * 64
    h = torch.empty_like(x)
    f = torch.empty_like(x) if d_ff % 8 == 0 else None
    act = torch.empty((B, L, ld), device=dev, dtype=x.dtype)
    phi = torch.empty((B, H, HIP_D_STATE // 2), device=dev, dtype=torch.float32)
    ok = torch.empty((1,), device=dev, dtype=torch.bool) if checked and L > 1 else None
    ws = torch.empty((_lib.load().sisa_prefill_workspace_bytes(B, L, H),), device=dev, dtype=torch.uint8)
    like = x.new_empty((B, H, 0, HIP_D_HEAD))
    gates = torch.empty((B, H, 0), device=dev, dtype=torch.float32)
    slab = cache.room(layer_idx, L, dict(k=like, v=like, b=x.new_empty((B, H, 0, HIP_D_STATE)), g=gates, fgate=gates),
                      phi)
    buf = slab.buffers
    args = _lib.PrefillArgs(B, L, H, d_ff, _lib.dtype_code(x.dtype), *eps, A.MONOTONE_TOL, x.data_ptr(), _lib.ptr(res),
                            *weights, lambda_raw.data_ptr(),
                            *(_lib.view(buf[n]) for n in ("k", "v", "b", "g", "fgate")), phi.data_ptr(), h.data_ptr(),
                            act.data_ptr(), _lib.ptr(f), ld, _lib.ptr(ok), ws.data_ptr())
    _fill(cache, layer_idx, "sisa_prefill", args, x)
    if ok is not None:
        torch._assert_async(ok, "sisa_attention_hip: the cumulative log-decay g increases along the sequence")
    slab.filled = L
    return h, F.linear(act[..., :d_ff], w_down) if f is None else f


def prefill(proj: Tensor, z: Tensor, lam: Tensor, n_head: int, cache, layer_idx: int) -> Tensor:
    """The fused layer core on a prompt that also fills the layer's (empty) cache: ``proj`` (B, L, NPAD), ``z``
    (B, L, H) as :func:`sisa_amd.kernels.fused_prep.sisa_fused` takes them. The check of ``g`` is the unfused route's,
    which a prefill ran before. Returns y (B, L, H*64). Inference only."""
    B, L, _ = proj.shape
    lay = P.fused_layout(n_head)
    pp = P.prep_forward(proj, z, n_head)
    q, k, v = (P._heads(proj, lay[n], n_head) for n in ("Q", "K", "V"))
    c, b = pp.state_views()
    fw = A.attn_forward(q, k, v, c, b, pp.g, lam, pp.f)
    phi = torch.empty((B, n_head, HIP_D_STATE // 2), device=proj.device, dtype=torch.float32)
    slab = cache.room(layer_idx, L, dict(k=k, v=v, b=b, g=pp.g, fgate=pp.f), phi)
    buf = slab.buffers
    _fill(cache, layer_idx, "sisa_cache_fill", _lib.CacheFillArgs(
        B, n_head, L, _lib.dtype_code(proj.dtype), proj.data_ptr(), proj.stride(0), proj.stride(1), lay["K"], lay["V"],
        pp.br.data_ptr(), pp.g.data_ptr(), pp.f.data_ptr(), pp.totals.data_ptr(),
        *(_lib.view(buf[n]) for n in ("k", "v", "b", "g", "fgate")), phi.data_ptr()), proj)
    slab.filled = L
    return fw.o.transpose(1, 2).flatten(2)
