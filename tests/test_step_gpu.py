"""Generation on sisa_step / sisa_cache_fill (csrc/step.hip) against the module path and the dense fp64 model, and the
calls that must keep the module path."""
import ctypes
import os
import subprocess

import pytest
import torch

from model_utils import rel_err, tiny_model, token_ids
from oracle import model64 as M64

DEV = "cuda:0"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _decode(model, ids, prompt, capacity=None):
    from sisa_amd import SISACache
    cache = SISACache(capacity)
    with torch.no_grad():
        parts = [model(ids[:, :prompt], cache=cache).logits]
        parts += [model(ids[:, t:t + 1], cache=cache).logits for t in range(prompt, ids.shape[1])]
    return torch.cat(parts, 1).float(), cache


def _count(monkeypatch):
    from sisa_amd.kernels import _lib
    calls, real = {}, _lib.call

    def call(name, args, t):
        calls[name] = calls.get(name, 0) + 1
        return real(name, args, t)
    monkeypatch.setattr(_lib, "call", call)
    return calls


def _watched(model):
    """The same model with a hook that does nothing on one projection: the modules are called one by one."""
    return [blk.attn.W_Q.register_forward_hook(lambda *a: None) for blk in model.layers]


# prompts of 1 to 1,105 rows (tiles of 128, remainders of 1 to 127); rows: one, two and four column groups of the products
# and their edges; widths below and above eight 32-element steps, a head count that is not a multiple of the 16-row groups'
# 16; hidden widths that are no multiple of 32, 16, 8 or 2; prompts of one position, of a chunk's edge and past it
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,d_ff,prompt,steps", [(1, 2, 256, 1, 3), (4, 12, 2744, 64, 3), (16, 3, 40, 5, 2),
                                                   (17, 5, 329, 65, 2), (33, 2, 250, 7, 2), (64, 16, 1000, 3, 2)])
def test_step_matches_modules(B, H, d_ff, prompt, steps, dtype, monkeypatch):
    model = tiny_model(seed=B, theta_scale=0.25, attn_impl="auto", n_head=H, d_model=64 * H, d_ff=d_ff).to(DEV).to(
        dtype).eval()
    ids = token_ids(B, prompt + steps, seed=H).to(DEV)
    ref = M64.logits64(model, M64.params64(model, requires_grad=False), ids)
    calls = _count(monkeypatch)
    got, cache = _decode(model, ids, prompt, None if B % 2 else prompt + steps)
    assert calls["sisa_step"] == 2 * steps and calls["sisa_prefill"] == 2
    assert "sisa_decode_attn" not in calls and "sisa_attn_fwd" not in calls
    monkeypatch.setattr("sisa_amd.kernels.step.PREFILL_ROWS", 0)       # the long prompts' route: fused, launch by launch
    calls.clear()
    long, held = _decode(model, ids, prompt)
    assert calls["sisa_step"] == 2 * steps and calls["sisa_cache_fill"] == 2 and "sisa_prefill" not in calls
    hooks = _watched(model)
    calls.clear()
    want, kept = _decode(model, ids, prompt)
    assert not {"sisa_step", "sisa_cache_fill", "sisa_prefill"} & set(calls) and calls["sisa_decode_attn"] == 2 * steps
    for h in hooks:
        h.remove()
    # both round the same quantities to the compute dtype: neither is further from fp64 than the other by more than
    # the spread of such errors over a few hundred logits
    assert rel_err(got, ref) <= 1.25 * rel_err(want, ref) + 1e-3
    assert rel_err(long, ref) <= 1.25 * rel_err(want, ref) + 1e-3
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for a, b in ((c.get(layer), kept.get(layer)) for layer in range(2) for c in (cache, held)):
        assert a.length == b.length == prompt + steps
        error = {n: rel_err(getattr(a, n), getattr(b, n)) for n in ("k", "v", "b", "g", "fgate", "phi")}
        # two roundings to the compute dtype each side; a phase that is off by d radians turns b~ by d more, and the
        # phases, sums of rounded rates, are largest at the last position
        turn = 2 * eps * float(b.phi.pow(2).mean().sqrt())
        bound = dict(k=4 * eps, v=4 * eps, b=4 * eps + turn, g=2 * eps, fgate=2 * eps, phi=2 * eps)
        assert all(error[n] <= bound[n] for n in error), (error, bound)


@pytest.mark.gpu
def test_calls_that_keep_the_module_path(monkeypatch):
    """What a step does not stand for: gradients, autocast, fp32, several new positions, more rows than it takes, a
    forced implementation other than the fused one, a subclass, a patched forward, a cache of another dtype."""
    from sisa_amd import SISACache
    calls = _count(monkeypatch)

    def steps_of(model, ids, n=1, **kw):
        cache = SISACache()
        calls.clear()
        with torch.no_grad():
            model(ids[:, :8], cache=cache)
        with kw.get("ctx", torch.no_grad)():
            model(ids[:, 8:8 + n], cache=cache)
        return calls.get("sisa_step", 0)

    ids = token_ids(3, 12, seed=1).to(DEV)
    model = tiny_model(seed=1, attn_impl="auto").to(DEV).to(torch.bfloat16).eval()
    assert steps_of(model, ids) == 2
    assert steps_of(model, ids, n=2) == 0
    assert steps_of(model, ids, ctx=torch.enable_grad) == 0
    assert steps_of(model, ids, ctx=lambda: torch.autocast("cuda", dtype=torch.bfloat16)) == 0
    assert steps_of(model, token_ids(65, 12, seed=1).to(DEV)) == 0
    model.set_attn_impl("hip")
    assert steps_of(model, ids) == 0
    model.set_attn_impl("auto")
    model.layers[0].ffn.w_down.forward = model.layers[0].ffn.w_down.forward
    assert steps_of(model, ids) == 1
    assert steps_of(tiny_model(seed=1, attn_impl="auto").to(DEV).eval(), ids) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,N", [(torch.bfloat16, 54560), (torch.bfloat16, 54561), (torch.float32, 27617)])
def test_decode_at_the_streaming_line(dtype, N):
    """Caches just below and above 256 MiB (15 heads: 4,920 or 9,720 bytes a position) give each row what its head alone,
    far below it, gives: the loads' cache policy is all that changes, in 16 bits, and nothing in fp32."""
    from sisa_amd.kernels.decode import sisa_decode_hip
    gen = torch.Generator(device=DEV).manual_seed(3)

    def draw(*shape, dt=dtype):
        return torch.randn(shape, generator=gen, device=DEV).to(dt)
    H = 15
    k, v, b = draw(1, H, N, 64), draw(1, H, N, 64), draw(1, H, N, 32)
    q, c, lam = draw(1, H, 1, 64), draw(1, H, 1, 32), draw(H, dt=torch.float32).abs()
    g, f = (-0.01 * draw(1, H, N, dt=torch.float32).abs().cumsum(2) for _ in range(2))
    out = sisa_decode_hip(q, k, v, c, b, g[:, :, -1:], g, lam, f[:, :, -1:], f, N - 1)
    for h in (0, 7, 14):
        s = slice(h, h + 1)
        one = sisa_decode_hip(q[:, s], k[:, s], v[:, s], c[:, s], b[:, s], g[:, s, -1:], g[:, s], lam[s], f[:, s, -1:],
                              f[:, s], N - 1)
        assert torch.equal(out[:, s], one)


@pytest.mark.gpu
def test_step_refuses_what_it_cannot_run():
    from sisa_amd.kernels import _lib
    x = torch.zeros(1, 64, device=DEV, dtype=torch.bfloat16)
    for bad in (dict(B=0), dict(L=0), dict(B=100, L=100), dict(dtype=_lib.F32), dict(H=65), {}):
        args = _lib.PrefillArgs(**{**dict(B=1, L=4, H=1, FF=64, dtype=_lib.BF16, act_ld=64), **bad})
        with pytest.raises(RuntimeError):
            _lib.call("sisa_prefill", args, x)
    for bad in (dict(B=0), dict(B=65), dict(D=63), dict(D=64 * 17, H=17), dict(pos=0), dict(dtype=_lib.F32), {}):
        args = _lib.StepArgs(**{**dict(B=1, H=1, D=64, FF=64, dtype=_lib.BF16, pos=1), **bad})
        with pytest.raises(RuntimeError):
            _lib.call("sisa_step", args, x)


def test_step_struct_layout_matches_c(tmp_path):
    from sisa_amd.kernels import _lib
    pairs = {"StepArgs": "sisa_step_args", "CacheFillArgs": "sisa_cache_fill_args",
             "PrefillArgs": "sisa_prefill_args"}
    lines, expect = ["#include <stdio.h>", "#include <stddef.h>", '#include "sisa_hip_step.h"', "int main(void) {"], []
    for py, c in pairs.items():
        cls = getattr(_lib, py)
        lines.append(f'printf("%zu\\n", sizeof({c}));')
        expect.append(ctypes.sizeof(cls))
        for name, _ in cls._fields_:
            lines.append(f'printf("%zu\\n", offsetof({c}, {name}));')
            expect.append(getattr(cls, name).offset)
    lines += ["return 0;", "}"]
    (tmp_path / "layout.c").write_text("\n".join(lines))
    exe = tmp_path / "layout"
    subprocess.run(["gcc", "-std=c99", "-I", os.path.join(ROOT, "include"), str(tmp_path / "layout.c"), "-o", str(exe)],
                   check=True)
    got = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()
    assert [int(v) for v in got] == expect


@pytest.mark.gpu
def test_fp32_generation_with_the_fused_implementation_requested():
    """Cached fp32 calls under attn_impl="hip_fused" run the unfused kernels, as a call without a cache cannot."""
    ids = token_ids(2, 9, seed=4).to(DEV)
    model = tiny_model(seed=4, theta_scale=0.25, attn_impl="hip_fused").to(DEV).eval()
    got, _ = _decode(model, ids, 6)
    model.set_attn_impl("hip")
    want, _ = _decode(model, ids, 6)
    assert torch.equal(got, want)


def test_failed_cache_fill_leaves_no_entry(monkeypatch):
    """A prefill on the fused route whose last launch fails leaves the layer's entry empty, to be filled again."""
    from types import SimpleNamespace

    from sisa_amd import SISACache
    from sisa_amd.kernels import _lib, step
    B, L, H = 1, 3, 2
    proj = torch.zeros(B, L, step.P.fused_layout(H)["NPAD"], dtype=torch.bfloat16)
    rows, gates = torch.zeros(B, L, H, 32, dtype=torch.bfloat16), torch.zeros(B, H, L)
    prepped = step.P.Prepped(rows, rows, gates, gates, gates, gates, torch.zeros(B * H, 1, 18))
    monkeypatch.setattr(step.P, "prep_forward", lambda *a: prepped)
    monkeypatch.setattr(step.A, "attn_forward", lambda *a: SimpleNamespace(o=torch.zeros(B, H, L, 64)))

    def fail(*a):
        raise RuntimeError("no launch")
    monkeypatch.setattr(_lib, "call", fail)
    cache = SISACache()
    with pytest.raises(RuntimeError, match="no launch"):
        step.prefill(proj, torch.zeros(B, L, H), torch.ones(H), H, cache, 0)
    assert len(cache) == 0 and cache.get(0) is None


def test_prefill_takes_what_it_is_faster_at_and_can_reach():
    """Wide models hand over to the library's GEMMs at fewer tokens. The products read their operands by 32-bit offsets:
    activations or weights of 2 GiB keep the fused route, and the entry point refuses them."""
    from sisa_amd.kernels import _lib, step
    for width, most in ((64, 8192), (1024, 8192), (1088, 3855), (1536, 2730), (2048, 2048), (4096, 1024)):
        assert step.prefill_takes(1, width, 2736) and step.prefill_takes(most, width, 2736)
        assert not step.prefill_takes(most + 1, width, 2736)
    assert step.prefill_takes(8192, 64, 130_000)
    assert not step.prefill_takes(8192, 64, 131_072) and not step.prefill_takes(1, 4096, 262_144)
    lib = _lib.load()
    for L, H, ff in ((8192, 1, 131_072), (1, 64, 262_144)):
        pointers = {n: 256 for n, t in _lib.PrefillArgs._fields_ if t is ctypes.c_void_p and n != "res"}
        args = _lib.PrefillArgs(B=1, L=L, H=H, FF=ff, dtype=_lib.BF16, act_ld=ff, **pointers)
        assert lib.sisa_prefill(ctypes.byref(args), None) != 0
        assert "2 GiB" in lib.sisa_last_error().decode()


@pytest.mark.gpu
def test_calls_refused_by_size_or_type_cost_nothing_more(monkeypatch):
    """Steps that the kernels do not take for their size or type keep the module path before the modules are looked at."""
    from sisa_amd import SISACache
    from sisa_amd.kernels import step
    ids = token_ids(65, 12, seed=1).to(DEV)
    for rows, n, dtype in ((65, 1, torch.bfloat16), (3, 2, torch.bfloat16), (3, 1, torch.float32)):
        model, cache = tiny_model(seed=1, attn_impl="auto").to(DEV).to(dtype).eval(), SISACache()
        with torch.no_grad():
            model(ids[:rows, :8], cache=cache)
            looked = []
            monkeypatch.setattr(step, "plain_linears", lambda *a: looked.append(a))
            model(ids[:rows, 8:8 + n], cache=cache)
            monkeypatch.undo()
        assert not looked, (rows, n, dtype)


def _unregister(module):
    """Its weight as a plain attribute, as wrappers that shard or flatten parameters leave it."""
    w = module._parameters.pop("weight")
    module.__dict__["weight"] = w.detach()
    return w


def test_step_weights_of_unregistered_parameters():
    from sisa_amd.kernels import step
    model = tiny_model(seed=1).to(torch.bfloat16)
    blk, x = model.layers[0], torch.zeros(1, 1, 128, dtype=torch.bfloat16)

    def parts():
        return (step.plain_linears(blk.attn._modules, blk.ffn._modules), blk.attn_norm.weight, blk.ffn_norm.weight, 2, x)
    assert parts()[0] is not None
    _unregister(blk.ffn.w_down)
    assert step.step_weights(*parts()) is None
    _unregister(blk.attn.alpha_proj)
    assert step.step_weights(*parts()) is None


@pytest.mark.gpu
def test_generation_with_unregistered_parameters():
    ids = token_ids(2, 5, seed=6).to(DEV)
    for of in (lambda b: b.ffn.w_gate, lambda b: b.attn_norm, lambda b: b.attn.W_Q):
        model = tiny_model(seed=6, theta_scale=0.25, attn_impl="auto").to(DEV).to(torch.bfloat16).eval()
        want, _ = _decode(model, ids, 3)
        _unregister(of(model.layers[0]))
        got, _ = _decode(model, ids, 3)
        assert rel_err(got, want) <= 2.0 ** -5        # another route in 16 bits, not other values


# more heads than the 16 and 32 outputs of the norm kernels' narrower forms, head counts that are no multiple of the four
# outputs a lane stores at once, the widest model; prompts at the line from which wide models take the library's products
@pytest.mark.gpu
@pytest.mark.parametrize("H,d_ff,B,L", [(17, 200, 2, 70), (33, 329, 3, 5), (64, 264, 1, 130), (24, 136, 1, 2730)])
def test_prompts_of_wide_models(H, d_ff, B, L, monkeypatch):
    model = tiny_model(seed=H, theta_scale=0.25, attn_impl="auto", n_head=H, d_model=64 * H, d_ff=d_ff).to(DEV).to(
        torch.bfloat16).eval()
    ids = token_ids(B, L, seed=H).to(DEV)
    calls = _count(monkeypatch)
    got, cache = _decode(model, ids, L)
    assert calls["sisa_prefill"] == 2
    hooks = _watched(model)
    calls.clear()
    want, kept = _decode(model, ids, L)
    assert "sisa_prefill" not in calls
    for h in hooks:
        h.remove()
    ref = M64.logits64(model, M64.params64(model, requires_grad=False), ids)
    # both round the same quantities to bf16: neither is further from fp64 than the other by more than the spread of such
    # errors
    assert rel_err(got, ref) <= 1.25 * rel_err(want, ref) + 1e-3
    for layer in range(2):
        a, b = cache.get(layer), kept.get(layer)
        assert a.length == b.length == L
        # the first layer's entries are projections of the same rows: two roundings to bf16 each side
        assert layer or all(rel_err(getattr(a, n), getattr(b, n)) <= 4 * 2.0 ** -8 for n in ("k", "v", "g", "fgate", "phi"))
