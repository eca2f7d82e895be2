"""The calls whose speed matters to a user of sisa_amd, as cases that a timing program can run and check.

A case is a dict of plain values; its ``"kind"`` names the entry point:

* ``fused``    -- ``sisa_fused``, the layer core between the projection GEMM and W_O: scoring (forward) or training
                  (forward and all gradients);
* ``attn``     -- ``sisa_attention(impl="hip")`` on prepared operands: forward, or forward and all gradients;
* ``lmce``     -- ``linear_cross_entropy``, the tied LM head's loss: evaluation, or loss with both gradients;
* ``norm``     -- ``rms_norm_forget_add_hip``: residual add, RMSNorm and forget-gate logits, forward and backward;
* ``block``    -- one ``SISABlock`` under bf16 autocast, forward and backward, every parameter's gradient;
* ``decode``   -- ``sisa_decode_hip``: one token's attention against a filled cache;
* ``generate`` -- a whole ``SISAForCausalLM`` with a cache: prefill, then one-token steps; logits of every step.

Head size 64 and state size 32 throughout (the only ones the kernels take); widths, depths and the vocabulary are
those of the presets in ``sisa_amd/config.py``; the value distributions are those of ``sisa_amd/workloads.py``.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from sisa_amd import SISABlock, SISACache, SISAConfig, SISAForCausalLM, sisa_attention
from sisa_amd.kernels.decode import sisa_decode_hip
from sisa_amd.kernels.fused_prep import sisa_fused
from sisa_amd.kernels.linear_ce import linear_cross_entropy
from sisa_amd.kernels.norm import rms_norm_forget_add_hip

DEVICE = "cuda"
D_HEAD, D_STATE = 64, 32
VOCAB = 50277
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}
PRESET_OF_WIDTH = {512: "sisa-50m", 768: "sisa-152m", 1024: "sisa-369m"}


# ------------------------------------------------------------------------------------------------ the cases
def listed() -> list[dict]:
    return [
        # the layer core of a training step at the benchmark's headline shape
        dict(name="fused_train_4x4096_h8", kind="fused", B=4, T=4096, H=8, dtype="bf16", forget=True, train=True,
             long_lived=False),
        # the same in fp16 at the length of a packed batch of short documents, not a multiple of any tile
        dict(name="fused_train_6x1001_h12_fp16", kind="fused", B=6, T=1001, H=12, dtype="fp16", forget=True,
             train=True, long_lived=False),
        # long-context training: one sequence, slow decay
        dict(name="fused_train_1x16384_h16", kind="fused", B=1, T=16384, H=16, dtype="bf16", forget=True, train=True,
             long_lived=True),
        # scoring one ragged document batch without gradients
        dict(name="fused_score_2x3001_h12", kind="fused", B=2, T=3001, H=12, dtype="bf16", forget=True, train=False,
             long_lived=False),
        # the accuracy path: a small fp32 attention with gradients, as a numerics study or a test of a model runs it
        dict(name="attn_train_1x256_h4_fp32", kind="attn", B=1, T=256, H=4, dtype="fp32", forget=True, train=True),
        # LM-head loss of a training step: 16,384 tokens, 768 wide
        dict(name="lmce_train_16384_d768", kind="lmce", N=16384, D=768, V=VOCAB, dtype="bf16", ignored=0.0,
             train=True),
        # LM-head loss of a fine-tuning step on one sequence, prompt tokens masked out of the loss
        dict(name="lmce_train_1023_d512", kind="lmce", N=1023, D=512, V=VOCAB, dtype="bf16", ignored=0.3, train=True),
        # held-out loss of the largest preset's head
        dict(name="lmce_eval_4094_d1024", kind="lmce", N=4094, D=1024, V=VOCAB, dtype="bf16", ignored=0.0,
             train=False),
        # the attention norm of the largest preset, forward and backward, in a model's fp32 residual stream
        dict(name="norm_train_5000_d1024_h16", kind="norm", N=5000, D=1024, H=16, dtype="bf16"),
        # one decoder block of the training step at the benchmark's model configuration
        dict(name="block_train_8x2048_d768", kind="block", B=8, T=2048, D=768),
        # one generated token's attention per layer after a long prompt, batch of 8
        dict(name="decode_8x16384_h12", kind="decode", B=8, H=12, T=16384, dtype="bf16"),
        # a chat turn: prompt and the first generated tokens of the 152M model in bf16
        dict(name="generate_4x200_plus6_d768", kind="generate", B=4, T=200, steps=6, D=768),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["fused", "fused", "fused", "attn", "attn", "lmce", "lmce", "norm", "block", "decode",
                       "generate"])
    if kind == "fused":
        H = rng.choice([4, 8, 12, 16])
        T = _log_int(rng, 33, 16384)
        room = min(131072 // T, 16 * 16384 ** 2 // (H * T * T))      # at most the long case's tokens and pairs
        B = _log_int(rng, 1, max(1, min(16, room)))
        return dict(kind=kind, B=B, T=T, H=H, dtype=rng.choice(["bf16", "bf16", "fp16"]), forget=rng.random() < 0.85,
                    train=rng.random() < 0.7, long_lived=rng.random() < 0.3)
    if kind == "attn":
        dtype = rng.choice(["bf16", "fp16", "fp32"])
        H = rng.choice([4, 8, 12])
        T = _log_int(rng, 17, 1024 if dtype == "fp32" else 6000)
        B = rng.randint(1, 2)
        return dict(kind=kind, B=B, T=T, H=H, dtype=dtype, forget=rng.random() < 0.75, train=rng.random() < 0.6)
    if kind == "lmce":
        train = rng.random() < 0.7           # fp16 for evaluation only: unscaled fp16 gradients underflow at 1 / (N V)
        return dict(kind=kind, N=_log_int(rng, 50, 12000), D=rng.choice([512, 768, 1024]),
                    V=rng.choice([VOCAB, VOCAB, 32000, 8191]), dtype="bf16" if train else rng.choice(["bf16", "fp16"]),
                    ignored=rng.choice([0.0, 0.3]), train=train)
    if kind == "norm":
        D = rng.choice([512, 768, 1024])
        return dict(kind=kind, N=_log_int(rng, 30, 16384), D=D, H=D // 64, dtype=rng.choice(["bf16", "bf16", "fp16"]))
    if kind == "block":
        D = rng.choice([512, 768, 1024])
        T = _log_int(rng, 65, 2048)
        return dict(kind=kind, B=rng.randint(1, max(1, min(8, 12288 // T))), T=T, D=D)
    if kind == "decode":
        return dict(kind=kind, B=rng.randint(1, 8), H=rng.choice([8, 12, 16]), T=_log_int(rng, 65, 12288),
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    return dict(kind=kind, B=rng.randint(1, 4), T=_log_int(rng, 17, 400), steps=rng.randint(2, 6),
                D=rng.choice([512, 768]))


# ------------------------------------------------------------------------------------------------ inputs
def _columns(H: int) -> dict:
    """Start columns of the fused projection (documented by ``fused_layout``) and its padded width."""
    cols, at = {}, 0
    for name, width in (("Q", 64), ("K", 64), ("V", 64), ("B", 32), ("C", 32), ("TH", 16), ("A", 1)):
        cols[name] = at
        at += width * H
    cols["NTOT"], cols["NPAD"] = at, -(-at // 16) * 16
    return cols


def _config(D: int) -> SISAConfig:
    return SISAConfig.preset(PRESET_OF_WIDTH[D])


def _fill_parameters(module, cfg: SISAConfig, gen) -> None:
    """Weights of a trained model's scale: the initialisation's, with a non-zero W_C and spread gains and gates."""
    for name, p in module.named_parameters():
        noise = torch.randn(p.shape, generator=gen, device=DEVICE)
        if name.endswith("norm.weight"):
            value = 1.0 + 0.1 * noise
        elif name.endswith("alpha_proj.bias"):
            value = cfg.decay_bias_init + 0.5 * noise
        elif name.endswith("forget_proj.bias"):
            value = cfg.forget_bias_init + 0.5 * noise
        elif name.endswith("lambda_raw"):
            value = cfg.lambda_raw_init + 0.3 * noise
        elif name.endswith("theta_proj.weight"):
            value = cfg.theta_init_std * noise
        else:
            value = cfg.init_std * noise
        p.data.copy_(value)


def prepare(case: dict, seed: int) -> dict:
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]

    def normal(*shape, mean=0.0, std=1.0, dtype=torch.float32):
        return (mean + std * torch.randn(shape, generator=gen, device=DEVICE)).to(dtype)

    if kind == "fused":
        B, T, H = case["B"], case["T"], case["H"]
        dt, cols = DTYPES[case["dtype"]], _columns(H)
        a_mean, a_std, z_std = (-7.0, 1.0, 1.0) if case["long_lived"] else (-5.0, 0.5, 0.5)
        proj = torch.zeros((B, T, cols["NPAD"]), device=DEVICE, dtype=dt)
        proj[..., :cols["TH"]] = normal(B, T, cols["TH"], dtype=dt)
        proj[..., cols["TH"]:cols["A"]] = normal(B, T, 16 * H, std=0.01, dtype=dt)
        proj[..., cols["A"]:cols["NTOT"]] = normal(B, T, H, mean=a_mean, std=a_std, dtype=dt)
        state = dict(proj=proj, z=normal(B, T, H, mean=4.0, std=z_std) if case["forget"] else None,
                     lam=F.softplus(normal(H, mean=-1.0, std=0.3)))
        if case["train"]:
            state["dy"] = normal(B, T, 64 * H, dtype=dt)
    elif kind == "attn":
        B, T, H = case["B"], case["T"], case["H"]
        dt = DTYPES[case["dtype"]]
        state = {n: normal(B, H, T, D_HEAD, dtype=dt) for n in ("q", "k", "v")}
        state.update({n: normal(B, H, T, D_STATE, dtype=dt) for n in ("c", "b")})
        state["g"] = torch.cumsum(-F.softplus(normal(B, H, T, mean=-5.0, std=0.5)), -1)
        state["f"] = torch.cumsum(F.logsigmoid(normal(B, H, T, mean=4.0, std=0.5)), -1) if case["forget"] else None
        state["lam"] = F.softplus(normal(H, mean=-1.0, std=0.3))
        if case["train"]:
            state["do"] = normal(B, H, T, D_HEAD, dtype=dt)
    elif kind == "lmce":
        N, D, V = case["N"], case["D"], case["V"]
        labels = torch.randint(0, V, (N,), generator=gen, device=DEVICE)
        if case["ignored"]:
            labels[:int(case["ignored"] * N)] = -100
        state = dict(hidden=normal(N, D, dtype=DTYPES[case["dtype"]]), weight=normal(V, D, std=0.02), labels=labels)
    elif kind == "norm":
        N, D, H = case["N"], case["D"], case["H"]
        dt = DTYPES[case["dtype"]]
        state = dict(x=normal(N, D), res=normal(N, D, dtype=dt), weight=normal(D, mean=1.0, std=0.1),
                     wf=normal(H, D, std=0.02), bf=normal(H, mean=4.0, std=0.5), dh=normal(N, D),
                     dy=normal(N, D, dtype=dt), dz=normal(N, H))
    elif kind == "block":
        cfg = _config(case["D"])
        with torch.device(DEVICE):
            block = SISABlock(cfg)
        _fill_parameters(block, cfg, gen)
        return dict(case=case, block=block, x=normal(case["B"], case["T"], case["D"]).requires_grad_(True),
                    dy=normal(case["B"], case["T"], case["D"]))
    elif kind == "decode":
        B, H, T = case["B"], case["H"], case["T"]
        dt, room = DTYPES[case["dtype"]], T + 64           # the cache slab holds the tokens still to come, too
        slab = dict(k=normal(B, H, room, D_HEAD, dtype=dt), v=normal(B, H, room, D_HEAD, dtype=dt),
                    b=normal(B, H, room, D_STATE, dtype=dt),
                    g=torch.cumsum(-F.softplus(normal(B, H, room, mean=-5.0, std=0.5)), -1),
                    f=torch.cumsum(F.logsigmoid(normal(B, H, room, mean=4.0, std=0.5)), -1))
        return dict(case=case, **{n: t[:, :, :T] for n, t in slab.items()}, q=normal(B, H, 1, D_HEAD, dtype=dt),
                    c=normal(B, H, 1, D_STATE, dtype=dt), g_q=slab["g"][:, :, T - 1:T].clone(),
                    f_q=slab["f"][:, :, T - 1:T].clone(), lam=F.softplus(normal(H, mean=-1.0, std=0.3)))
    else:
        cfg = _config(case["D"])
        with torch.device(DEVICE):
            model = SISAForCausalLM(cfg)
        _fill_parameters(model, cfg, gen)
        ids = torch.randint(0, cfg.vocab_size, (case["B"], case["T"] + case["steps"]), generator=gen, device=DEVICE)
        return dict(case=case, model=model.to(torch.bfloat16).eval(), ids=ids)
    grads = {"fused": ("proj", "z", "lam"), "attn": ("q", "k", "v", "c", "b", "g", "lam", "f"),
             "lmce": ("hidden", "weight"), "norm": ("x", "res", "weight", "wf", "bf")}[kind]
    if case.get("train", True):
        for n in grads:
            if state[n] is not None:
                state[n].requires_grad_(True)
    state["case"] = case
    return state


# ------------------------------------------------------------------------------------------------ one pass
def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "fused":
        y = sisa_fused(state["proj"], state["z"], state["lam"], case["H"])
        if not case["train"]:
            return [y]
        leaves = [t for t in (state["proj"], state["z"], state["lam"]) if t is not None]
        return [y.detach(), *torch.autograd.grad(y, leaves, state["dy"])]
    if kind == "attn":
        o = sisa_attention(state["q"], state["k"], state["v"], state["c"], state["b"], state["g"], state["lam"],
                           state["f"], impl="hip")
        if not case["train"]:
            return [o]
        leaves = [state[n] for n in ("q", "k", "v", "c", "b", "g", "lam", "f") if state[n] is not None]
        return [o.detach(), *torch.autograd.grad(o, leaves, state["do"])]
    if kind == "lmce":
        if not case["train"]:
            with torch.no_grad():
                return [linear_cross_entropy(state["hidden"], state["weight"], state["labels"])]
        loss = linear_cross_entropy(state["hidden"], state["weight"], state["labels"])
        return [loss.detach(), *torch.autograd.grad(loss, (state["hidden"], state["weight"]))]
    if kind == "norm":
        outs = rms_norm_forget_add_hip(state["x"], state["res"], state["weight"], 1e-6, state["wf"], state["bf"],
                                       DTYPES[case["dtype"]])
        leaves = [state[n] for n in ("x", "res", "weight", "wf", "bf")]
        grads = torch.autograd.grad(outs, leaves, (state["dh"], state["dy"], state["dz"]))
        return [*(t.detach() for t in outs), *grads]
    if kind == "block":
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = state["block"](state["x"])
        return [y.detach(), *torch.autograd.grad(y, [state["x"], *state["block"].parameters()], state["dy"])]
    if kind == "decode":
        return [sisa_decode_hip(state["q"], state["k"], state["v"], state["c"], state["b"], state["g_q"], state["g"],
                                state["lam"], state["f_q"], state["f"], case["T"] - 1)]
    model, ids, T = state["model"], state["ids"], case["T"]
    with torch.no_grad():
        cache = SISACache(capacity=ids.shape[1])
        logits = [model(ids[:, :T], cache=cache, logits_to_keep=1).logits]
        for t in range(T, ids.shape[1]):
            logits.append(model(ids[:, t:t + 1], cache=cache, logits_to_keep=1).logits)
    return logits


# ------------------------------------------------------------------------------------------------ necessary work
def work(case: dict) -> dict:
    """Bytes and floating-point operations of one pass that no implementation can leave out: every input read and
    every output written once, the causal half of the attention's products, the GEMMs' products."""
    kind = case["kind"]
    if kind in ("fused", "attn"):
        B, T, H, es, train = case["B"], case["T"], case["H"], BYTES[case["dtype"]], case["train"]
        pairs = B * H * T * (T + 1) / 2
        flops = pairs * (4 * D_HEAD + 2 * D_STATE + (10 * D_HEAD + 6 * D_STATE if train else 0))
        gates = 4 * (1 + case["forget"])
        if kind == "fused":
            inputs, outputs = B * T * H * (273 * es + 4 * case["forget"]), B * T * H * 64 * es
        else:
            inputs, outputs = B * T * H * (256 * es + gates), B * T * H * 64 * es
        return dict(bytes=(inputs + outputs) * (2 if train else 1), flops=flops)
    if kind == "lmce":
        N, D, V, train = case["N"], case["D"], case["V"], case["train"]
        return dict(bytes=(N * D * 2 + V * D * 4) * (2 if train else 1) + 8 * N, flops=2.0 * N * V * D * (3 if train
                                                                                                         else 1))
    if kind == "norm":
        N, D, H = case["N"], case["D"], case["H"]
        return dict(bytes=N * (D * (4 + 2 + 4 + 2 + 4 + 2 + 4 + 2) + 8 * H), flops=6.0 * N * D * H + 20.0 * N * D)
    if kind == "block":
        B, T, D = case["B"], case["T"], case["D"]
        H, ff, rows = D // 64, _config(D).d_ff, B * T
        params = D * (273 * H + H + D + 3 * ff)
        return dict(bytes=rows * D * 4 * 4 + params * 8,
                    flops=6.0 * rows * params + 1152.0 * B * H * T * (T + 1) / 2)
    if kind == "decode":
        B, H, T, es = case["B"], case["H"], case["T"], BYTES[case["dtype"]]
        return dict(bytes=B * H * T * (160 * es + 8), flops=320.0 * B * H * T)
    cfg, B, T, steps = _config(case["D"]), case["B"], case["T"], case["steps"]
    params = cfg.num_parameters()
    body = params - cfg.vocab_size * cfg.d_model
    return dict(bytes=(1 + steps) * (2.0 * params + 2 * B * cfg.vocab_size),
                flops=2.0 * B * ((T + steps) * body + (1 + steps) * (params - body)))


# ------------------------------------------------------------------------------------------------ tolerances
def tolerance(case: dict) -> dict:
    """Largest relative error of an output between two correct implementations at the same precision: about four
    times what the outputs were seen to differ from 64-bit arithmetic by.

    Seen (bf16; fp16 is an eighth of it): attention outputs and gradients 2.5e-3 to 4e-3; LM-head gradients 2.3e-3 to
    3.2e-3, its mean loss alone 8e-7 to 4e-6; norm outputs 1.7e-3; a block's parameter gradients up to 2.4e-2, a whole
    model's logits 1.4e-2. The fused layer's theta gradient, a sum over all later positions of terms that cancel, is
    off by about 4e-4 sqrt(T) through the rounding of the rotated B and C: two such results differ by up to about
    sqrt(2) times that. Decode accumulates in fp32 and returns fp32 (2e-7), the fp32 attention is within 7e-7."""
    kind, scale = case["kind"], {"bf16": 1.0, "fp16": 0.125, "fp32": 0.0}[case.get("dtype", "bf16")]
    if kind == "decode" or scale == 0.0:
        return {"rel": 1e-5}
    if kind == "lmce" and not case["train"]:
        return {"rel": 1e-4}
    if kind == "fused" and case["train"]:
        return {"rel": scale * max(1.5e-2, 6e-4 * math.sqrt(case["T"]))}
    return {"rel": scale * {"fused": 1.5e-2, "attn": 1.5e-2, "lmce": 1.2e-2, "norm": 7e-3, "block": 6e-2,
                            "generate": 5e-2}[kind]}


# ------------------------------------------------------------------------------------------------ 64-bit results
def _rotated(x, phi):
    re, im = x[..., 0::2], x[..., 1::2]
    cos, sin = torch.cos(phi), torch.sin(phi)
    return torch.stack((re * cos - im * sin, re * sin + im * cos), -1).flatten(-2)


def _attend(q, k, v, c, b, g, f, lam):
    """Dense attention of (n, T, .) heads in the operands' precision; ``lam`` (n,), ``f`` may be None."""
    T = q.shape[1]
    future = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1)
    decay = (g[:, :, None] - g[:, None, :]).masked_fill(future, 0.0).exp()
    s = q @ k.transpose(1, 2) / math.sqrt(D_HEAD) + lam[:, None, None] * decay * (c @ b.transpose(1, 2))
    if f is not None:
        s = s + (f[:, :, None] - f[:, None, :])
    return s.masked_fill(future, float("-inf")).softmax(-1) @ v


def _attend_grads(ops: dict, lam, do):
    """Output and gradients of (B, H, T, .) float64 operands, some heads at a time; ``do`` None: the output alone.
    Gradients of a head's slices and, summed over the batch, of ``lam``."""
    B, H, T, _ = ops["q"].shape
    names = [n for n in ops if ops[n] is not None]
    flat = {n: ops[n].reshape(B * H, *ops[n].shape[2:]) for n in names}
    lam_all = lam.repeat(B)
    out, grads = [], {n: [] for n in (*names, "lam")}
    per = max(1, int(2.7e8 / (T * T)))
    for i in range(0, B * H, per):
        part = {n: flat[n][i:i + per].detach().requires_grad_(do is not None) for n in names}
        lam_i = lam_all[i:i + per].detach().requires_grad_(do is not None)
        o = _attend(part["q"], part["k"], part["v"], part["c"], part["b"], part["g"], part.get("f"), lam_i)
        out.append(o.detach())
        if do is not None:
            dpart = torch.autograd.grad(o, [*part.values(), lam_i], do.reshape(B * H, T, -1)[i:i + per])
            for n, d in zip((*part, "lam"), dpart):
                grads[n].append(d)
    o = torch.cat(out).view(B, H, T, -1)
    if do is None:
        return o, None
    full = {n: torch.cat(ds).view(ops[n].shape) for n, ds in grads.items() if n != "lam"}
    full["lam"] = torch.cat(grads["lam"]).view(B, H).sum(0)
    return o, full


def _split_heads(x, H: int):
    return x.unflatten(-1, (H, -1)).transpose(1, 2)


def _fused_operands(proj, z, H: int) -> dict:
    cols = _columns(H)

    def part(a, b):
        return _split_heads(proj[..., cols[a]:cols[b]], H)

    phi = part("TH", "A").cumsum(2)
    ops = dict(q=part("Q", "K"), k=part("K", "V"), v=part("V", "B"), c=_rotated(part("C", "TH"), phi),
               b=_rotated(part("B", "C"), phi), g=(-F.softplus(part("A", "NTOT").squeeze(-1))).cumsum(2))
    ops["f"] = None if z is None else F.logsigmoid(z.transpose(1, 2)).cumsum(2)
    return ops


def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w


def _block64(x, P: dict, H: int):
    """One decoder block of a (1, T, D) input with the parameters ``P`` by their names in ``SISABlock``."""
    def lin(t, name):
        return F.linear(t, P[name + ".weight"], P.get(name + ".bias"))

    def heads(name):
        return _split_heads(lin(n, "attn." + name), H)

    n = _rms(x, P["attn_norm.weight"])
    phi = heads("theta_proj").cumsum(2)
    c, b = _rotated(heads("W_C"), phi), _rotated(heads("W_B"), phi)
    g = (-F.softplus(lin(n, "attn.alpha_proj"))).transpose(1, 2).cumsum(2)
    f = F.logsigmoid(lin(n, "attn.forget_proj")).transpose(1, 2).cumsum(2)
    lam = F.softplus(P["attn.lambda_raw"])
    y = torch.cat([_attend(heads("W_Q")[i], heads("W_K")[i], heads("W_V")[i], c[i], b[i], g[i], f[i], lam)[None]
                   for i in range(x.shape[0])])
    x = x + lin(y.transpose(1, 2).flatten(2), "attn.W_O")
    m = _rms(x, P["ffn_norm.weight"])
    return x + lin(F.silu(lin(m, "ffn.w_gate")) * lin(m, "ffn.w_up"), "ffn.w_down")


def exact(case: dict, seed: int):
    state = prepare(case, seed)
    kind = case["kind"]

    def wide(t):
        return None if t is None else t.detach().double()

    if kind == "fused":
        H = case["H"]
        proj, z, lam = wide(state["proj"]).requires_grad_(True), wide(state["z"]), wide(state["lam"])
        if z is not None:
            z.requires_grad_(True)
        ops = _fused_operands(proj, z, H)
        do = _split_heads(wide(state["dy"]), H) if case["train"] else None
        o, grads = _attend_grads(ops, lam, do)
        y = o.transpose(1, 2).flatten(2)
        if not case["train"]:
            return [y]
        names = [n for n in ops if ops[n] is not None]
        leaves = [proj] if z is None else [proj, z]
        return [y, *torch.autograd.grad([ops[n] for n in names], leaves, [grads[n] for n in names]), grads["lam"]]
    if kind == "attn":
        ops = {n: wide(state[n]) for n in ("q", "k", "v", "c", "b", "g", "f")}
        o, grads = _attend_grads(ops, wide(state["lam"]), wide(state["do"]) if case["train"] else None)
        if not case["train"]:
            return [o]
        return [o, *(grads[n] for n in ("q", "k", "v", "c", "b", "g", "lam", "f") if n in grads)]
    if kind == "lmce":
        x, W, labels = wide(state["hidden"]), wide(state["weight"]), state["labels"]
        valid = (labels != -100).sum()
        loss, dx, dW = x.new_zeros(()), torch.empty_like(x), torch.zeros_like(W)
        for i in range(0, x.shape[0], 2048):
            xi, li = x[i:i + 2048], labels[i:i + 2048]
            keep, rows = li != -100, torch.arange(li.numel(), device=li.device)
            logp = torch.log_softmax(xi @ W.t(), -1)
            target = li.clamp(min=0)
            loss = loss - (logp[rows, target] * keep).sum() / valid
            if case["train"]:
                G = logp.exp()
                G[rows, target] -= 1.0
                G *= keep[:, None] / valid
                dx[i:i + 2048] = G @ W
                dW += G.t() @ xi
        return [loss, dx, dW] if case["train"] else [loss]
    if kind == "norm":
        x, res, w, wf, bf = (wide(state[n]).requires_grad_(True) for n in ("x", "res", "weight", "wf", "bf"))
        h = x + res
        y = _rms(h, w)
        outs = (h, y, F.linear(y, wf, bf))
        grads = torch.autograd.grad(outs, (x, res, w, wf, bf), tuple(wide(state[n]) for n in ("dh", "dy", "dz")))
        return [*(t.detach() for t in outs), *grads]
    if kind == "block":
        names = [n for n, _ in state["block"].named_parameters()]
        P = {n: wide(p).requires_grad_(True) for n, p in state["block"].named_parameters()}
        x, dy = wide(state["x"]), wide(state["dy"])
        ys, dxs, total = [], [], None
        for i in range(case["B"]):
            xi = x[i:i + 1].requires_grad_(True)
            y = _block64(xi, P, case["D"] // 64)
            got = torch.autograd.grad(y, [xi, *(P[n] for n in names)], dy[i:i + 1])
            ys.append(y.detach())
            dxs.append(got[0])
            total = list(got[1:]) if total is None else [a + b for a, b in zip(total, got[1:])]
        return [torch.cat(ys), torch.cat(dxs), *total]
    if kind == "decode":
        q, k, v, c, b, g, f, lam = (wide(state[n]) for n in ("q", "k", "v", "c", "b", "g", "f", "lam"))
        s = (q * k).sum(-1) / math.sqrt(D_HEAD) + lam[:, None] * (wide(state["g_q"]) - g).exp() * (c * b).sum(-1)
        p = (s + wide(state["f_q"]) - f).softmax(-1)
        return [(p[..., None] * v).sum(2, keepdim=True)]
    model, ids, T = state["model"], state["ids"], case["T"]
    P = {n: wide(p) for n, p in model.named_parameters()}
    with torch.no_grad():
        x = F.embedding(ids, P["embed.weight"])
        for i in range(model.config.n_layer):
            pre = f"layers.{i}."
            x = _block64(x, {n[len(pre):]: p for n, p in P.items() if n.startswith(pre)}, model.config.n_head)
        logits = _rms(x, P["final_norm.weight"])[:, T - 1:] @ P["embed.weight"].t()
    return [logits[:, i:i + 1] for i in range(logits.shape[1])]
