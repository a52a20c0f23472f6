"""The work whose time is measured: calls of the public entry points over their real range.

Kinds of case:

* ``flash``    one training call of ``flash_pn_fir_tau_attention``: O and the gradients of q, k,
               v and tau for a given dO, bf16 or fp32, any head size, with or without silent keys;
* ``mha``      one training call of the ``PnFirTauFlashMHA`` module under bf16 autocast: its
               output, the gradient of its input and of every parameter;
* ``scores``   one training call of ``hip_pn_fir_tau_scores`` on materialised scores: W and the
               gradients of the scores and of tau;
* ``fir``      the key FIR over [B, H, N, d] keys and its adjoint;
* ``lm``       inference of the language model ``WikiLM``: logits of a batch of token sequences.

``flash`` operands are either separate [B, H, N, d] tensors or (``packed``) head views of one
projection's rows [B, N, 3, H, d], as the modules hand them over.
"""
from __future__ import annotations

import math

import torch

from paper_01_anti_decoy_pnfirtau_amd import PnFirConfig, PnFirTauFlashMHA, causal_gaussian_taps
from paper_01_anti_decoy_pnfirtau_amd.hip_pnfirtau import (flash_pn_fir_tau_attention,
                                                           hip_causal_fir_heads,
                                                           hip_pn_fir_tau_scores)
from paper_01_anti_decoy_pnfirtau_amd.wikilm import WikiLM, WikiLMConfig

GAMMA = 0.5  # the modules' default silence gamma


def _flash(name, B, H, N, d, dtype="bf16", tau=0.0, silent=False, packed=False):
    return dict(name=name, kind="flash", B=B, H=H, N=N, d=d, dtype=dtype, tau=tau, silent=silent,
                packed=packed)


def listed():
    return [
        # Training on long sequences, the benchmark's headline shape: the largest call.
        _flash("flash_long", 4, 16, 8192, 64),
        # Wide heads (the wide-head ladder of the benchmark).
        _flash("flash_wide", 8, 8, 4096, 128),
        # Long sequences where a raised tau leaves half of the key tiles silent.
        _flash("flash_silent", 4, 16, 4096, 64, tau=0.25, silent=True),
        # One long sequence of ragged length in a batch of its own, from a packed projection.
        _flash("flash_one", 1, 8, 3001, 64, packed=True),
        # Many short sequences of narrow heads (the reference's kernel benchmark).
        _flash("flash_narrow", 64, 4, 256, 16),
        # A head size without a kernel of its own, ragged length.
        _flash("flash_head80", 4, 8, 1000, 80),
        # The fp32 path (parity runs with reduced precision switched off).
        _flash("flash_f32", 1, 8, 2048, 64, dtype="f32"),
        # One attention layer of the benchmark's language model in training.
        dict(name="mha_train", kind="mha", B=32, N=512, D=256, H=4, tau=0.0),
        # Materialised scores (the module with attention dropout, or asked for its weights).
        dict(name="scores", kind="scores", B=32, H=4, N=512, dtype="bf16", tau=0.0),
        # The same for a ragged sequence length.
        dict(name="scores_ragged", kind="scores", B=4, H=8, N=777, dtype="bf16", tau=0.1),
        # The key FIR and its adjoint on the benchmark's keys.
        dict(name="fir", kind="fir", B=8, H=8, N=2048, d=64, dtype="bf16", per_head=True),
        # Logits of one short prompt: the smallest call, all latency.
        dict(name="lm_prompt", kind="lm", B=1, N=100, D=64, H=4, layers=6, vocab=23168),
    ]


def _log(rng, lo, hi):
    """An integer spread evenly over the logarithm of lo .. hi."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["flash", "flash", "flash", "flash32", "mha", "scores", "scores", "fir", "lm"])
    if kind in ("flash", "flash32"):
        f32 = kind == "flash32"
        d = rng.choice([16, 32, 64, 64, 128] if f32 else [16, 32, 48, 64, 64, 64, 80, 96, 128, 128])
        N = _log(rng, 64, 3000 if f32 else 8192)
        H = rng.choice([1, 2, 4, 8, 12, 16])
        B = _log(rng, 1, 64)
        # at most the work of the longest listed case (an fp32 call costs about 25 times as much)
        cap = 4 * 16 * 8192 * 8192 * 64 / (25 if f32 else 1)
        while B > 1 and B * H * N * N * max(d, 64) > cap:
            B //= 2
        while H > 1 and B * H * N * N * max(d, 64) > cap:
            H //= 2
        silent = not f32 and rng.random() < 0.25
        tau = 0.25 if silent else rng.choice([0.0, 0.0, -0.5, 0.2])
        return dict(kind="flash", B=B, H=H, N=N, d=d, dtype="f32" if f32 else "bf16", tau=tau,
                    silent=silent, packed=rng.random() < 0.5)
    if kind == "mha":
        D, H = rng.choice([(64, 4), (128, 4), (256, 4), (512, 8), (768, 12), (1024, 8)])
        return dict(kind="mha", B=_log(rng, 1, 32), N=_log(rng, 32, 2048), D=D, H=H,
                    tau=rng.choice([0.0, -0.5, 0.1]))
    if kind == "scores":
        N = _log(rng, 50, 3000)
        H = rng.choice([1, 4, 8])
        B = max(1, min(_log(rng, 1, 32), 32 * 4 * 512 * 512 * 4 // (H * N * N)))
        return dict(kind="scores", B=B, H=H, N=N, dtype=rng.choice(["bf16", "bf16", "f32"]),
                    tau=rng.choice([0.0, 0.1, -0.5]))
    if kind == "fir":
        return dict(kind="fir", B=_log(rng, 1, 32), H=rng.choice([1, 4, 8, 16]),
                    N=_log(rng, 64, 8192), d=rng.choice([16, 32, 64, 80, 128]),
                    dtype=rng.choice(["bf16", "bf16", "f32"]), per_head=rng.random() < 0.5)
    return dict(kind="lm", B=_log(rng, 1, 32), N=_log(rng, 16, 256), D=rng.choice([64, 128, 256]),
                H=4, layers=rng.choice([2, 6]), vocab=23168)


# ------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _dtype(case):
    return torch.float32 if case["dtype"] == "f32" else torch.bfloat16


def _flash_inputs(case, seed):
    """q, k, v, dO.  Head size 128 and up takes N(0, 1/sqrt(d)) operands, as the benchmark's wide
    heads; v and dO carry a mean, as activations do.  ``silent``: every other block of 64 keys
    is zero, so that with tau > 0 its tiles hold no positive score."""
    B, H, N, d = case["B"], case["H"], case["N"], case["d"]
    g = _gen(seed)
    std = 1.0 if d < 128 else d ** -0.25
    if case["packed"]:
        rows = _randn(g, B, N, 3, H, d)
        q, k, v = (rows[:, :, i].transpose(1, 2) for i in range(3))
    else:
        q, k, v = (_randn(g, B, H, N, d) for _ in range(3))
    q, k, v = q * std, k * std, v * std + 0.25
    if case["silent"]:
        for j in range(0, N, 128):
            k[:, :, j:j + 64] = 0
    dO = _randn(g, B, H, N, d) + 0.25
    if case["packed"]:  # the three head views of one tensor of projection rows
        rows = torch.stack([t.transpose(1, 2) for t in (q, k, v)], 2).to(_dtype(case))
        q, k, v = (rows[:, :, i].transpose(1, 2) for i in range(3))
        return q, k, v, dO.to(_dtype(case))
    return tuple(t.to(_dtype(case)) for t in (q, k, v, dO))


def _scores_inputs(case, seed):
    B, H, N = case["B"], case["H"], case["N"]
    g = _gen(seed)
    raw = (_randn(g, B, H, N, N) * 8.0).to(_dtype(case))  # q . k of unit rows at d = 64
    dw = (_randn(g, B, H, N, N) + 0.25).to(_dtype(case))
    return raw, dw


def _fir_inputs(case, seed):
    g = _gen(seed)
    shape = (case["B"], case["H"], case["N"], case["d"])
    k, gy = _randn(g, *shape).to(_dtype(case)), _randn(g, *shape).to(_dtype(case))
    if case["per_head"]:
        taps = torch.rand(case["H"], 7, generator=g, device="cuda")
        taps = taps / taps.sum(-1, keepdim=True)
    else:
        taps = causal_gaussian_taps(7, "cuda")
    return k, gy, taps


def _module(case, seed):
    with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
        torch.manual_seed(seed)
        if case["kind"] == "mha":
            cfg = PnFirConfig(d_model=case["D"], n_heads=case["H"], tau_init=case["tau"])
            return PnFirTauFlashMHA(cfg).cuda()
        cfg = WikiLMConfig(d_model=case["D"], n_heads=case["H"], n_layers=case["layers"],
                           d_ff=4 * case["D"], max_seq=256)
        return WikiLM(case["vocab"], cfg, "pn_fir_tau_flash").cuda().eval()


def _mha_inputs(case, module, seed):
    """x is a LayerNorm's output (fp32 under autocast).  dy follows the layer's own output, as a
    loss's gradient does, beside noise: with noise alone the gradient of tau is a sum that cancels."""
    g = _gen(seed)
    x = _randn(g, case["B"], case["N"], case["D"])
    with torch.no_grad():
        y = _mha64(x.double(), *(t.double() for t in _mha_weights(module)), case["H"])
    dy = (y / y.std()).float() + 0.5 * _randn(g, case["B"], case["N"], case["D"])
    return x, dy.to(torch.bfloat16)


def _mha_weights(module):
    return module.qkv.weight, module.out.weight, module.score_tau, module.fir_taps


def _tokens(case, seed):
    u = torch.rand(case["B"], case["N"], generator=_gen(seed), device="cuda")
    return (case["vocab"] * u ** 4).long().clamp_(max=case["vocab"] - 1)  # frequent tokens first


def prepare(case, seed):
    kind = case["kind"]
    if kind == "flash":
        q, k, v, dO = _flash_inputs(case, seed)
        tau = torch.tensor(case["tau"], device="cuda")
        return dict(kind=kind, args=[t.requires_grad_() for t in (q, k, v, tau)], dO=dO)
    if kind == "scores":
        raw, dw = _scores_inputs(case, seed)
        tau = torch.tensor(case["tau"], device="cuda")
        return dict(kind=kind, args=[raw.requires_grad_(), tau.requires_grad_()], dO=dw)
    if kind == "fir":
        k, gy, taps = _fir_inputs(case, seed)
        return dict(kind=kind, k=k.requires_grad_(), gy=gy, taps=taps)
    if kind == "mha":
        module = _module(case, seed)
        x, dy = _mha_inputs(case, module, seed)
        return dict(kind=kind, module=module, x=x.requires_grad_(), dy=dy)
    return dict(kind=kind, module=_module(case, seed), x=_tokens(case, seed))


def run(state):
    kind = state["kind"]
    if kind == "flash":
        o = flash_pn_fir_tau_attention(*state["args"], gamma=GAMMA)
        return [o.detach(), *torch.autograd.grad(o, state["args"], state["dO"])]
    if kind == "scores":
        w = hip_pn_fir_tau_scores(*state["args"], scale=0.125, gamma=GAMMA)
        return [w.detach(), *torch.autograd.grad(w, state["args"], state["dO"])]
    if kind == "fir":
        y = hip_causal_fir_heads(state["k"], state["taps"])
        return [y.detach(), *torch.autograd.grad(y, [state["k"]], state["gy"])]
    if kind == "mha":
        with torch.autocast("cuda", torch.bfloat16):
            y = state["module"](state["x"])
        wrt = [state["x"], *state["module"].parameters()]
        return [y.detach(), *torch.autograd.grad(y, wrt, state["dy"])]
    with torch.no_grad(), torch.autocast("cuda", torch.bfloat16):
        return state["module"](state["x"])


# -------------------------------------------------------------------------- the bare work
def work(case):
    kind = case["kind"]
    if kind == "lm":
        rows, D, V = case["B"] * case["N"], case["D"], case["vocab"]
        layer = 12 * D * D
        att = 4 * case["B"] * D * case["N"] * (case["N"] + 1) // 2
        return dict(bytes=4 * (V * D + case["layers"] * layer) + 2 * rows * V,
                    flops=2 * rows * (V * D + case["layers"] * layer) + case["layers"] * att)
    if kind == "mha":
        rows, D = case["B"] * case["N"], case["D"]
        att = 14 * case["B"] * D * case["N"] * (case["N"] + 1) // 2
        # x, y, dy, dx; the weights read and their gradients written (fp32)
        return dict(bytes=rows * D * (4 + 2 + 2 + 4) + 2 * 4 * 4 * D * D,
                    flops=3 * 2 * rows * 4 * D * D + att)
    es = 4 if case["dtype"] == "f32" else 2
    if kind == "flash":
        n = case["B"] * case["H"] * case["N"] * case["d"]
        pairs = case["B"] * case["H"] * case["N"] * (case["N"] + 1) // 2
        # 2 products forward, 5 backward (the scores once more)
        return dict(bytes=8 * n * es, flops=14 * case["d"] * pairs // (2 if case["silent"] else 1))
    if kind == "scores":
        n = case["B"] * case["H"] * case["N"] * case["N"]
        return dict(bytes=3 * n * es, flops=30 * n)  # half of raw and dW, all of W and dScores
    n = case["B"] * case["H"] * case["N"] * case["d"]
    return dict(bytes=4 * n * es, flops=2 * 14 * n)


def tolerance(case):
    """About four times the largest error against exact() that any output showed, over the listed
    cases and some dozens of drawn ones."""
    kind = case["kind"]
    if kind == "lm":
        return dict(rel=1.6e-2)  # 0.004: six layers of bf16 products
    if kind == "mha":
        return dict(rel=1e-1)  # 0.025: bf16 projections under u^10, whose gradient takes nine of u
    if case["dtype"] == "f32":
        return dict(rel={"flash": 6e-6, "scores": 2e-6, "fir": 1e-6}[kind])
    return dict(rel={"flash": 1.5e-2, "scores": 7e-3, "fir": 7e-3}[kind])


# ---------------------------------------------------------------- the same in 64 bits, plainly
def _attend(q, k, v, tau, scale, dO=None):
    """pn_fir_tau attention of one head, q, k, v [N, d] in 64 bits: O, and with dO the gradients
    (dq, dk, dv, dtau); ties of a row's peak share its gradient."""
    n = q.shape[0]
    u = (q @ k.T).mul_(scale).sub_(tau).clamp_(min=0).tril_()
    p = u ** 10
    z = p.sum(-1, keepdim=True) + 1e-12
    m = u.amax(-1, keepdim=True)
    gate = m / (m + GAMMA)
    w = p.div_(z)
    o = gate * (w @ v)
    if dO is None:
        return o
    dv = (gate * w).T @ dO
    dw = dO @ v.T
    dgate = (w * dw).sum(-1, keepdim=True)
    peak = (u == m) & (u > 0)
    share = dgate * GAMMA / (m + GAMMA) ** 2 / peak.sum(-1, keepdim=True).clamp(min=1)
    du = u.pow_(9).mul_(10.0 * gate / z).mul_(dw.sub_(dgate))
    du += peak * share
    ds = du * scale
    assert ds.shape == (n, n)
    return o, ds @ k, ds.T @ q, dv, -du.sum()


class _Attend(torch.autograd.Function):
    """_attend over [B, H, N, d], one head at a time."""

    @staticmethod
    def forward(ctx, q, k, v, tau, scale):
        ctx.save_for_backward(q, k, v, tau)
        ctx.scale = scale
        o = torch.empty_like(q)
        for b in range(q.shape[0]):
            for h in range(q.shape[1]):
                o[b, h] = _attend(q[b, h], k[b, h], v[b, h], tau, scale)
        return o

    @staticmethod
    def backward(ctx, dO):
        q, k, v, tau = ctx.saved_tensors
        grads = [torch.empty_like(q) for _ in range(3)]
        dtau = torch.zeros_like(tau)
        for b in range(q.shape[0]):
            for h in range(q.shape[1]):
                _, *g, dt = _attend(q[b, h], k[b, h], v[b, h], tau, ctx.scale, dO[b, h])
                for out, part in zip(grads, g):
                    out[b, h] = part
                dtau += dt
        return *grads, dtau, None


def _fir64(x, taps):
    """Causal FIR along the next to last axis; taps broadcast against x, the newest last."""
    y = torch.zeros_like(x)
    n, K = x.shape[-2], taps.shape[-1]
    for u in range(min(K, n)):
        y[..., u:, :] += taps[..., K - 1 - u] * x[..., :n - u, :]
    return y


def _mha64(x, w_qkv, w_out, tau, taps, H):
    B, N, D = x.shape
    q, k, v = (x @ w_qkv.T).split(D, dim=-1)
    k = _fir64(k, taps)
    q, k, v = (t.reshape(B, N, H, D // H).transpose(1, 2).contiguous() for t in (q, k, v))
    o = _Attend.apply(q, k, v, tau, 1.0 / math.sqrt(D // H))
    return o.transpose(1, 2).reshape(B, N, D) @ w_out.T


def _exact_scores(case, seed):
    raw, dw = (t.double() for t in _scores_inputs(case, seed))
    w, draw_, dtau = torch.empty_like(raw), torch.empty_like(raw), 0.0
    for b in range(case["B"]):
        u = (raw[b] * 0.125 - case["tau"]).clamp_(min=0).tril_()
        z = (u ** 10).sum(-1, keepdim=True) + 1e-12
        m = u.amax(-1, keepdim=True)
        gate = m / (m + GAMMA)
        share = u ** 10 / z
        w[b] = gate * share
        dgate = (share * dw[b]).sum(-1, keepdim=True)
        peak = (u == m) & (u > 0)
        du = u ** 9 * (10.0 * gate / z) * (dw[b] - dgate)
        du += peak * (dgate * GAMMA / (m + GAMMA) ** 2 / peak.sum(-1, keepdim=True).clamp(min=1))
        draw_[b] = du * 0.125
        dtau = dtau - du.sum()
    return [w, draw_, dtau]


@torch.no_grad()
def _exact_lm(case, seed):
    model, x = _module(case, seed), _tokens(case, seed)
    p = {n: t.double() for n, t in model.state_dict().items()}

    def norm(h, name):
        return torch.nn.functional.layer_norm(h, h.shape[-1:], p[name + ".weight"], p[name + ".bias"])

    h = p["embed.weight"][x] + p["pos.weight"][:case["N"]]
    for i in range(case["layers"]):
        b = f"blocks.{i}."
        h = h + _mha64(norm(h, b + "ln1"), p[b + "attn.qkv.weight"], p[b + "attn.out.weight"],
                       p[b + "attn.score_tau"], p[b + "attn.fir_taps"], case["H"])
        f = norm(h, b + "ln2") @ p[b + "ffn.0.weight"].T + p[b + "ffn.0.bias"]
        f = torch.nn.functional.gelu(f)
        h = h + f @ p[b + "ffn.2.weight"].T + p[b + "ffn.2.bias"]
    return norm(h, "ln_f") @ p["head.weight"].T


def exact(case, seed):
    kind = case["kind"]
    if kind == "flash":
        q, k, v, dO = (t.double() for t in _flash_inputs(case, seed))
        outs = [torch.empty_like(q) for _ in range(4)]
        dtau = 0.0
        for b in range(case["B"]):
            for h in range(case["H"]):
                *parts, dt = _attend(q[b, h], k[b, h], v[b, h], case["tau"],
                                     1.0 / math.sqrt(case["d"]), dO[b, h])
                for out, part in zip(outs, parts):
                    out[b, h] = part
                dtau = dtau + dt
        return [*outs, dtau]
    if kind == "scores":
        return _exact_scores(case, seed)
    if kind == "fir":
        k, gy, taps = (t.double() for t in _fir_inputs(case, seed))
        t = taps[:, None, None, :] if case["per_head"] else taps
        return [_fir64(k, t), _fir64(gy.flip(-2), t).flip(-2)]
    if kind == "mha":
        module = _module(case, seed)
        x, dy = (t.double() for t in _mha_inputs(case, module, seed))
        params = [t.detach().double().requires_grad_() for t in module.parameters()]
        names = [n for n, _ in module.named_parameters()]
        by = dict(zip(names, params))
        x.requires_grad_()
        y = _mha64(x, by["qkv.weight"], by["out.weight"], by["score_tau"],
                   module.fir_taps.double(), case["H"])
        return [y.detach(), *torch.autograd.grad(y, [x, *params], dy)]
    return _exact_lm(case, seed)
