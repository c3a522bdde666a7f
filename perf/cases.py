"""The performance cases of kernelforge_amd: what its users run, over the ranges they run it at.

``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges;
``prepare`` makes a case's inputs on the GPU from a seed, ``run`` is one pass
through the public entry points, ``work`` the bytes and operations the pass
cannot do without, ``tolerance`` what another correct implementation at the
same precision may differ by, and ``exact`` the result in 64 bits from plain
torch.

A case's ``path`` is one of
  norm        ``custom_rms_norm`` (the factory kernel) on [batch, rows, dim]
  norm_train  the ``RMSNorm`` module, forward and backward
  linattn     ``qkv_attn_matmul`` on a packed qkv[B, N, 3, H*D]
  litela      a LiteLA block: projections, optional q/k norm and rotary
              embedding, linear attention; eager or as a captured graph
  fwd         ``flash_attention`` with its log-sum-exp (prefill, cross
              attention, decoding)
  train       ``flash_attention`` forward and backward
  jvp         ``flash_attention_jvp`` from a forward's cached results
  fwd_jvp     ``flash_attention_fwd_jvp``, the fused forward and tangent
"""

import math

import torch

from kernelforge_amd.flash_attention_jvp import flash_attention, flash_attention_fwd_jvp, flash_attention_jvp
from kernelforge_amd.rmsnorm import RMSNorm, custom_rms_norm
from kernelforge_amd.SANA_LinearAttention import (CUDAGraphJointLiteLA, LiteLA, optimized_joint_litela,
                                                  qkv_attn_matmul)

DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float": torch.float32}
EPS = {"norm": 1e-6, "linattn": 1e-15}


def _attn(name, path, B, Nq, Nk, Hq, Hkv, D, causal=False, dtype="bfloat16"):
    return dict(name=name, path=path, B=B, Nq=Nq, Nk=Nk, Hq=Hq, Hkv=Hkv, D=D, causal=causal, dtype=dtype)


def listed():
    return [
        # The norm of one short sequence at the smallest model width: latency.
        dict(name="norm_short", path="norm", batch=1, rows=128, dim=1152, dtype="bfloat16"),
        # The norm of a 16k-token batch at an LLM's width: memory bandwidth.
        dict(name="norm_16k", path="norm", batch=1, rows=16384, dim=4096, dtype="bfloat16"),
        # A training step's norm: bf16 activations and the module's default
        # fp32 weight, forward and both gradients.
        dict(name="norm_train", path="norm_train", batch=2, rows=4096, dim=2240, dtype="bfloat16", wdtype="float"),
        # Linear attention of a 64x64-latent image batch, 70 heads of 32.
        dict(name="linattn_image", path="linattn", B=2, N=4096, H=70, D=32, dtype="bfloat16", out="bfloat16"),
        # The same operator at wider heads, a ragged sequence and fp32 results.
        dict(name="linattn_heads64", path="linattn", B=2, N=3001, H=18, D=64, dtype="bfloat16", out="float"),
        # Serving one 32x32-latent image through a captured block.
        dict(name="litela_serving", path="litela", B=1, N=1024, H=36, norm=False, rope=False, graph=True,
             dtype="bfloat16"),
        # The full block of a large model: q/k norm and rotary embedding, eager.
        dict(name="litela_norm_rope", path="litela", B=2, N=4096, H=70, norm=True, rope=True, graph=False,
             dtype="bfloat16"),
        # Self attention of a short ragged sequence: latency.
        _attn("attn_short", "fwd", 1, 333, 333, 16, 16, 64),
        # Decoding: a few new tokens of two sequences against a long cache, grouped heads.
        _attn("attn_decode", "fwd", 2, 4, 8192, 32, 8, 128, causal=True),
        # A causal training step with grouped heads on a ragged length.
        _attn("attn_train", "train", 2, 2500, 2500, 16, 4, 128, causal=True),
        # The tangent from cached results at a diffusion transformer's head dim.
        _attn("attn_jvp_dim72", "jvp", 2, 1024, 1024, 16, 16, 72),
        # The fused forward and tangent of a long sequence.
        _attn("attn_fwd_jvp_long", "fwd_jvp", 2, 4096, 4096, 16, 16, 128),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 8e12, w["flops"] / 2.5e15)


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= most:
            return case


def _draw(rng):
    path = rng.choice(["norm", "norm_train", "linattn", "linattn", "litela", "litela", "fwd", "decode", "train",
                       "jvp", "fwd_jvp"])
    dtype = rng.choice(["bfloat16", "bfloat16", "bfloat16", "float16"])
    if path in ("norm", "norm_train"):
        batch = rng.choice([1, 1, 2, 4])
        rows = _logint(rng, 16, 16384) // batch + 1
        # Whole 16-byte vectors mostly (model widths); now and then any width.
        dim = _logint(rng, 32, 1024) * 8 if rng.random() < 0.85 else _logint(rng, 250, 8000)
        dtype = rng.choice(["bfloat16", "bfloat16", "float16", "float"])
        case = dict(path=path, batch=batch, rows=rows, dim=dim, dtype=dtype)
        if path == "norm_train":
            case["wdtype"] = rng.choice(["float", dtype])
        return case
    if path == "linattn":
        D = rng.choice([32, 32, 32, 64, 128, 16])
        B = rng.choice([1, 1, 2, 4])
        case = dict(path=path, B=B, N=_logint(rng, 200, 16384 // B),
                    H=max(1, _logint(rng, 256, 2560) // D), D=D,
                    dtype=rng.choice(["bfloat16", "bfloat16", "float16", "float"]), out=None)
        case["out"] = rng.choice(["float", case["dtype"]])
        return case
    if path == "litela":
        rope = rng.random() < 0.4
        return dict(path=path, B=rng.choice([1, 1, 2]), N=_logint(rng, 200, 6000), H=_logint(rng, 12, 70),
                    norm=rng.random() < 0.4, rope=rope, graph=not rope and rng.random() < 0.5, dtype=dtype)
    D = rng.choice([64, 64, 72, 96, 128, 128, 128, 80, 256])
    Hkv = rng.choice([1, 2, 4, 8, 16])
    Hq = Hkv * rng.choice([1, 1, 2, 4])
    B = rng.choice([1, 1, 2, 4])
    causal = rng.random() < 0.4
    if path == "decode":
        Nq, Nk = _logint(rng, 1, 32), _logint(rng, 1000, 32768)
        path = "fwd"
    else:
        Nq = _logint(rng, 100, 6000)
        # Self attention mostly; cross attention over a shorter or longer text.
        Nk = Nq if rng.random() < 0.7 else _logint(rng, 64, 4000)
        if causal and Nk < Nq:
            Nk = Nq
    return dict(path=path, B=B, Nq=Nq, Nk=Nk, Hq=Hq, Hkv=Hkv, D=D, causal=causal, dtype=dtype)


# ---------------------------------------------------------------------------
# Inputs.
# ---------------------------------------------------------------------------
def _inputs(case, seed):
    """The case's tensors, from the seed alone."""
    g = torch.Generator("cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]

    def randn(*shape, dtype=dt, scale=1.0, shift=0.0):
        return (torch.randn(shape, generator=g, device="cuda") * scale + shift).to(dtype)

    path = case["path"]
    if path in ("norm", "norm_train"):
        shape = (case["batch"], case["rows"], case["dim"])
        wdt = DTYPES[case.get("wdtype", case["dtype"])]
        t = dict(x=randn(*shape), w=randn(case["dim"], dtype=wdt, scale=0.1, shift=1.0))
        if path == "norm_train":
            t["dy"] = randn(*shape, dtype=torch.promote_types(dt, wdt))
        return t
    if path == "linattn":
        return dict(qkv=randn(case["B"], case["N"], 3, case["H"] * case["D"]))
    if path == "litela":
        C = case["H"] * 32
        t = dict(x=randn(case["B"], case["N"], C), wqkv=randn(3 * C, C, scale=C ** -0.5),
                 wproj=randn(C, C, scale=C ** -0.5), bproj=randn(C, scale=0.02))
        if case["norm"]:
            t["qw"], t["kw"] = randn(C, scale=0.1, shift=1.0), randn(C, scale=0.1, shift=1.0)
        if case["rope"]:
            pos = torch.arange(case["N"], device="cuda", dtype=torch.float32)
            freq = 10000.0 ** (-torch.arange(16, device="cuda", dtype=torch.float32) / 16)
            angle = (pos[:, None] * freq).repeat_interleave(2, dim=1)
            t["cos"], t["sin"] = angle.cos(), angle.sin()
        return t
    qs = (case["B"], case["Nq"], case["Hq"], case["D"])
    ks = (case["B"], case["Nk"], case["Hkv"], case["D"])
    t = dict(q=randn(*qs), k=randn(*ks), v=randn(*ks))
    if path in ("jvp", "fwd_jvp"):
        t |= dict(tq=randn(*qs), tk=randn(*ks), tv=randn(*ks))
    if path == "train":
        t["dout"] = randn(*qs)
    return t


def prepare(case, seed):
    t = _inputs(case, seed)
    path = case["path"]
    state = dict(case=case, t=t)
    if path == "norm":
        state["kernel"] = custom_rms_norm(case["batch"], case["rows"], case["dim"], EPS["norm"], case["dtype"])
    elif path == "norm_train":
        with torch.device("cuda"):
            module = RMSNorm(case["dim"], eps=EPS["norm"])
        module = module.to(t["w"].dtype)
        with torch.no_grad():
            module.weight.copy_(t["w"])
        t["x"].requires_grad_(True)
        state["module"] = module
    elif path == "linattn":
        state["kernel"] = qkv_attn_matmul(case["B"], case["H"], case["D"], case["N"], EPS["linattn"],
                                          case["dtype"], case["out"])
    elif path == "litela":
        C = case["H"] * 32
        dt = DTYPES[case["dtype"]]
        with torch.device("cuda"):
            if case["graph"]:
                kw = dict(batch=case["B"], seq_len=case["N"], dtype=dt)
                if case["norm"]:
                    kw["qk_norm"] = True
                module = optimized_joint_litela(C, C, **kw)
            else:
                module = LiteLA(C, C, qk_norm=case["norm"])
        module = module.to(dt)
        with torch.no_grad():
            module.qkv.weight.copy_(t["wqkv"])
            module.proj.weight.copy_(t["wproj"])
            module.proj.bias.copy_(t["bproj"])
            if case["norm"]:
                module.q_norm.weight.copy_(t["qw"])
                module.k_norm.weight.copy_(t["kw"])
        state["module"] = CUDAGraphJointLiteLA(module) if case["graph"] else module
        state["rope"] = (t["cos"], t["sin"]) if case["rope"] else None
    elif path == "jvp":
        state["out"], state["lse"] = flash_attention(t["q"], t["k"], t["v"], causal=case["causal"], return_lse=True)
    elif path == "train":
        for name in ("q", "k", "v"):
            t[name].requires_grad_(True)
    return state


def run(state):
    case, t = state["case"], state["t"]
    path = case["path"]
    if path == "norm":
        return state["kernel"](t["x"], t["w"])
    if path == "norm_train":
        module = state["module"]
        y = module(t["x"])
        return (y.detach(), *torch.autograd.grad(y, (t["x"], module.weight), t["dy"]))
    if path == "linattn":
        return state["kernel"](t["qkv"])
    if path == "litela":
        if case["graph"]:
            return state["module"](t["x"])
        with torch.inference_mode():
            return state["module"](t["x"], rotary_emb=state["rope"])
    q, k, v, causal = t["q"], t["k"], t["v"], case["causal"]
    if path == "fwd":
        return flash_attention(q, k, v, causal=causal, return_lse=True)
    if path == "train":
        out = flash_attention(q, k, v, causal=causal)
        return (out.detach(), *torch.autograd.grad(out, (q, k, v), t["dout"]))
    if path == "jvp":
        return flash_attention_jvp(q, k, v, t["tq"], t["tk"], t["tv"], state["out"], state["lse"], causal=causal)
    return flash_attention_fwd_jvp(q, k, v, t["tq"], t["tk"], t["tv"], causal=causal)


def work(case):
    path = case["path"]
    es = DTYPES[case["dtype"]].itemsize
    if path in ("norm", "norm_train"):
        n = case["batch"] * case["rows"] * case["dim"]
        if path == "norm":
            return dict(bytes=2 * n * es + case["dim"] * es, flops=4 * n)
        ws = DTYPES[case["wdtype"]].itemsize
        ys = torch.promote_types(DTYPES[case["dtype"]], DTYPES[case["wdtype"]]).itemsize
        # Forward: x in, y out; backward: x and dy in, dx out.
        return dict(bytes=n * (3 * es + 2 * ys) + 2 * case["dim"] * ws, flops=14 * n)
    if path == "linattn":
        n = case["B"] * case["N"] * case["H"] * case["D"]
        return dict(bytes=3 * n * es + n * DTYPES[case["out"]].itemsize, flops=4 * n * (case["D"] + 1))
    if path == "litela":
        M, C = case["B"] * case["N"], case["H"] * 32
        return dict(bytes=(2 * M * C + 4 * C * C) * es, flops=8 * M * C * C + 4 * M * C * 33)
    B, Nq, Nk, Hq, Hkv, D = (case[k] for k in ("B", "Nq", "Nk", "Hq", "Hkv", "D"))
    pairs = Nq * (Nk - Nq) + Nq * (Nq + 1) // 2 if case["causal"] else Nq * Nk
    products = {"fwd": 2, "train": 7, "jvp": 5, "fwd_jvp": 6}[path]
    nq, nk = B * Nq * Hq * D, B * Nk * Hkv * D
    elems = {"fwd": 2 * nq + 2 * nk,                   # q, out; k, v
             "train": 6 * nq + 6 * nk,                 # q, out; q, out, dout, dq; k, v; k, v, dk, dv
             "jvp": 4 * nq + 4 * nk,                   # q, tq, out, tangent; k, v, tk, tv
             "fwd_jvp": 4 * nq + 4 * nk}[path]
    lse = {"fwd": 1, "train": 2, "jvp": 1, "fwd_jvp": 1}[path] * B * Hq * Nq * 4
    return dict(bytes=elems * es + lse, flops=2 * products * B * Hq * pairs * D)


def tolerance(case):
    # About four times the distance from the 64-bit result, which is the
    # storage type's rounding (of the result, and of the intermediate values
    # that the operator defines in that type).
    if case["dtype"] == "float":
        return {"rel": 2e-6}
    half = case["dtype"] == "float16"
    if case["path"] == "norm" or case["path"] == "norm_train":
        return {"rel": 1e-3 if half else 8e-3}
    if case["path"] == "linattn":
        if case["out"] == "float":
            return {"rel": 2e-5}
        return {"rel": 1e-3 if half else 8e-3}
    if case["path"] == "litela":
        return {"rel": 2e-3 if half else 1.4e-2}
    return {"rel": 1.5e-3 if half else 1e-2}


# ---------------------------------------------------------------------------
# The results in 64 bits.
# ---------------------------------------------------------------------------
def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _linear_attention(qkv, H, D, eps):
    """relu(q) S / (relu(q) z + eps) per (batch, head) of qkv[B, N, 3, H*D]."""
    B, N = qkv.shape[:2]
    out = torch.empty(B, N, H * D, device=qkv.device, dtype=torch.float64)
    for b in range(B):
        for h in range(H):
            q, k, v = (qkv[b, :, p, h * D:(h + 1) * D] for p in range(3))
            q, k = q.relu(), k.relu()
            num = q @ (k.T.contiguous() @ v)
            out[b, :, h * D:(h + 1) * D] = num / (q @ k.sum(0)[:, None] + eps)
    return out


def _litela(case, t):
    B, N, H = case["B"], case["N"], case["H"]
    C = H * 32
    d = {k: v.double() for k, v in t.items()}
    qkv = (d["x"].reshape(-1, C) @ d["wqkv"].T.contiguous()).reshape(B, N, 3, C)
    for part, name in ((0, "qw"), (1, "kw")):
        if case["norm"]:
            qkv[:, :, part] = _rms(qkv[:, :, part], d[name], 1e-5)
        if case["rope"]:
            x = qkv[:, :, part].reshape(B, N, H, 16, 2)
            turned = torch.stack((-x[..., 1], x[..., 0]), dim=-1).reshape(B, N, H, 32)
            x = x.reshape(B, N, H, 32)
            qkv[:, :, part] = (x * d["cos"][:, None] + turned * d["sin"][:, None]).reshape(B, N, C)
    out = _linear_attention(qkv, H, 32, 1e-15)
    return (out.reshape(-1, C) @ d["wproj"].T.contiguous() + d["bproj"]).reshape(B, N, C)


def _attention(case, t):
    B, Nq, Nk, Hq, Hkv, D = (case[k] for k in ("B", "Nq", "Nk", "Hq", "Hkv", "D"))
    path, scale, group = case["path"], D ** -0.5, Hq // Hkv
    d = {k: v.detach() for k, v in t.items()}

    def empty(like):
        return torch.zeros(like.shape, device="cuda", dtype=torch.float64)

    out, lse = empty(d["q"]), torch.empty(B, Hq, Nq, device="cuda", dtype=torch.float64)
    tout = empty(d["q"])
    dq, dk, dv = empty(d["q"]), empty(d["k"]), empty(d["v"])
    mask = None
    if case["causal"]:
        mask = torch.arange(Nk, device="cuda") > torch.arange(Nq, device="cuda")[:, None] + (Nk - Nq)
    for b in range(B):
        for h in range(Hq):
            kv = h // group
            q = d["q"][b, :, h].double()
            k, v = d["k"][b, :, kv].double(), d["v"][b, :, kv].double()
            s = scale * (q @ k.T.contiguous())
            if mask is not None:
                s.masked_fill_(mask, -math.inf)
            lse[b, h] = torch.logsumexp(s, -1)
            p = torch.exp(s.sub_(lse[b, h][:, None]))
            out[b, :, h] = p @ v
            if path in ("jvp", "fwd_jvp"):
                tq = d["tq"][b, :, h].double()
                tk, tv = d["tk"][b, :, kv].double(), d["tv"][b, :, kv].double()
                ts = scale * (tq @ k.T.contiguous() + q @ tk.T.contiguous())
                ts = p * (ts - (p * ts).sum(-1, keepdim=True))
                tout[b, :, h] = ts @ v + p @ tv
            if path == "train":
                do = d["dout"][b, :, h].double()
                dv[b, :, kv] += p.T.contiguous() @ do
                dp = do @ v.T.contiguous()
                ds = scale * p * (dp - (p * dp).sum(-1, keepdim=True))
                dq[b, :, h] = ds @ k
                dk[b, :, kv] += ds.T.contiguous() @ q
    return {"fwd": (out, lse), "train": (out, dq, dk, dv), "jvp": tout, "fwd_jvp": (out, lse, tout)}[path]


def exact(case, seed):
    t = _inputs(case, seed)
    path = case["path"]
    if path == "norm":
        return _rms(t["x"].double(), t["w"].double(), EPS["norm"])
    if path == "norm_train":
        x, w = t["x"].double().requires_grad_(True), t["w"].double().requires_grad_(True)
        y = _rms(x, w, EPS["norm"])
        return (y.detach(), *torch.autograd.grad(y, (x, w), t["dy"].double()))
    if path == "linattn":
        return _linear_attention(t["qkv"].double(), case["H"], case["D"], EPS["linattn"])
    if path == "litela":
        return _litela(case, t)
    return _attention(case, t)
