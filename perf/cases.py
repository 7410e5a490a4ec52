"""The work that users of this package have it do, as cases to time and to check.

A case names a public entry point and its sizes:

* ``block``  one attention block (``LocalLatentAttentionTriton``), a training pass (output, input gradient and every
  parameter gradient) or a forward under ``no_grad``, in bf16 autocast with fp32 weights or in fp32;
* ``op``     the autograd op ``LLAttnFunction`` on head tensors, forward and backward;
* ``ffn``    the language model's feed-forward, forward and backward under bf16 autocast;
* ``norm``   the residual add with the RMSNorm that follows it, forward and backward;
* ``head``   the tied LM head with cross entropy, loss and gradients;
* ``lm``     the logits of the next token after a prompt: one whole forward of the model, as generation runs it.

``listed()`` gives the cases, ``draw(rng)`` one more of the same ranges; ``prepare`` makes what a program holds
before the call, ``run`` is one pass, ``exact`` the same values in float64 from plain torch.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "local-latent-attention_amd"))

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
DEVICE = "cuda"

# the architectures of the presets and benchmark configurations: d_model, heads, latent width, latent heads
ARCH = {
    "default": dict(d_model=128, n_heads=4, latent_dim=64, latent_heads=2),
    "small": dict(d_model=256, n_heads=4, latent_dim=32, latent_heads=2),
    "1024": dict(d_model=1024, n_heads=16, latent_dim=64, latent_heads=2),
    "0.55b": dict(d_model=1408, n_heads=16, latent_dim=512, latent_heads=8),
    "0.60b": dict(d_model=1536, n_heads=16, latent_dim=384, latent_heads=8),
}
# d_model, d_ff, layers, vocabulary of the 0.55b language model
LM = dict(d_model=1408, d_ff=4096, n_layers=22, vocab=32000, max_seq_len=2048)


def _block(name, arch, B, T, window, latents, dtype="bf16", grad=True, query_block=0):
    c = dict(kind="block", B=B, T=T, window=window, local_block=256, latents=latents, query_block=query_block,
             dtype=dtype, grad=grad, **ARCH[arch])
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest training pass: the test configuration in fp32, where launches and latency count
        _block("block_small_fp32", "small", 2, 512, 128, 8, dtype="fp32"),
        # a 0.55b layer in fp32 (no autocast) on one prompt of a ragged length
        _block("block_055b_fp32", "0.55b", 1, 1000, 64, 16, dtype="fp32"),
        # the benchmark layer: 0.55b preset, B16 T2048, a training pass under bf16 autocast
        _block("block_055b", "0.55b", 16, 2048, 64, 16),
        # long context: a wide window and many latents
        _block("block_long", "1024", 2, 16384, 512, 256),
        # macro-block latent queries
        _block("block_macro", "1024", 4, 8192, 256, 128, query_block=64),
        # the other preset at a small batch of a ragged length (a micro-batch of gradient accumulation)
        _block("block_060b_ragged", "0.60b", 3, 1337, 64, 16),
        # one layer's forward over a prompt, nothing kept for a backward (generation)
        _block("block_055b_prompt", "0.55b", 1, 333, 64, 16, grad=False),
        # the op on head tensors of 128 dims, a ragged length
        dict(name="op_dh128", kind="op", B=2, H=8, T=3001, Dh=128, window=256, local_block=256, Lh=4, Ldh=64,
             chunk=100, query_block=0, dtype="bf16"),
        # the feed-forward of a 0.55b layer at the benchmark's token count
        dict(name="ffn_055b", kind="ffn", B=16, T=2048, d_model=1408, d_ff=4096),
        # the residual stream's norm there
        dict(name="norm_055b", kind="norm", B=16, T=2048, d_model=1408),
        # the tied head and the loss over a 32000-token vocabulary
        dict(name="head_055b", kind="head", B=8, T=2048, d_model=1408, vocab=32000),
        # the whole 0.55b model on a prompt of 1024 tokens, as each step of generation runs it
        dict(name="lm_055b_prompt", kind="lm", B=1, T=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "block", "block", "block", "op", "ffn", "norm", "head", "lm"])
    if kind == "block":
        arch = rng.choice(sorted(ARCH))
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        T = _log_int(rng, 16, 16384 if arch == "1024" else 4096)
        if dtype == "fp32":
            T = min(T, 2048)
        most = 32768 if dtype == "bf16" else 1200 if arch in ("0.55b", "0.60b") else 4096
        T = min(T, most)
        B = rng.randint(1, max(1, min(16, most // T)))
        return _block(None, arch, B, T, rng.choice([16, 64, 64, 128, 200, 256, 512]), rng.choice([8, 16, 16, 50, 128]),
                      dtype=dtype, grad=rng.random() < 0.7, query_block=rng.choice([0, 0, 0, 16, 64, 100]))
    if kind == "op":
        T = _log_int(rng, 32, 4096)
        B = rng.randint(1, max(1, min(8, 8192 // T)))
        qb = rng.choice([0, 0, 48])
        return dict(kind="op", B=B, H=rng.choice([2, 4, 8, 12]), T=T, Dh=rng.choice([32, 64, 80, 96, 128]),
                    window=rng.choice([16, 64, 100, 256]), local_block=rng.choice([128, 256]), Lh=rng.choice([2, 4]),
                    Ldh=rng.choice([16, 32, 64]), chunk=rng.choice([16, 64, 100]), query_block=qb,
                    dtype=rng.choice(["bf16", "bf16", "fp32"]))
    if kind == "ffn":
        d, f = rng.choice([(128, 256), (1024, 4096), (1408, 4096), (1536, 4096)])
        T = _log_int(rng, 64, 2048)
        return dict(kind="ffn", B=rng.randint(1, 15), T=T, d_model=d, d_ff=f)
    if kind == "norm":
        return dict(kind="norm", B=rng.randint(1, 15), T=_log_int(rng, 16, 2048),
                    d_model=rng.choice([128, 256, 1024, 1408]))
    if kind == "head":
        return dict(kind="head", B=rng.randint(1, 7), T=_log_int(rng, 64, 2048), d_model=rng.choice([128, 1024, 1408]),
                    vocab=rng.choice([128, 8000, 32000]))
    return dict(kind="lm", B=1, T=_log_int(rng, 8, 1000))


# ---------------------------------------------------------------------------
# inputs: tensors made from the seed alone
# ---------------------------------------------------------------------------

class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(seed)

    def normal(self, shape, std=1.0, dtype=F32):
        return (torch.randn(shape, generator=self.g, device=DEVICE) * std).to(dtype)

    def ints(self, hi, shape):
        return torch.randint(0, hi, shape, generator=self.g, device=DEVICE)


def _block_params(r, d, ld, dh, n_layers=22):
    """One block's parameters as the language model initialises them (0.02 normal, residual outputs scaled down),
    with small biases and gate vectors of the size that nn.Linear gives them."""
    res = 1.0 / math.sqrt(2 * n_layers)
    p = {}
    for name, n_out, n_in, s in (("qkv_proj", 3 * d, d, 1.0), ("rq_proj", ld, d, 1.0), ("rkv_proj", 2 * ld, d, 1.0),
                                 ("r_out", d, ld, res), ("out", d, d, res)):
        p[name + ".weight"] = r.normal((n_out, n_in), 0.02 * s)
        p[name + ".bias"] = r.normal((n_out,), 0.02)
    p["gate_local.weight"] = r.normal((1, dh), 1.0 / math.sqrt(dh))
    p["gate_remote.weight"] = r.normal((1, dh), 1.0 / math.sqrt(dh))
    return p


def _ffn_params(r, d, f, n_layers=22):
    return {"w1.weight": r.normal((f, d), 0.02), "w1.bias": r.normal((f,), 0.02),
            "w2.weight": r.normal((d, f), 0.02 / math.sqrt(2 * n_layers)), "w2.bias": r.normal((d,), 0.02)}


def _inputs(c, seed):
    """Parameters and inputs of a case by name."""
    r, k = _Rand(seed), c["kind"]
    dt = F32 if c.get("dtype") == "fp32" else BF16
    if k == "block":
        t = _block_params(r, c["d_model"], c["latent_dim"], c["d_model"] // c["n_heads"])
        t["x"] = r.normal((c["B"], c["T"], c["d_model"]), 1.0, dt)
        if c["grad"]:
            t["dy"] = r.normal((c["B"], c["T"], c["d_model"]), 1.0, dt)
        return t
    if k == "op":
        B, H, T, Dh, Lh, Ldh = (c[n] for n in ("B", "H", "T", "Dh", "Lh", "Ldh"))
        qb = min(T, c["query_block"]) if c["query_block"] > 1 else 1
        nq, nc = -(-T // qb), -(-T // c["chunk"])
        t = {n: r.normal((B, H, T, Dh), 1.0, dt) for n in ("Q", "K", "V", "dO")}
        t["GQ"] = r.normal((B, Lh, nq, Ldh), 1.0, dt)
        t["GK"], t["GV"] = (r.normal((B, Lh, nc, Ldh), 1.0, dt) for _ in range(2))
        t["gate_l"], t["gate_r"] = (r.normal((1, Dh), 1.0 / math.sqrt(Dh)) for _ in range(2))
        t["r_w"] = r.normal((H * Dh, Lh * Ldh), 1.0 / math.sqrt(Lh * Ldh))
        t["r_b"] = r.normal((H * Dh,), 0.02)
        return t
    if k == "ffn":
        t = _ffn_params(r, c["d_model"], c["d_ff"])
        t["x"], t["dy"] = (r.normal((c["B"], c["T"], c["d_model"]), 1.0, BF16) for _ in range(2))
        return t
    if k == "norm":
        s = (c["B"], c["T"], c["d_model"])
        return {"x": r.normal(s, 1.5), "res": r.normal(s, 0.5, BF16), "w": 1.0 + r.normal((c["d_model"],), 0.1),
                "ds": r.normal(s), "dy": r.normal(s, 1.0, BF16)}
    if k == "head":
        n, V, D = c["B"] * c["T"], c["vocab"], c["d_model"]
        w = r.normal((V, D), 0.02)
        targets = r.ints(V, (n,))
        # hidden states of a partly trained model: each leans towards its target's row by an amount of its own
        lean = torch.rand((n, 1), generator=r.g, device=DEVICE) * 0.3
        h = r.normal((n, D)) + lean * w[targets] / 0.02
        h = h * torch.rsqrt(h.square().mean(-1, keepdim=True))
        return {"w": w, "h": h.to(BF16).view(c["B"], c["T"], D), "targets": targets.view(c["B"], c["T"])}
    if k == "lm":
        a, t = ARCH["0.55b"], {}
        for i in range(LM["n_layers"]):
            for n, v in _block_params(r, a["d_model"], a["latent_dim"], a["d_model"] // a["n_heads"]).items():
                t[f"blocks.{i}.attn.{n}"] = v
            for n, v in _ffn_params(r, LM["d_model"], LM["d_ff"]).items():
                t[f"blocks.{i}.ff.{n}"] = v
            for n in ("norm1", "norm2"):
                t[f"blocks.{i}.{n}.weight"] = 1.0 + r.normal((LM["d_model"],), 0.1)
        t["norm.weight"] = 1.0 + r.normal((LM["d_model"],), 0.1)
        t["embedding.weight"] = r.normal((LM["vocab"], LM["d_model"]), 0.02)
        t["position.weight"] = r.normal((LM["max_seq_len"], LM["d_model"]), 0.02)
        t["ids"] = r.ints(LM["vocab"], (c["B"], c["T"]))
        return t
    raise ValueError(f"unknown case kind {k!r}")


def _load(module, t):
    """Copy the tensors into the module's parameters of the same names."""
    with torch.no_grad():
        for n, p in module.named_parameters():
            p.copy_(t[n])
    return module


def prepare(case, seed):
    c, t = case, _inputs(case, seed)
    s = {"case": c}
    if c["kind"] == "block":
        from llattn_amd import LocalLatentAttentionTriton
        with torch.device(DEVICE):
            m = LocalLatentAttentionTriton(c["d_model"], c["n_heads"], c["latent_heads"], c["latent_dim"],
                                           c["latents"], c["window"], local_block_size=c["local_block"],
                                           latent_query_block_size=c["query_block"])
        s["m"] = _load(m, t)
        s["x"] = t["x"].requires_grad_(c["grad"])
        s["dy"] = t.get("dy")
    elif c["kind"] == "op":
        s.update({n: (v if n == "dO" else v.requires_grad_(True)) for n, v in t.items()})
    elif c["kind"] == "ffn":
        from llattn_amd.config import ModelConfig
        from llattn_amd.lm import FeedForward
        with torch.device(DEVICE):
            m = FeedForward(ModelConfig(d_model=c["d_model"], d_ff=c["d_ff"]))
        s["m"] = _load(m, t)
        s["x"], s["dy"] = t["x"].requires_grad_(True), t["dy"]
    elif c["kind"] in ("norm", "head"):
        s.update(t)
        for n in ("x", "res", "w", "h"):
            if n in s:
                s[n].requires_grad_(True)
    else:
        from llattn_amd.lm import build_model
        with torch.device(DEVICE):
            m = build_model("0.55b", vocab_size=LM["vocab"], max_seq_len=LM["max_seq_len"])
        s["m"], s["ids"] = _load(m, t), t["ids"]
    return s


def _autocast(c):
    return torch.autocast(device_type="cuda", dtype=BF16, enabled=c.get("dtype", "bf16") == "bf16")


def _fresh(*tensors):
    for t in tensors:
        t.grad = None


def run(s):
    c = s["case"]
    k = c["kind"]
    if k in ("block", "ffn"):
        m, x = s["m"], s["x"]
        if k == "block" and not c["grad"]:
            with torch.no_grad(), _autocast(c):
                return [m(x)]
        params = list(m.parameters())
        _fresh(x, *params)
        with _autocast(c):
            y = m(x)
        y.backward(s["dy"])
        return [y.detach(), x.grad, *(p.grad for p in params)]
    if k == "op":
        from llattn_amd import LLAttnFunction
        ins = [s[n] for n in ("Q", "K", "V", "GQ", "GK", "GV", "gate_l", "gate_r", "r_w")]
        _fresh(*ins, s["r_b"])
        y = LLAttnFunction.apply(*ins, c["window"], c["chunk"], s["r_b"], c["local_block"], c["query_block"])
        y.backward(s["dO"])
        return [y.detach(), *(t.grad for t in ins), s["r_b"].grad]
    if k == "norm":
        from llattn_amd.norm import add_rms_norm
        _fresh(s["x"], s["res"], s["w"])
        with _autocast(c):
            total, y = add_rms_norm(s["x"], s["res"], s["w"], 1e-6)
        torch.autograd.backward([total, y], [s["ds"], s["dy"]])
        return [total.detach(), y.detach(), s["x"].grad, s["res"].grad, s["w"].grad]
    if k == "head":
        from llattn_amd.xent import lm_head_loss
        _fresh(s["h"], s["w"])
        with _autocast(c):
            loss, pred = lm_head_loss(s["h"], s["w"], s["targets"])
        loss.backward()
        return [loss.detach(), pred, s["h"].grad, s["w"].grad]
    with _autocast(c):
        return [s["m"].next_token_logits(s["ids"])]


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------

def _layout(T, window, local_block, latents, query_block):
    """(local block, chunk, chunks, query block, queries) of a sequence length."""
    chunk = -(-T // min(latents, T))
    qb = min(T, query_block) if query_block > 1 else 1
    return min(T, max(window, local_block)), chunk, -(-T // chunk), qb, -(-T // qb)


def _key_counts(T, window, bs, chunk, nc, qb, nq):
    i, s = torch.arange(T), torch.arange(nq)
    lo = torch.maximum((i - window).clamp(min=0), i // bs * bs - window + 1)
    return int((i - lo).clamp(min=0).sum()), int(torch.minimum(s * qb // chunk, torch.tensor(nc)).sum())


def _block_flops(c, latents):
    B, T, d, ld = c["B"], c["T"], c["d_model"], c["latent_dim"]
    bs, chunk, nc, qb, nq = _layout(T, c["window"], c["local_block"], latents, c["query_block"])
    keys, lats = _key_counts(T, c["window"], bs, chunk, nc, qb, nq)
    return B * (2 * T * d * 4 * d + 2 * nq * d * 2 * ld + 2 * nc * d * 2 * ld + 4 * keys * d + 4 * lats * ld + 4 * T * d)


def work(case):
    c, k = case, case["kind"]
    if k == "block":
        n, d, ld, es = c["B"] * c["T"], c["d_model"], c["latent_dim"], 4 if c["dtype"] == "fp32" else 2
        params = 4 * (4 * d * d + 4 * d * ld + 4 * d + 3 * ld + d + 2 * d // c["n_heads"])
        flops = _block_flops(c, c["latents"])
        if c["grad"]:
            return {"bytes": 4 * n * d * es + 2 * params, "flops": 3 * flops}
        return {"bytes": 2 * n * d * es + params, "flops": flops}
    if k == "op":
        es, n, hd, ld = 4 if c["dtype"] == "fp32" else 2, c["B"] * c["T"], c["H"] * c["Dh"], c["Lh"] * c["Ldh"]
        T, qb = c["T"], min(c["T"], c["query_block"]) if c["query_block"] > 1 else 1
        nq, nc = -(-T // qb), -(-T // c["chunk"])
        keys, lats = _key_counts(T, c["window"], min(T, max(c["window"], c["local_block"])), c["chunk"], nc, qb, nq)
        # q, k, v, dO, dq, dk, dv, out; latents and their gradients; r_out and its gradient
        b = 8 * n * hd * es + 2 * c["B"] * (nq + 2 * nc) * ld * es + 8 * hd * ld
        return {"bytes": b, "flops": 3 * c["B"] * (4 * keys * hd + 4 * lats * ld + 2 * nq * ld * hd + 4 * T * hd)}
    n, d = c["B"] * c["T"], c.get("d_model", LM["d_model"])
    if k == "ffn":
        return {"bytes": 8 * n * d + 16 * d * c["d_ff"], "flops": 12 * n * d * c["d_ff"]}
    if k == "norm":  # x, res, ds, dy read; sum, y, dx, dres written
        return {"bytes": n * d * (4 + 2 + 4 + 2 + 4 + 2 + 4 + 2), "flops": 16 * n * d}
    if k == "head":
        return {"bytes": 4 * n * d + 8 * c["vocab"] * d + 8 * n, "flops": 6 * n * d * c["vocab"]}
    blk = dict(ARCH["0.55b"], B=c["B"], T=c["T"], window=64, local_block=256, query_block=0)
    flops = LM["n_layers"] * (_block_flops(blk, 16) + 4 * n * d * LM["d_ff"]) + 2 * c["B"] * d * LM["vocab"]
    params = LM["n_layers"] * (4 * d * d + 4 * d * 512 + 2 * d * LM["d_ff"]) + LM["vocab"] * d
    return {"bytes": 4 * params + 2 * c["B"] * LM["vocab"], "flops": flops}


def tolerance(case):
    """About four times the largest error against ``exact`` that an output of the kind shows: 1.6e-6 in fp32, 6.5e-3
    for the gradients of a bf16 block or op, 4.3e-3 for the feed-forward's, 1.7e-3 (one bf16 rounding) for the norm's,
    2.6e-3 for the head's, 7.3e-3 for the logits of the whole model."""
    k = case["kind"]
    if k in ("block", "op"):
        return {"rel": 1e-5 if case["dtype"] == "fp32" else 0.025}
    if k == "head":
        return {"rel": 0.01, "differ": 0.01}
    return {"rel": {"ffn": 0.016, "norm": 0.007, "lm": 0.03}[k]}


# ---------------------------------------------------------------------------
# the same values in float64, from plain torch
# ---------------------------------------------------------------------------

def _masked_softmax(s, allowed):
    """Softmax over the allowed entries of the last dim; a row without any gives zeros."""
    s = s.masked_fill(~allowed, float("-inf"))
    some = allowed.any(-1, keepdim=True)
    return torch.softmax(torch.where(some, s, torch.zeros_like(s)), -1) * some


def _local64(q, k, v, window, bs):
    """Causal window attention of [B, H, T, Dh]: query i of the block that starts at a sees the keys j < i with
    j >= i - window and j > a - window."""
    T, outs = q.shape[2], []
    for a in range(0, T, bs):
        b, ka = min(a + bs, T), max(0, a - window + 1)
        i, j = torch.arange(a, b, device=q.device)[:, None], torch.arange(ka, b, device=q.device)[None]
        s = torch.matmul(q[:, :, a:b], k[:, :, ka:b].transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
        outs.append(torch.matmul(_masked_softmax(s, (j < i) & (j >= i - window)), v[:, :, ka:b]))
    return torch.cat(outs, 2)


def _core64(q, k, v, gq, gk, gv, gate_l, gate_r, r_w, r_b, window, bs, chunk, qb):
    """[B, T, H, Dh]: latent attention, its projection, local attention and the gate between the two."""
    B, H, T, Dh = q.shape
    nq, nc = gq.shape[2], gk.shape[2]
    see = torch.arange(nc, device=q.device)[None] < (torch.arange(nq, device=q.device) * qb // chunk)[:, None]
    s = torch.matmul(gq, gk.transpose(-1, -2).contiguous()) / math.sqrt(gq.shape[-1])
    lat = torch.matmul(_masked_softmax(s, see), gv).transpose(1, 2).reshape(B, nq, -1)
    remote = F.linear(lat, r_w, r_b)[:, torch.arange(T, device=q.device) // qb].view(B, T, H, Dh)
    local = _local64(q, k, v, window, bs).transpose(1, 2)
    g = torch.sigmoid((local * gate_l).sum(-1, keepdim=True) - (remote * gate_r).sum(-1, keepdim=True))
    return g * local + (1.0 - g) * remote


def _block64(p, x, n_heads, latent_heads, window, local_block, latents, query_block):
    B, T, D = x.shape
    bs, chunk, nc, qb, nq = _layout(T, window, local_block, latents, query_block)
    split = lambda t, n: t.view(B, t.shape[1], n, -1).transpose(1, 2)  # noqa: E731
    q, k, v = (split(t, n_heads) for t in F.linear(x, p["qkv_proj.weight"], p["qkv_proj.bias"]).chunk(3, -1))

    def segments(seg, n, counts):
        pad = F.pad(x, (0, 0, 0, n * seg - T)).view(B, n, seg, D).sum(2)
        return pad / counts

    real = torch.full((nc, 1), float(chunk), dtype=x.dtype, device=x.device)
    real[-1] = T - (nc - 1) * chunk
    gk, gv = (split(t, latent_heads)
              for t in F.linear(segments(chunk, nc, real), p["rkv_proj.weight"], p["rkv_proj.bias"]).chunk(2, -1))
    gq = split(F.linear(segments(qb, nq, float(qb)) if query_block > 1 else x, p["rq_proj.weight"], p["rq_proj.bias"]),
               latent_heads)
    y = _core64(q, k, v, gq, gk, gv, p["gate_local.weight"][0], p["gate_remote.weight"][0], p["r_out.weight"],
                p["r_out.bias"], window, bs, chunk, qb)
    return F.linear(y.reshape(B, T, D), p["out.weight"], p["out.bias"])


def _ffn64(p, x):
    return F.linear(F.gelu(F.linear(x, p["w1.weight"], p["w1.bias"])), p["w2.weight"], p["w2.bias"])


def _lm64(t, ids):
    a = ARCH["0.55b"]
    w = lambda n: t[n].to(F64)  # noqa: E731
    norm = lambda x, n: F.rms_norm(x, (x.shape[-1],), w(n), 1e-6)  # noqa: E731
    x = w("embedding.weight")[ids] + w("position.weight")[: ids.shape[1]]
    for i in range(LM["n_layers"]):
        pre = f"blocks.{i}."
        attn = {n[len(pre) + 5:]: v.to(F64) for n, v in t.items() if n.startswith(pre + "attn.")}
        ff = {n[len(pre) + 3:]: v.to(F64) for n, v in t.items() if n.startswith(pre + "ff.")}
        x = x + _block64(attn, norm(x, pre + "norm1.weight"), a["n_heads"], a["latent_heads"], 64, 256, 16, 0)
        x = x + _ffn64(ff, norm(x, pre + "norm2.weight"))
    return norm(x, "norm.weight")[:, -1] @ w("embedding.weight").t()


# the parameters in the order in which the modules hold them
_BLOCK_ORDER = [f"{n}.{k}" for n in ("qkv_proj", "rq_proj", "rkv_proj", "r_out", "out") for k in ("weight", "bias")] + \
    ["gate_local.weight", "gate_remote.weight"]
_FFN_ORDER = ["w1.weight", "w1.bias", "w2.weight", "w2.bias"]


def exact(case, seed):
    c, k, t = case, case["kind"], _inputs(case, seed)
    if k == "lm":
        with torch.no_grad():
            return [_lm64(t, t["ids"])]
    wide = {n: v.to(F64).requires_grad_(n not in ("dy", "dO", "ds")) for n, v in t.items() if v.is_floating_point()}
    if k == "block":
        with torch.set_grad_enabled(c["grad"]):
            y = _block64(wide, wide["x"], c["n_heads"], c["latent_heads"], c["window"], c["local_block"], c["latents"],
                         c["query_block"])
        if not c["grad"]:
            return [y]
        y.backward(wide["dy"])
        return [y.detach(), wide["x"].grad, *(wide[n].grad for n in _BLOCK_ORDER)]
    if k == "op":
        names = ("Q", "K", "V", "GQ", "GK", "GV", "gate_l", "gate_r", "r_w")
        qb = min(c["T"], c["query_block"]) if c["query_block"] > 1 else 1
        a = [wide[n] for n in names]
        y = _core64(*a, wide["r_b"], c["window"], min(c["T"], max(c["window"], c["local_block"])), c["chunk"],
                    qb).transpose(1, 2)
        y.backward(wide["dO"])
        return [y.detach(), *(v.grad for v in a), wide["r_b"].grad]
    if k == "ffn":
        y = _ffn64(wide, wide["x"])
        y.backward(wide["dy"])
        return [y.detach(), wide["x"].grad, *(wide[n].grad for n in _FFN_ORDER)]
    if k == "norm":
        total = wide["x"] + wide["res"]
        y = F.rms_norm(total, (c["d_model"],), wide["w"], 1e-6)
        torch.autograd.backward([total, y], [wide["ds"], wide["dy"]])
        return [total.detach(), y.detach(), wide["x"].grad, wide["res"].grad, wide["w"].grad]
    # head: loss and gradients; the predicted tokens have no float64 counterpart (ties of bf16 logits)
    logits = wide["h"].view(-1, c["d_model"]) @ wide["w"].t()
    loss = F.cross_entropy(logits, t["targets"].view(-1))
    loss.backward()
    return [loss.detach(), None, wide["h"].grad, wide["w"].grad]
