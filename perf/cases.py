"""The performance cases of this package: what a user's program has it do,
through the public entry points, over the sizes, types and directions that
are used in earnest.

A case is a dict of plain values; its "kind" names the path:

  ops    the fused element ops of `hydra_amd.kernels` (RMSNorm, QK-norm,
         RoPE, SwiGLU), forward and backward
  block  token embedding + HydraBlock, inference
  attn   the CCGQAAttention module: inference, or a training step
         (optionally of a padded batch)
  core   ccgqa_attention_fused on given q, k, v: a training step
  mod    Mixture-of-Depths routing around a pre-norm: top-k, gather,
         weighted residual scatter, forward and backward
  ce     the chunked LM-head cross-entropy, forward and backward
  model  HydraModel's logits

`listed()` holds the named cases, `draw(rng)` gives others of the same
ranges.  `exact()` restates each path in 64-bit torch.
"""
from __future__ import annotations

import math
import os

import torch
import torch.nn.functional as F

# Padded batches use key-padding semantics (a program that pads its batches
# sets this once at its start; calls without a mask do not look at it).
os.environ.setdefault("HYDRA_CCGQA_MASK_SEMANTICS", "key_padding")

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
GRAD = 0.02  # the incoming gradients' scale
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}

# (dim, n_heads, n_kv_heads) of attention layers at 4x compression: the debug
# shape (head_dim 16), the 250M one (64), the module's own default head counts
# at dim 1024 (16), the published timing's (64), the 1B model's (16), and the
# group sizes and head dims between them.
LAYERS = [(512, 8, 2), (1024, 4, 1), (1024, 16, 4), (2048, 8, 2), (1792, 28, 4), (768, 6, 2), (1024, 8, 8),
          (2048, 4, 1)]


def listed():
    return [
        # a short prompt's element ops: nothing but launches and latency
        dict(name="ops_small", kind="ops", dtype="bf16", B=1, S=61, dim=512, heads=8, kv_heads=2, head_dim=16,
             hidden=1365),
        # the element ops of one layer's training step at 16k tokens
        dict(name="ops_large", kind="ops", dtype="bf16", B=8, S=2048, dim=768, heads=12, kv_heads=4, head_dim=64,
             hidden=2048),
        # the debug-size block in fp32, where new models are brought up
        dict(name="block_fp32", kind="block", dtype="fp32", B=2, S=512, dim=512, heads=8, kv_heads=2, vocab=32000),
        # prefill of long sequences through one attention layer (250M model)
        dict(name="attn_infer_long", kind="attn", dtype="bf16", train=False, padded=False, B=4, S=4096, dim=1024,
             heads=4, kv_heads=1),
        # prefill of one prompt of any length (the module's default heads)
        dict(name="attn_infer_ragged", kind="attn", dtype="bf16", train=False, padded=False, B=1, S=1003, dim=1024,
             heads=16, kv_heads=4),
        # one attention layer's training step (the published timing's shape)
        dict(name="attn_train", kind="attn", dtype="bf16", train=True, padded=False, B=4, S=1024, dim=2048, heads=8,
             kv_heads=2),
        # the same for a batch of sequences of unequal length, padded
        dict(name="attn_train_padded", kind="attn", dtype="bf16", train=True, padded=True, B=8, S=777, dim=1024,
             heads=4, kv_heads=1),
        # the attention core alone, training, long sequences
        dict(name="core_bf16", kind="core", dtype="bf16", causal=True, B=4, heads=4, kv_heads=1, S=4096, head_dim=64),
        # the attention core of a program that trains in fp16
        dict(name="core_fp16", kind="core", dtype="fp16", causal=True, B=2, heads=8, kv_heads=2, S=1500, head_dim=64),
        # Mixture-of-Depths around a sublayer at 75% capacity (500M model)
        dict(name="mod_train", kind="mod", dtype="bf16", B=8, L=4096, dim=1280, capacity=0.75),
        # the LM head's loss over two chunks of tokens
        dict(name="ce_train", kind="ce", dtype="bf16", tokens=8192, dim=768, vocab=32000, ignored=0.1),
        # a whole forward: four blocks of the 1B model's width, every recursion
        dict(name="model_logits", kind="model", dtype="bf16", B=2, S=2048, dim=1792, heads=28, kv_heads=4, blocks=4,
             recursions=4, vocab=32000),
    ]


def _log_int(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["ops", "block", "attn", "attn", "core", "core", "mod", "ce", "model"])
    if kind == "ops":
        hd = rng.choice([16, 32, 64, 128])
        kv = rng.choice([1, 2, 4])
        S = _log_int(rng, 16, 4096)
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "fp32"]), B=max(1, min(8, 16384 // S)), S=S,
                    dim=rng.choice([512, 768, 1024, 1280, 1536, 1792]), heads=kv * rng.choice([1, 3, 4]), kv_heads=kv,
                    head_dim=hd, hidden=rng.choice([1365, 2048, 2560, 2816]))
    if kind == "block":
        dim, h, kv = rng.choice([(512, 8, 2), (512, 8, 4), (768, 12, 4), (768, 6, 2)])
        return dict(kind=kind, dtype=rng.choice(["fp32", "fp32", "bf16"]), B=rng.randint(1, 4), S=_log_int(rng, 32, 1024),
                    dim=dim, heads=h, kv_heads=kv, vocab=32000)
    if kind == "attn":
        dim, h, kv = rng.choice(LAYERS)
        train = rng.random() < 0.5
        S = _log_int(rng, 64, 4096)
        return dict(kind=kind, dtype="bf16", train=train, padded=train and rng.random() < 0.4,
                    B=rng.randint(1, max(1, min(8, 8192 // S))), S=S, dim=dim, heads=h, kv_heads=kv)
    if kind == "core":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        kv = rng.choice([1, 2, 4])
        S = _log_int(rng, 64, 4096 if dtype == "bf16" else 2048)
        return dict(kind=kind, dtype=dtype, causal=rng.random() < 0.8, B=rng.randint(1, max(1, min(4, 8192 // S))),
                    heads=kv * rng.choice([1, 2, 3, 4]), kv_heads=kv, S=S, head_dim=rng.choice([16, 32, 64, 64, 128]))
    if kind == "mod":
        L = _log_int(rng, 64, 12000)
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "fp32"]), B=max(1, min(8, 32768 // L)), L=L,
                    dim=rng.choice([512, 768, 1024, 1280]), capacity=rng.choice([0.125, 0.5, 0.75]))
    if kind == "ce":
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "fp32"]), tokens=_log_int(rng, 64, 6000),
                    dim=rng.choice([512, 640, 768]), vocab=rng.choice([4099, 16000, 32000]),
                    ignored=rng.choice([0.0, 0.1, 0.5]))
    dim, h, kv = rng.choice([(512, 8, 2), (768, 12, 4), (1024, 16, 4), (1792, 28, 4)])
    S = _log_int(rng, 64, 2048)
    return dict(kind="model", dtype="bf16", B=rng.randint(1, max(1, min(4, 3072 // S))), S=S, dim=dim, heads=h,
                kv_heads=kv, blocks=rng.randint(2, 4), recursions=rng.randint(2, 4), vocab=rng.choice([16000, 32000]))


# ------------------------------------------------------------------ inputs
class _Random:
    """Inputs on the GPU from a seed alone."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float32, grad=False):
        t = torch.randn(*shape, generator=self.g, device="cuda").mul_(std).add_(mean).to(dtype)
        return t.requires_grad_(grad)

    def ints(self, hi, *shape, lo=0):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda")

    def fill(self, module, dtype, std=0.02):
        """N(0, std) weights, N(1, 0.1) norm gains, N(0, 0.1) biases; the key
        temperature of the QK-norm keeps its initial value."""
        module = module.to(dtype)
        with torch.no_grad():
            for name, p in module.named_parameters():
                if "key_temperature" in name:
                    continue
                if "norm" in name:
                    p.copy_(self.normal(*p.shape, std=0.1, mean=1.0))
                elif name.endswith("bias"):
                    p.copy_(self.normal(*p.shape, std=0.1))
                else:
                    p.copy_(self.normal(*p.shape, std=std))
        return module


def _rope_tables(head_dim, length):
    """cos, sin [length, head_dim/2] fp32 of angles taken in fp32 (theta 1e4)."""
    freqs = 1.0 / (10000.0 ** (torch.arange(0, head_dim, 2, dtype=torch.float32) / head_dim))
    ang = torch.outer(torch.arange(length, dtype=torch.float32), freqs)
    return ang.cos().cuda(), ang.sin().cuda()


def _mlp_hidden(dim, ratio=2.67):
    return (int(dim * ratio) + 255) // 256 * 256


def prepare(case, seed):
    r, dt, kind = _Random(seed), DTYPES[case["dtype"]], case["kind"]
    s = {"case": case}
    if kind == "ops":
        B, S, dim, hd, hid = case["B"], case["S"], case["dim"], case["head_dim"], case["hidden"]
        H, K = case["heads"], case["kv_heads"]
        s["ins"] = [r.normal(B, S, dim, dtype=dt, grad=True), r.normal(dim, std=0.1, mean=1.0, dtype=dt, grad=True),
                    r.normal(B, H, S, hd, dtype=dt, grad=True), r.normal(B, K, S, hd, dtype=dt, grad=True),
                    r.normal(B, H, S, hd, dtype=dt, grad=True), r.normal(B, S, 2 * hid, dtype=dt, grad=True)]
        s["rope"] = _rope_tables(hd, S)
        s["grads"] = [r.normal(*shape, std=GRAD, dtype=dt) for shape in
                      ((B, S, dim), (B, H, S, hd), (B, K, S, hd), (B, H, S, hd), (B, S, hid))]
    elif kind == "block":
        from hydra_amd.model.framework import HydraBlock
        with torch.device("cuda"):
            block = HydraBlock(case["dim"], n_heads=case["heads"], n_kv_heads=case["kv_heads"], max_seq_len=1024)
        s["block"] = r.fill(block, dt).eval()
        s["table"] = r.normal(case["vocab"], case["dim"], std=0.02, dtype=dt)
        s["ids"] = r.ints(case["vocab"], case["B"], case["S"])
    elif kind == "attn":
        from hydra_amd.attention import CCGQAAttention
        B, S = case["B"], case["S"]
        with torch.device("cuda"):
            layer = CCGQAAttention(case["dim"], n_heads=case["heads"], n_kv_heads=case["kv_heads"], max_seq_len=4096)
        s["layer"] = r.fill(layer, dt).train(case["train"])
        s["x"] = r.normal(B, S, case["dim"], dtype=dt, grad=case["train"])
        s["mask"] = None
        if case["padded"]:  # right-padded: sequences of half the length or more
            length = r.ints(S + 1, B, 1, lo=(S + 1) // 2)
            length[0] = S
            s["mask"] = (torch.arange(S, device="cuda") < length).long()
        if case["train"]:
            s["gout"] = r.normal(B, S, case["dim"], std=GRAD, dtype=dt)
            if s["mask"] is not None:
                s["gout"] *= s["mask"][..., None].to(dt)  # no loss on padding
    elif kind == "core":
        B, H, K, S, hd = (case[n] for n in ("B", "heads", "kv_heads", "S", "head_dim"))
        s["ins"] = [r.normal(B, h, S, hd, dtype=dt, grad=True) for h in (H, K, K)]
        s["gout"] = r.normal(B, H, S, hd, std=GRAD, dtype=dt)
    elif kind == "mod":
        from hydra_amd.routing import router_k
        B, L, dim = case["B"], case["L"], case["dim"]
        scores = r.normal(B, L)
        dup = r.normal(B, L).argsort(1)[:, :L // 20]  # 5% of the entries repeat another one
        s["scores"] = scores.scatter(1, dup, scores.gather(1, r.ints(L, B, L // 20)))
        s["k"] = router_k(L, case["capacity"])
        s["x"] = r.normal(B, L, dim, dtype=dt, grad=True)
        s["gain"] = r.normal(dim, std=0.1, mean=1.0, dtype=dt, grad=True)
        s["weights"] = torch.sigmoid(r.normal(B, s["k"])).requires_grad_()
        s["gout"] = r.normal(B, L, dim, std=GRAD, dtype=dt)
    elif kind == "ce":
        n = case["tokens"]
        s["h"] = r.normal(n, case["dim"], dtype=dt, grad=True)
        s["w"] = r.normal(case["vocab"], case["dim"], std=0.02, dtype=dt, grad=True)
        t = r.ints(case["vocab"], n)
        t[r.normal(n).sigmoid() < case["ignored"]] = -100
        s["t"] = t
    else:
        from hydra_amd.model.framework import HydraModel
        with torch.device("cuda"):
            model = HydraModel(vocab_size=case["vocab"], dim=case["dim"], n_mor_blocks=case["blocks"],
                               recursions_per_block=case["recursions"], n_heads=case["heads"],
                               n_kv_heads=case["kv_heads"], max_seq_len=2048, adaptive=False)
        s["model"] = r.fill(model, dt).eval()
        with torch.no_grad():  # the model's own scale of the residual branches
            for name, p in model.named_parameters():
                if "o_proj" in name or "down" in name:
                    p.mul_(1.0 / math.sqrt(2 * model.effective_layers))
        s["ids"] = r.ints(case["vocab"], case["B"], case["S"])
    return s


# --------------------------------------------------------------- one pass
def _attn_grads(layer):
    """The layer's parameters whose gradients a step returns, and how they are
    laid out: the k conv's and the temperature's (one value) together."""
    return [layer.qkv_proj.weight, layer.o_proj.weight, layer.q_conv.conv1.weight, layer.q_conv.conv2.weight,
            layer.k_conv.conv1.weight, layer.k_conv.conv2.weight, layer.key_temperature]


def _with_attn_grads(out, grads):
    return {"out": out.detach(), "x": grads[0], "qkv": grads[1], "o": grads[2], "q1": grads[3], "q2": grads[4],
            "k": torch.cat([g.reshape(-1) for g in grads[5:]])}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "ops":
        from hydra_amd.kernels import fused_qk_norm, fused_rms_norm, fused_rope, fused_swiglu
        x, w, q, k, xr, gate_up = s["ins"]
        y = fused_rms_norm(x, w)
        qn, kn = fused_qk_norm(q, k, 1.0, math.sqrt(case["head_dim"]))
        rot = fused_rope(xr, *s["rope"])
        gate, up = gate_up.chunk(2, dim=-1)
        outs = [y, qn, kn, rot, fused_swiglu(gate, up)]
        grads = torch.autograd.grad(outs, s["ins"], s["grads"])
        return [o.detach() for o in outs], list(grads)
    if kind == "block":
        from hydra_amd.model.framework import embedding_lookup
        with torch.no_grad():
            return s["block"](embedding_lookup(s["table"], s["ids"], math.sqrt(case["dim"])))
    if kind == "attn":
        if not case["train"]:
            with torch.no_grad():
                return s["layer"](s["x"])
        out = s["layer"](s["x"], mask=s["mask"])
        return _with_attn_grads(out, torch.autograd.grad(out, [s["x"]] + _attn_grads(s["layer"]), s["gout"]))
    if kind == "core":
        from hydra_amd.attention.backends.ccgqa.kernels import ccgqa_attention_fused
        out = ccgqa_attention_fused(*s["ins"], is_causal=case["causal"])
        return [out.detach(), *torch.autograd.grad(out, s["ins"], s["gout"])]
    if kind == "mod":
        from hydra_amd.kernels import fused_rms_norm
        from hydra_amd.routing import gather_by_indices, mod_topk, weighted_residual_scatter
        x = s["x"]
        desc, srt, mask = mod_topk(s["scores"], s["k"], mask_dtype=x.dtype)
        y = fused_rms_norm(gather_by_indices(x, srt, distinct=True), s["gain"])
        out = weighted_residual_scatter(x.clone(), y, srt, s["weights"])
        grads = torch.autograd.grad(out, [x, s["gain"], s["weights"]], s["gout"])
        return [desc, srt, mask, out.detach(), *grads]
    if kind == "ce":
        from hydra_amd.kernels import fused_chunked_cross_entropy
        loss = fused_chunked_cross_entropy(s["h"], s["w"], s["t"])
        return [loss.detach(), *torch.autograd.grad(loss, [s["h"], s["w"]])]
    with torch.no_grad():
        return s["model"](s["ids"])


# ------------------------------------------------------ what a pass needs
def _layer_work(B, S, dim, H, K, e):
    """(flops, weight bytes, activation bytes) of one attention layer forward."""
    n, L = B * S, dim // 4
    hd = L // H
    kv = K * hd
    macs = n * dim * (L + 2 * kv) + 3 * n * (L * hd + L * L + kv * hd + kv * kv) + n * L * dim
    core = 2 * B * H * hd * S * (S + 1) // 2
    weights = dim * (L + 2 * kv) + 3 * (L * hd + L * L + kv * hd + kv * kv) + L * dim
    return 2 * (macs + core), e * weights, e * 2 * n * dim


def work(case):
    kind, e = case["kind"], SIZE[case["dtype"]]
    if kind == "ops":
        n = case["B"] * case["S"]
        elems = n * case["dim"] + n * case["head_dim"] * (2 * case["heads"] + case["kv_heads"])
        # one value in and one out forward, one more of each backward; SwiGLU: gate, up and the gradient in
        hid = n * case["hidden"]
        return {"bytes": e * (4 * elems + (2 + 1 + 1 + 2) * hid), "flops": 24 * elems + 20 * hid}
    if kind == "block":
        n, dim, hidden = case["B"] * case["S"], case["dim"], _mlp_hidden(case["dim"])
        f, wb, ab = _layer_work(case["B"], case["S"], dim, case["heads"], case["kv_heads"], e)
        return {"bytes": wb + e * (3 * dim * hidden + 2 * n * dim), "flops": f + 2 * n * 3 * dim * hidden}
    if kind == "attn":
        f, wb, ab = _layer_work(case["B"], case["S"], case["dim"], case["heads"], case["kv_heads"], e)
        if not case["train"]:
            return {"bytes": wb + ab, "flops": f}
        return {"bytes": 2 * wb + 2 * ab, "flops": 3 * f}
    if kind == "core":
        B, H, K, S, hd = (case[n] for n in ("B", "heads", "kv_heads", "S", "head_dim"))
        pairs = B * H * (S * (S + 1) // 2 if case["causal"] else S * S)
        # forward two products of each visible pair, backward five
        return {"bytes": e * 2 * B * S * hd * (2 * H + 2 * K), "flops": 14 * pairs * hd}
    if kind == "mod":
        n, k = case["B"] * case["L"], case["B"] * max(1, int(case["L"] * case["capacity"]))
        # x, grad_out in, out, grad_x out; scores, mask, both index lists
        return {"bytes": e * 4 * n * case["dim"] + n * (4 + e) + 16 * k, "flops": 20 * k * case["dim"]}
    if kind == "ce":
        n, V, d = case["tokens"], case["vocab"], case["dim"]
        return {"bytes": e * 2 * (n + V) * d, "flops": 6 * n * V * d}
    n, dim, hidden = case["B"] * case["S"], case["dim"], _mlp_hidden(case["dim"])
    f, wb, ab = _layer_work(case["B"], case["S"], dim, case["heads"], case["kv_heads"], e)
    mlp = 2 * n * 3 * dim * hidden * case["recursions"]
    return {"bytes": case["blocks"] * (wb + e * 3 * dim * hidden) + e * case["vocab"] * (dim + n),
            "flops": case["blocks"] * (f + mlp) + 2 * n * dim * case["vocab"]}


# ------------------------------------------------------------- tolerances
# Relative 2-norm errors that another order of the sums shows at the same
# precision, times about four (measured against exact()).
_TOL = {
    ("ops", "bf16"): 8e-3, ("ops", "fp32"): 4e-6,
    ("block", "fp32"): 5e-6, ("block", "bf16"): 2e-2,
    ("core", "bf16"): 1.2e-2, ("core", "fp16"): 1.2e-3, ("core", "fp32"): 5e-6,
    ("mod", "bf16"): 8e-3, ("mod", "fp32"): 4e-6,
    ("ce", "bf16"): 8e-3, ("ce", "fp32"): 1e-5,
    ("model", "bf16"): 3e-2,
}


def tolerance(case):
    if case["kind"] == "attn":
        return {"rel": 2.5e-2 if case["train"] else 1.5e-2}
    return {"rel": _TOL[case["kind"], case["dtype"]]}


# ------------------------------------------------------- in 64 bits
def _rms(x, w, eps=1e-6):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _rotate(x, cos, sin):
    """x [..., S, hd] on interleaved pairs."""
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)


def _attend(q, k, v, causal, mask=None):
    B, H, S, hd = q.shape
    g = H // k.shape[1]
    outs = []
    for b in range(B):  # one sequence's scores at a time
        sc = q[b] @ k[b].repeat_interleave(g, 0).transpose(-1, -2) * hd ** -0.5
        if causal:
            sc = sc.masked_fill(torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1), -math.inf)
        if mask is not None:
            sc = sc.masked_fill(mask[b] == 0, -math.inf)
        outs.append(torch.softmax(sc, -1) @ v[b].repeat_interleave(g, 0))
    return torch.stack(outs)


def _conv(x, w, groups):
    """Causal conv of x [B, S, C] with w [C, C/groups, taps]."""
    B, S, C = x.shape
    taps = w.shape[-1]
    xp = F.pad(x, (0, 0, taps - 1, 0)).view(B, S + taps - 1, groups, C // groups)
    wg = w.view(groups, C // groups, C // groups, taps)
    y = 0
    for t in range(taps):
        xs = xp[:, t:t + S].reshape(B * S, groups, C // groups).transpose(0, 1)
        y = y + xs @ wg[..., t].transpose(1, 2)
    return y.transpose(0, 1).reshape(B, S, C)


def _ccgqa(p, x, H, K, mask=None):
    """The CCGQA layer from its parameters p (by name) and x."""
    B, S, dim = x.shape
    L = dim // 4
    hd = L // H
    kv = K * hd
    qkv = x @ p["qkv_proj.weight"].t()
    q0, k0, vc, vp = qkv.split([L, kv, kv // 2, kv - kv // 2], -1)
    v = torch.cat([vc, F.pad(vp, (0, 0, 1, 0))[:, :S]], -1)
    q = _conv(_conv(q0, p["q_conv.conv1.weight"], H), p["q_conv.conv2.weight"], 1).view(B, S, H, hd)
    k = _conv(_conv(k0, p["k_conv.conv1.weight"], K), p["k_conv.conv2.weight"], 1).view(B, S, K, hd)
    q0, k0 = q0.reshape(B, S, H, hd), k0.reshape(B, S, K, hd)
    if H == K:
        q, k = q + 0.5 * (q0 + k0), k + 0.5 * (q0 + k0)
    else:
        q, k = q + 0.5 * k0.mean(2, keepdim=True), k + 0.5 * q0.mean(2, keepdim=True)
    q, k, v = (t.transpose(1, 2) for t in (q, k, v.view(B, S, K, hd)))
    q = F.normalize(q, dim=-1)
    k = F.normalize(k, dim=-1) * p["key_temperature"]
    cos, sin = (t.double() for t in _rope_tables(hd, S))
    o = _attend(_rotate(q, cos, sin), _rotate(k, cos, sin), v, True, mask)
    return o.transpose(1, 2).reshape(B, S, L) @ p["o_proj.weight"].t()


def _swiglu_mlp(x, w_in, w_out):
    g, u = (x @ w_in.t()).chunk(2, -1)
    return (F.silu(g) * u) @ w_out.t()


def _params(module, prefix=""):
    return {n[len(prefix):]: t.detach().double() for n, t in module.named_parameters() if n.startswith(prefix)}


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    leaf = lambda t: t.detach().double().requires_grad_()  # noqa: E731
    if kind == "ops":
        ins = [leaf(t) for t in s["ins"]]
        x, w, q, k, xr, gate_up = ins
        unit = lambda t: t * torch.rsqrt(t.pow(2).sum(-1, keepdim=True) + 1e-8)  # noqa: E731
        g, u = gate_up.chunk(2, -1)
        outs = [_rms(x, w), unit(q), unit(k) * math.sqrt(case["head_dim"]),
                _rotate(xr, *(t.double() for t in s["rope"])), F.silu(g) * u]
        grads = torch.autograd.grad(outs, ins, [t.double() for t in s["grads"]])
        return [o.detach() for o in outs], list(grads)
    if kind == "block":
        p = _params(s["block"])
        h = s["table"].double()[s["ids"]] * math.sqrt(case["dim"])
        att = {n[len("attention."):]: t for n, t in p.items() if n.startswith("attention.")}
        h = h + _ccgqa(att, _rms(h, p["norm1.weight"]), case["heads"], case["kv_heads"])
        return h + _swiglu_mlp(_rms(h, p["norm2.weight"]), p["mlp.gate_up.weight"], p["mlp.down.weight"])
    if kind == "attn":
        p, x = _params(s["layer"]), s["x"].detach().double()
        if not case["train"]:
            return _ccgqa(p, x, case["heads"], case["kv_heads"])
        for t in p.values():
            t.requires_grad_()
        x.requires_grad_()
        out = _ccgqa(p, x, case["heads"], case["kv_heads"], s["mask"])
        wrt = [x] + [p[n] for n in ("qkv_proj.weight", "o_proj.weight", "q_conv.conv1.weight", "q_conv.conv2.weight",
                                    "k_conv.conv1.weight", "k_conv.conv2.weight", "key_temperature")]
        return _with_attn_grads(out, torch.autograd.grad(out, wrt, s["gout"].double()))
    if kind == "core":
        ins = [leaf(t) for t in s["ins"]]
        out = _attend(*ins, case["causal"])
        return [out.detach(), *torch.autograd.grad(out, ins, s["gout"].double())]
    if kind == "mod":
        x, gain, weights = leaf(s["x"]), leaf(s["gain"]), leaf(s["weights"])
        order = torch.sort(s["scores"], dim=1, descending=True, stable=True).indices[:, :s["k"]]
        srt = order.sort(1).values
        at = srt[..., None].expand(-1, -1, case["dim"])
        y = _rms(x.gather(1, at), gain) * weights[..., None]
        out = x.scatter_add(1, at, y)
        grads = torch.autograd.grad(out, [x, gain, weights], s["gout"].double())
        mask = torch.zeros_like(s["scores"]).scatter_(1, srt, 1.0)
        return [order, srt, mask.double(), out.detach(), *grads]
    if kind == "ce":
        h, w = leaf(s["h"]), leaf(s["w"])
        loss = F.cross_entropy(h @ w.t(), s["t"], ignore_index=-100)
        return [loss.detach(), *torch.autograd.grad(loss, [h, w])]
    p = _params(s["model"])
    with torch.no_grad():
        h = p["tok_emb.weight"][s["ids"]] * math.sqrt(case["dim"])
        for i in range(case["blocks"]):
            b = {n[len("layers.%d." % i):]: t for n, t in p.items() if n.startswith("layers.%d." % i)}
            att = {n[len("attention."):]: t for n, t in b.items() if n.startswith("attention.")}
            h = h + 0.5 * _ccgqa(att, _rms(h, b["norm1.weight"]), case["heads"], case["kv_heads"])
            for j in range(case["recursions"]):
                z = h + b["mor_executor.recursion_bias"][j].view(-1) + b["mor_executor.recursion_embed.weight"][j]
                h = h + _swiglu_mlp(_rms(z, b["norm2.weight"]), b["mlp.gate_up.weight"], b["mlp.down.weight"])
            h = _rms(h, b["final_norm.weight"])
        return _rms(h, p["norm.weight"]) @ p["tok_emb.weight"].t()
