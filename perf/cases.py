"""The work that is timed: one call each of the operators that a robotics policy or a small
language model runs under this library, and one whole action-expert block.

``listed()`` names twelve cases; ``draw`` gives further ones of the same ranges.  Sizes are those
of the repository's configurations, tests and benchmark (action-expert widths 2048 / 8192, 16
query and 4 key/value heads of 128, 64 experts of width 768, 32 packed sequences), the published
operator shapes beside them, or generic ones.
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                        "robotics-batch-invariant-ops_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import batch_invariant_ops as bio  # noqa: E402
from model_invariance.adapters.synthetic_vla import SyntheticVLAAdapter  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # one token of one request through the MLP's first linear: the smallest call, bound by
        # latency and by streaming the weights
        dict(name="linear_decode", kind="linear", dtype="bf16", rows=1, k=2048, n=8192, bias=True),
        # a batch of eight prefixes of 246 tokens through a wide down projection
        dict(name="linear_prefill", kind="linear", dtype="bf16", rows=8 * 246, k=6144, n=2048, bias=False),
        # a float32 policy head's matrix product, row-major weights
        dict(name="mm_fp32", kind="mm", dtype="fp32", m=408, k=768, n=4096),
        # log-probabilities of a decoding batch over a vocabulary of odd size
        dict(name="log_softmax_vocab", kind="rows", op="log_softmax", dtype="fp32", rows=32, cols=50257),
        # causal prefill of a batch, grouped-query heads
        dict(name="sdpa_prefill", kind="sdpa", dtype="bf16", batch=8, hq=16, hkv=4, lq=1024, lk=1024, d=128,
             mode="causal"),
        # one decoding step of a batch against its key/value cache
        dict(name="sdpa_decode", kind="sdpa", dtype="bf16", batch=8, hq=16, hkv=4, lq=1, lk=2048, d=128,
             mode="full"),
        # vision-encoder attention in float32, head size off the powers of two
        dict(name="sdpa_fp32", kind="sdpa", dtype="fp32", batch=8, hq=16, hkv=16, lq=256, lk=256, d=72,
             mode="full"),
        # a packed batch of 32 sequences of 64 to 2048 tokens
        dict(name="varlen_prefill", kind="varlen", dtype="bf16", seqs=32, shortest=64, longest=2048, hq=8, hkv=2,
             d=64, causal=True),
        # expert layer of a decoding batch
        dict(name="moe_decode", kind="moe", dtype="bf16", tokens=16, hidden=2048, inter=768, experts=64, top_k=8),
        # expert layer of a prefill: the largest call
        dict(name="moe_prefill", kind="moe", dtype="bf16", tokens=4096, hidden=2048, inter=768, experts=64,
             top_k=8),
        # patch embedding of a batch of camera images
        dict(name="conv_patches", kind="conv", dtype="bf16", batch=16, cin=3, size=224, cout=1024, ksize=14,
             stride=14, padding=0),
        # a whole action-expert block under the mode: linears, norms, attention, experts, head
        dict(name="policy_block", kind="block", dtype="bf16", batch=4, tokens=256),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    """One more case: every kind equally often, sizes over the logarithm of its range."""
    kind = rng.choice(["linear", "linear", "mm", "rows", "sdpa", "sdpa", "step", "step", "varlen", "moe", "moe",
                       "conv", "block"])
    if kind == "linear":
        k, n = rng.choice([(2048, 8192), (8192, 2048), (6144, 2048),
                           (_log_int(rng, 512, 8192) // 8 * 8, _log_int(rng, 512, 8192)),
                           (_log_int(rng, 512, 8192), _log_int(rng, 512, 8192) // 8 * 8)])
        return dict(kind="linear", dtype=rng.choice(["bf16", "bf16", "fp16"]), rows=_log_int(rng, 1, 4096), k=k, n=n,
                    bias=rng.random() < 0.5)
    if kind == "mm":
        return dict(kind="mm", dtype="fp32", m=_log_int(rng, 1, 2048), k=_log_int(rng, 64, 4096),
                    n=_log_int(rng, 64, 4096))
    if kind == "rows":
        cols = _log_int(rng, 64, 131072)
        return dict(kind="rows", op=rng.choice(["softmax", "log_softmax", "mean", "l2_norm"]),
                    dtype=rng.choice(["bf16", "fp32"]), rows=_log_int(rng, 1, max(2, (1 << 25) // cols)), cols=cols)
    if kind == "sdpa":  # prefill and encoder attention
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        hkv = rng.choice([1, 2, 4, 8])
        d = rng.choice([64, 72, 80, 128, 128]) if dtype == "fp32" else rng.choice([64, 72, 128, 128, 256])
        lq = _log_int(rng, 65, 1536)
        mode = rng.choice(["causal", "full", "bool", "add"])
        lk = lq if mode == "causal" else lq + rng.choice([0, 0, rng.randint(1, 512)])
        return dict(kind="sdpa", dtype=dtype, batch=rng.randint(1, 4), hq=hkv * rng.choice([1, 2, 4]), hkv=hkv, lq=lq,
                    lk=lk, d=d, mode=mode)
    if kind == "step":  # decoding steps and short action chunks against a cache
        hkv = rng.choice([1, 2, 4, 8])
        return dict(kind="sdpa", dtype=rng.choice(["bf16", "bf16", "fp16"]), batch=_log_int(rng, 1, 16),
                    hq=hkv * rng.choice([1, 2, 4, 8]), hkv=hkv, lq=rng.choice([1, 1, _log_int(rng, 1, 64)]),
                    lk=_log_int(rng, 64, 4096), d=rng.choice([64, 128, 128, 256]),
                    mode=rng.choice(["full", "full", "bool"]))
    if kind == "varlen":
        hkv = rng.choice([1, 2, 4, 8])
        return dict(kind="varlen", dtype=rng.choice(["bf16", "bf16", "fp16"]), seqs=_log_int(rng, 1, 32),
                    shortest=rng.choice([1, 64]), longest=_log_int(rng, 96, 2048), hq=hkv * rng.choice([1, 2, 4]),
                    hkv=hkv, d=rng.choice([64, 128]), causal=rng.random() < 0.75)
    if kind == "moe":
        if rng.random() < 0.25:
            return dict(kind="moe", dtype="fp32", tokens=_log_int(rng, 1, 512), hidden=768, inter=512, experts=32,
                        top_k=4)
        return dict(kind="moe", dtype="bf16", tokens=_log_int(rng, 1, 4096), hidden=2048, inter=768, experts=64,
                    top_k=8)
    if kind == "conv":
        if rng.random() < 0.5:
            patch = rng.choice([14, 16])
            return dict(kind="conv", dtype=rng.choice(["bf16", "fp32"]), batch=_log_int(rng, 1, 16), cin=3,
                        size=patch * rng.randint(8, 24), cout=rng.choice([384, 768, 1024]), ksize=patch, stride=patch,
                        padding=0)
        return dict(kind="conv", dtype=rng.choice(["bf16", "fp32"]), batch=_log_int(rng, 1, 8),
                    cin=rng.choice([16, 48, 64, 128]), size=rng.randint(15, 64), cout=rng.choice([32, 64, 128]),
                    ksize=3, stride=rng.choice([1, 2]), padding=1)
    return dict(kind="block", dtype="bf16", batch=rng.randint(1, 6), tokens=rng.randint(32, 256))


# ------------------------------------------------------------------------------ inputs ----
def _inputs(case, seed):
    """The operands of ``case``, made on the GPU from ``seed`` alone, with stock operators."""
    bio.disable_batch_invariant_mode()
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, dtype = case["kind"], _DTYPES[case["dtype"]]

    def normal(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)

    if kind == "linear":
        return dict(x=normal(1, case["rows"], case["k"]), w=normal(case["n"], case["k"], scale=0.02),
                    b=normal(case["n"], scale=0.02) if case["bias"] else None)
    if kind == "mm":
        return dict(a=normal(case["m"], case["k"]), b=normal(case["k"], case["n"], scale=0.02))
    if kind == "rows":
        return dict(x=normal(case["rows"], case["cols"], scale=3.0))
    if kind == "sdpa":
        b, hq, hkv, lq, lk, d = (case[x] for x in ("batch", "hq", "hkv", "lq", "lk", "d"))
        mask = None
        if case["mode"] == "bool":  # key padding: every sample's own number of visible keys
            seen = torch.randint(max(1, lk // 2), lk + 1, (b, 1, 1, 1), generator=g, device="cuda")
            mask = torch.arange(lk, device="cuda").view(1, 1, 1, lk) < seen
        elif case["mode"] == "add":
            mask = -10.0 * torch.rand(b, 1, lq, lk, generator=g, device="cuda")
            mask = mask.masked_fill(torch.rand(b, 1, lq, lk, generator=g, device="cuda") < 0.1, -math.inf).to(dtype)
        return dict(q=normal(b, hq, lq, d), k=normal(b, hkv, lk, d), v=normal(b, hkv, lk, d), mask=mask)
    if kind == "varlen":
        lengths = torch.randint(case["shortest"], case["longest"] + 1, (case["seqs"],),
                                generator=torch.Generator().manual_seed(4))
        offsets = torch.zeros(case["seqs"] + 1, dtype=torch.int32)
        offsets[1:] = lengths.cumsum(0)
        total, d = int(offsets[-1]), case["d"]
        return dict(q=normal(1, total, case["hq"], d), k=normal(1, total, case["hkv"], d),
                    v=normal(1, total, case["hkv"], d), offsets=offsets.cuda())
    if kind == "moe":
        e, h, i = case["experts"], case["hidden"], case["inter"]
        gate_up = normal(e, h, 2 * i, scale=0.02)
        down = normal(e, i, h, scale=0.02)
        logits = torch.randn(case["tokens"], e, generator=g, device="cuda")
        weights, chosen = torch.topk(torch.softmax(logits, dim=-1), case["top_k"], dim=-1)
        return dict(x=normal(case["tokens"], h), weights=weights, chosen=chosen,
                    gate=gate_up[..., :i].transpose(1, 2), up=gate_up[..., i:].transpose(1, 2),
                    down=down.transpose(1, 2))
    if kind == "conv":
        fan = case["cin"] * case["ksize"] ** 2
        return dict(x=normal(case["batch"], case["cin"], case["size"], case["size"]),
                    w=normal(case["cout"], case["cin"], case["ksize"], case["ksize"], scale=fan ** -0.5),
                    b=normal(case["cout"], scale=0.1))
    return dict(x=normal(case["batch"], case["tokens"], 2048))


def prepare(case, seed):
    state = dict(case=case, **_inputs(case, seed))
    if case["kind"] == "block":
        adapter = SyntheticVLAAdapter.preset("vla", tokens=case["tokens"])
        state["adapter"], state["model"] = adapter, adapter.load_model()
    return state


# -------------------------------------------------------------------------------- calls ----
_ROW_OPS = {
    "softmax": lambda x: bio.softmax(x, -1),
    "log_softmax": lambda x: bio.log_softmax(x, -1),
    "mean": lambda x: bio.mean_dim(x, -1),
    "l2_norm": lambda x: bio.linalg_vector_norm_batch_invariant(x, 2, -1),
}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return bio.linear_batch_invariant(state["x"], state["w"], state["b"])
    if kind == "mm":
        return bio.matmul_persistent(state["a"], state["b"])
    if kind == "rows":
        return _ROW_OPS[case["op"]](state["x"])
    if kind == "sdpa":
        return bio.scaled_dot_product_attention_batch_invariant(
            state["q"], state["k"], state["v"], state["mask"], is_causal=case["mode"] == "causal",
            enable_gqa=case["hq"] != case["hkv"])
    if kind == "varlen":
        return bio.varlen_scaled_dot_product_attention_batch_invariant(
            state["q"], state["k"], state["v"], state["offsets"], state["offsets"], is_causal=case["causal"],
            causal_type="BottomRight")
    if kind == "moe":
        return bio.deterministic_token_choice_moe(state["x"], state["weights"], state["chosen"], state["gate"],
                                                  state["up"], state["down"])
    if kind == "conv":
        s, p = case["stride"], case["padding"]
        return bio.conv2d_batch_invariant(state["x"], state["w"], state["b"], (s, s), (p, p), (1, 1), False, (0, 0), 1)
    # a program that serves a policy turns the mode on once and leaves it on
    bio.enable_batch_invariant_mode()
    return state["adapter"].run_model(state["model"], {"x": state["x"]})


# --------------------------------------------------------------------- necessary work ----
def _visible(lq, lk, causal):
    return lq * (lq + 1) // 2 if causal else lq * lk


def work(case):
    kind, e = case["kind"], _BYTES[case["dtype"]]
    if kind == "linear":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": e * (m * k + k * n + m * n + (n if case["bias"] else 0)), "flops": 2 * m * k * n}
    if kind == "mm":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": e * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    if kind == "rows":
        r, c = case["rows"], case["cols"]
        whole = case["op"] in ("softmax", "log_softmax")
        return {"bytes": e * r * (2 * c if whole else c + 1), "flops": r * c * (5 if whole else 2)}
    if kind == "sdpa":
        b, hq, hkv, lq, lk, d = (case[x] for x in ("batch", "hq", "hkv", "lq", "lk", "d"))
        mask = {"bool": b * lk, "add": e * b * lq * lk}.get(case["mode"], 0)
        return {"bytes": e * b * d * (2 * hq * lq + 2 * hkv * lk) + mask,
                "flops": 4 * b * hq * d * _visible(lq, lk, case["mode"] == "causal")}
    if kind == "varlen":
        lengths = torch.randint(case["shortest"], case["longest"] + 1, (case["seqs"],),
                                generator=torch.Generator().manual_seed(4)).tolist()
        pairs = sum(_visible(n, n, case["causal"]) for n in lengths)
        return {"bytes": e * sum(lengths) * case["d"] * (2 * case["hq"] + 2 * case["hkv"]),
                "flops": 4 * case["hq"] * case["d"] * pairs}
    if kind == "moe":
        t, h, i, n, k = (case[x] for x in ("tokens", "hidden", "inter", "experts", "top_k"))
        # experts that a call is expected to touch: each token picks k of n
        touched = n * (1.0 - (1.0 - k / n) ** t)
        return {"bytes": int(e * (3 * h * i * touched + 2 * t * h) + 12 * t * k), "flops": 6 * t * k * h * i}
    if kind == "conv":
        b, ci, co, kk = case["batch"], case["cin"], case["cout"], case["ksize"]
        out = (case["size"] + 2 * case["padding"] - kk) // case["stride"] + 1
        return {"bytes": e * (b * ci * case["size"] ** 2 + co * ci * kk * kk + co + b * co * out * out),
                "flops": 2 * b * co * out * out * ci * kk * kk}
    b, t = case["batch"], case["tokens"]
    n, d, hidden, inter, experts, top_k = b * t, 2048, 8192, 768, 8, 2
    weights = 2 * d * hidden + (d + 1024) * d + d * d + experts * d + 3 * experts * d * inter + 7 * d
    flops = 2 * n * (2 * d * hidden + (d + 1024) * d + d * d + experts * d + 3 * top_k * d * inter)
    return {"bytes": e * (weights + 2 * n * d), "flops": flops + 4 * b * 16 * 128 * _visible(t, t, True)}


# Largest relative difference (2-norm) of another correct implementation at the same precision:
# about four times what the calls measured against 64-bit arithmetic (a single 16-bit rounding of
# each output 1.7e-3 in bf16 and 2.1e-4 in fp16; the roundings inside attention 6.0e-3 / 6.8e-4, of
# the expert layer 6.2e-3 and of convolution plus bias 2.4e-3 in bf16; 32-bit sums up to 8.7e-7).
_REL = {("linear", "bf16"): 7e-3, ("linear", "fp16"): 8e-4, ("rows", "bf16"): 7e-3, ("sdpa", "bf16"): 2.4e-2,
        ("sdpa", "fp16"): 2.7e-3, ("varlen", "bf16"): 2.4e-2, ("varlen", "fp16"): 2.7e-3, ("moe", "bf16"): 2.5e-2,
        ("conv", "bf16"): 1e-2}


def tolerance(case):
    if case["kind"] == "block":
        # attention with its row sums in another order moved the actions by 5.3e-4 and one expert
        # choice in 2048 (a tie of 16-bit router logits)
        return {"rel": 4e-3, "differ": 4e-3}
    if case["dtype"] == "fp32":
        return {"rel": 4e-6}
    return {"rel": _REL[case["kind"], case["dtype"]]}


# ----------------------------------------------------------------------- 64-bit values ----
def _attention(q, k, v, visible=None, add=None):
    """One sample: q [hq, lq, d], k / v [hkv, lk, d] in float64; ``visible`` broadcasts to the scores."""
    group = q.shape[0] // k.shape[0]
    k, v = k.repeat_interleave(group, 0), v.repeat_interleave(group, 0)
    s = torch.bmm(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
    if add is not None:
        s = s + add
    if visible is not None:
        s = s.masked_fill(~visible, -math.inf)
    p = torch.softmax(s, dim=-1).nan_to_num(0.0)
    return torch.bmm(p, v)


def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        # the top-k choice of experts follows the 16-bit roundings of the layers before it: there
        # is no 64-bit value of the outputs behind it
        return None
    t = {n: (x.double() if torch.is_tensor(x) and x.is_floating_point() else x)
         for n, x in _inputs(case, seed).items()}
    if kind == "linear":
        y = t["x"] @ t["w"].t()
        return y + t["b"] if t["b"] is not None else y
    if kind == "mm":
        return t["a"] @ t["b"]
    if kind == "rows":
        x = t["x"]
        return {"softmax": lambda: torch.softmax(x, -1), "log_softmax": lambda: torch.log_softmax(x, -1),
                "mean": lambda: x.mean(-1), "l2_norm": lambda: x.square().sum(-1).sqrt()}[case["op"]]()
    if kind == "sdpa":
        lq, lk = case["lq"], case["lk"]
        tri = torch.ones(lq, lk, dtype=torch.bool, device="cuda").tril() if case["mode"] == "causal" else None
        out = []
        for i in range(case["batch"]):
            visible, add = tri, None
            if case["mode"] == "bool":
                visible = t["mask"][i]
            elif case["mode"] == "add":
                add = t["mask"][i]
            out.append(_attention(t["q"][i], t["k"][i], t["v"][i], visible, add))
        return torch.stack(out)
    if kind == "varlen":
        ends = t["offsets"].tolist()
        out = torch.zeros_like(t["q"])
        for a, b in zip(ends, ends[1:]):
            if a == b:
                continue
            q, k, v = (t[x][0, a:b].transpose(0, 1).contiguous() for x in "qkv")
            tri = torch.ones(b - a, b - a, dtype=torch.bool, device="cuda").tril() if case["causal"] else None
            out[0, a:b] = _attention(q, k, v, tri).transpose(0, 1)
        return out
    if kind == "moe":
        x, out = t["x"], torch.zeros_like(t["x"])
        for e in range(case["experts"]):
            token, slot = (t["chosen"] == e).nonzero(as_tuple=True)
            if token.numel():
                rows = x[token]
                y = (torch.nn.functional.silu(rows @ t["gate"][e].t()) * (rows @ t["up"][e].t())) @ t["down"][e].t()
                out.index_add_(0, token, y * t["weights"][token, slot, None])
        return out
    s, p, k = case["stride"], case["padding"], case["ksize"]
    x = torch.nn.functional.pad(t["x"], (p, p, p, p))
    n = (case["size"] + 2 * p - k) // s + 1
    out = t["b"].view(1, -1, 1, 1).expand(case["batch"], -1, n, n).clone()
    for i in range(k):
        for j in range(k):
            tap = x[:, :, i:i + s * (n - 1) + 1:s, j:j + s * (n - 1) + 1:s]
            out += (t["w"][:, :, i, j] @ tap.reshape(case["batch"], case["cin"], n * n)).view_as(out)
    return out
