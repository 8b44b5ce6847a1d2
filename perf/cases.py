"""Performance cases of the attention path: forward, first backward, double backward and
Hessian-vector product through the package's entry points.

listed() names the cases, draw(rng) gives one more of the same ranges, prepare(case, seed)
makes the inputs on the GPU, run(state) is one pass, work(case) its least bytes and flops,
tolerance(case) how far two correct implementations may differ, exact(case, seed) the
outputs in 64 bits from plain torch.

A case is one call pattern of a user's program (`kind`) at one size:

  forward  dot_product_attention without autograd (inference, prefill)
  train    dot_product_attention and the gradients of q, k, v for an upstream gradient
  hvp      the gradients and a Hessian-vector product: the gradient computed with
           create_graph, then differentiated along tangents of q, k, v
  double   the double backward alone on saved residuals, as a custom rule that holds
           (q, k, v, O, dO, L) calls it
"""

import math
import os
import sys

import torch

_PACKAGE_ROOT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash-hog_amd")
if _PACKAGE_ROOT not in sys.path:
    sys.path.insert(0, _PACKAGE_ROOT)

import flash_hog  # noqa: E402
from flash_hog import _hip  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_CAUSAL_CODE = {"none": 0, "top_left": 1, "bottom_right": 2}


def _case(name, kind, batch, n_q, n_k, heads, kv_heads, head_dim, dtype, causal):
    case = {"kind": kind, "batch": batch, "n_q": n_q, "n_k": n_k, "heads": heads, "kv_heads": kv_heads,
            "head_dim": head_dim, "dtype": dtype, "causal": causal}
    return {"name": name, **case} if name else case


def listed():
    return [
        # A short sequence on its own (12 heads, 64 wide): the smallest row of the
        # Hessian-vector-product table, where host time and launches weigh most.
        _case("hvp_b1_n512_h12_d64", "hvp", 1, 512, 512, 12, 12, 64, "bf16", "top_left"),
        # The double backward of one medium sequence: few rows for a large chip.
        _case("double_b1_n1024_h12_d64", "double", 1, 1024, 1024, 12, 12, 64, "bf16", "top_left"),
        # One longer sequence per step, as in curvature probes at batch 1.
        _case("hvp_b1_n4096_h12_d64", "hvp", 1, 4096, 4096, 12, 12, 64, "bf16", "top_left"),
        # The standard configuration of the double backward (bench.py's default).
        _case("double_b4_n2048_h16_d64", "double", 4, 2048, 2048, 16, 16, 64, "bf16", "top_left"),
        # A bidirectional encoder's sequence length that is no multiple of a tile, in fp16.
        _case("double_b8_n1000_h12_d64_fp16", "double", 8, 1000, 1000, 12, 12, 64, "fp16", "none"),
        # Long context: the largest case.
        _case("double_b1_n32768_h8_d64", "double", 1, 32768, 32768, 8, 8, 64, "bf16", "top_left"),
        # 128-wide heads at a training length.
        _case("double_b2_n8192_h16_d128", "double", 2, 8192, 8192, 16, 16, 128, "bf16", "top_left"),
        # An ordinary first-order training step with grouped heads.
        _case("train_b2_n2048_h32_kv8_d128", "train", 2, 2048, 2048, 32, 8, 128, "bf16", "top_left"),
        # Inference: a chunk of a prompt against the keys so far (bottom-right mask).
        _case("forward_b2_q1024_k4096_h32_kv8_d128", "forward", 2, 1024, 4096, 32, 8, 128, "bf16", "bottom_right"),
        # Many short sequences per step: throughput instead of latency.
        _case("hvp_b128_n512_h12_d64", "hvp", 128, 512, 512, 12, 12, 64, "bf16", "top_left"),
        # Full-precision inputs, as a second-order method's accuracy reference uses them.
        _case("hvp_b2_n2048_h8_d64_fp32", "hvp", 2, 2048, 2048, 8, 8, 64, "fp32", "top_left"),
        # The widest heads the kernels take.
        _case("hvp_b2_n2048_h8_d256", "hvp", 2, 2048, 2048, 8, 8, 256, "bf16", "top_left"),
    ]


# ------------------------------------------------------------------ more cases

_MAX_GFLOP = {"bf16": 1500.0, "fp16": 1500.0, "fp32": 60.0}


def draw(rng):
    """One case of the ranges above: any kind, 200 to 16384 tokens (logarithmic, mostly no
    multiple of a tile), batch 1 to 128, 1 to 32 heads, grouped or not, each dtype and
    mask, head dims of the kernels and ones between them (which the front-end pads)."""
    while True:
        kind = rng.choice(("forward", "train", "hvp", "double"))
        dtype = rng.choices(("bf16", "fp16", "fp32"), (6, 3, 1))[0]
        if kind == "double":  # the native entry point takes the kernels' own head dims
            dims = (64, 64, 128) if dtype == "fp32" else (64, 64, 64, 128, 128, 256)
        else:
            dims = (64, 64, 128, 40) if dtype == "fp32" else (64, 64, 64, 128, 128, 256, 80, 96)
        head_dim = rng.choice(dims)
        n_q = int(round(math.exp(rng.uniform(math.log(200), math.log(16384)))))
        if rng.random() < 0.4:
            n_q = max(256, n_q // 256 * 256)
        batch = int(round(math.exp(rng.uniform(0, math.log(128)))))
        kv_heads = rng.choice((1, 2, 4, 8, 12, 16))
        heads = kv_heads * rng.choice((1, 1, 1, 2, 4))
        causal = rng.choices(("none", "top_left", "bottom_right"), (3, 5, 2))[0]
        n_k = n_q
        if causal == "bottom_right" and kind in ("forward", "double"):
            n_k = int(n_q * rng.uniform(1.0, 4.0))
        if heads > 32 or n_k > 32768:
            continue
        case = _case(None, kind, batch, n_q, n_k, heads, kv_heads, head_dim, dtype, causal)
        w = work(case)
        if 1.0 <= w["flops"] / 1e9 <= _MAX_GFLOP[dtype] and w["bytes"] <= 3e9:
            return case


# ------------------------------------------------------------------ inputs and one pass

def _scale(case):
    return case["head_dim"] ** -0.5


def _tensors(case, seed):
    """q, k, v, the upstream gradient and the tangents of q, k, v: N(0, 1) in the case's dtype."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    q_shape = (case["batch"], case["n_q"], case["heads"], case["head_dim"])
    k_shape = (case["batch"], case["n_k"], case["kv_heads"], case["head_dim"])
    names = {"forward": ("q", "k", "v"), "train": ("q", "k", "v", "cot")}.get(
        case["kind"], ("q", "k", "v", "cot", "tq", "tk", "tv"))
    out = {}
    for name in names:
        shape = q_shape if name in ("q", "cot", "tq") else k_shape
        out[name] = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(_DTYPES[case["dtype"]])
    return out


def prepare(case, seed):
    x = _tensors(case, seed)
    state = {"case": case, **x}
    if case["kind"] in ("train", "hvp"):
        for name in ("q", "k", "v"):
            state[name] = x[name].requires_grad_()
    elif case["kind"] == "double":
        # the residuals that a forward left: O in the inputs' dtype, the logsumexp in fp32
        o, lse = _reference(case, x, torch.float32, ("o", "lse"))
        state["o"], state["lse"] = o.to(x["q"].dtype), lse
    return state


def _attention(case, s):
    alignment = "bottom_right" if case["causal"] == "bottom_right" else "top_left"
    return flash_hog.dot_product_attention(s["q"], s["k"], s["v"], case["causal"] != "none",
                                           causal_alignment=alignment)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "forward":
        with torch.no_grad():
            return _attention(case, s)
    if kind == "double":
        return _hip.attention_bwdbwd(s["q"], s["k"], s["v"], s["o"], s["cot"], s["tq"], s["tk"], s["tv"], s["lse"],
                                     _CAUSAL_CODE[case["causal"]], _scale(case))
    leaves = (s["q"], s["k"], s["v"])
    out = _attention(case, s)
    if kind == "train":
        return (out.detach(), *torch.autograd.grad(out, leaves, s["cot"]))
    grads = torch.autograd.grad(out, leaves, s["cot"], create_graph=True)
    products = torch.autograd.grad(grads, leaves, (s["tq"], s["tk"], s["tv"]))
    return (*(g.detach() for g in grads), *products)


# ------------------------------------------------------------------ least work

def _pairs(case):
    """Unmasked (query, key) pairs over all heads."""
    n_q, n_k = case["n_q"], case["n_k"]
    if case["causal"] == "none":
        per_head = n_q * n_k
    else:
        off = n_k - n_q if case["causal"] == "bottom_right" else 0
        rows = [min(n_k, max(0, i + off + 1)) for i in (0, n_q - 1)]
        # row i sees i + off + 1 keys (all sizes here have off >= 0 and n_k >= n_q)
        per_head = (rows[0] + rows[1]) * n_q // 2
    return per_head * case["batch"] * case["heads"]


def work(case):
    """Matrix products per pair: 2 (forward), 5 more (first backward), 12 more (double
    backward), each 2 * head_dim flops; bytes of the inputs and outputs of one pass."""
    item = 4 if case["dtype"] == "fp32" else 2
    d = case["head_dim"]
    q = case["batch"] * case["n_q"] * case["heads"] * d * item
    k = case["batch"] * case["n_k"] * case["kv_heads"] * d * item
    rows = case["batch"] * case["n_q"] * case["heads"] * 4
    products, size = {
        "forward": (2, 2 * q + 2 * k),                       # q k v -> out
        "train": (7, 4 * q + 4 * k),                         # q k v cot -> out dq dk dv
        "hvp": (19, 5 * q + 8 * k),                          # q k v cot tangents -> gradients, products
        "double": (12, 6 * q + 6 * k + rows),                # q k v o cot tangents lse -> dq2 dk2 dv2 ddo
    }[case["kind"]]
    return {"bytes": size, "flops": products * 2 * d * _pairs(case)}


# ------------------------------------------------------------------ accuracy

def tolerance(case):
    """About four times the distance of the outputs from their 64-bit values, which is 2.1e-3
    to 2.7e-3 (bf16), 2.8e-4 to 3.2e-4 (fp16) and 5e-7 to 1.8e-6 (fp32) over the listed sizes
    and drawn ones: 16-bit operands and results round at 2^-9 (bf16) or 2^-12 (fp16), and the
    probabilities and score gradients enter the products rounded; fp32 sums up to 2048 terms."""
    return {"rel": {"bf16": 1e-2, "fp16": 1.3e-3, "fp32": 8e-6}[case["dtype"]]}


def exact(case, seed):
    x = _tensors(case, seed)
    kind = case["kind"]
    if kind == "double":
        o, lse = _reference(case, x, torch.float32, ("o", "lse"))
        x["o"], x["lse"] = o.to(x["q"].dtype), lse  # the residuals as the call has them
        wanted = ("dq2", "dk2", "dv2", "ddo")
    else:
        wanted = {"forward": ("o",), "train": ("o", "dq", "dk", "dv"),
                  "hvp": ("dq", "dk", "dv", "dq2", "dk2", "dv2")}[kind]
    got = _reference(case, x, torch.float64, wanted)
    return got[0] if kind == "forward" else got


def _reference(case, x, dtype, wanted):
    """The attention outputs `wanted`, from the closed forms with the score matrices of some
    heads and query rows at a time: P = exp(S - L), dP = dO V', D = rowsum(O dO),
    dS = P (dP - D), ddS = T_q K' + Q T_k', dP2 = dO T_v' - dD dP - D ddS + dP ddS, ...
    (the row statistics dD = rowsum(P ddS), B = rowsum(P dP2))."""
    scale = _scale(case)
    n_q, n_k = case["n_q"], case["n_k"]
    group = case["heads"] // case["kv_heads"]
    off = n_k - n_q if case["causal"] == "bottom_right" else 0
    first = any(w in ("dq", "dk", "dv") for w in wanted)
    second = any(w in ("dq2", "dk2", "dv2", "ddo") for w in wanted)
    query_side = ("o", "dq", "dq2", "ddo")
    key_side = ("dk", "dv", "dk2", "dv2")
    out = {}
    for w in wanted:
        if w == "lse":
            out[w] = torch.empty((case["batch"], case["heads"], n_q), device="cuda", dtype=dtype)
        else:
            out[w] = torch.zeros(x["q" if w in query_side else "k"].shape, device="cuda", dtype=dtype)
    rows = min(n_q, 1024)
    heads_at_once = max(1, min(case["kv_heads"], (1 << 26) // (rows * n_k * group)))
    t = lambda m: m.transpose(-1, -2).contiguous()
    for b in range(case["batch"]):
        for hk0 in range(0, case["kv_heads"], heads_at_once):
            hk1 = min(hk0 + heads_at_once, case["kv_heads"])
            hq = slice(hk0 * group, hk1 * group)
            one = lambda name: x[name][b, :, hq].detach().to(dtype).transpose(0, 1).contiguous()
            per_group = lambda name: (x[name][b, :, hk0:hk1].detach().to(dtype).transpose(0, 1)
                                      .repeat_interleave(group, dim=0).contiguous())
            q, k, v = one("q"), per_group("k"), per_group("v")
            kT, vT = t(k), t(v)
            sums = {w: torch.zeros_like(k) for w in wanted if w in key_side}
            if first or second:
                do = one("cot")
            if second:
                tq, tk, tv = one("tq"), per_group("tk"), per_group("tv")
                tkT, tvT = t(tk), t(tv)
            for r0 in range(0, n_q, rows):
                r = slice(r0, min(r0 + rows, n_q))
                s = torch.matmul(q[:, r], kT).mul_(scale)
                if case["causal"] != "none":
                    i = torch.arange(r.start, r.stop, device="cuda")[:, None]
                    s.masked_fill_(torch.arange(n_k, device="cuda")[None, :] > i + off, float("-inf"))
                lse = x["lse"][b, hq, r].to(dtype) if "lse" in x else torch.logsumexp(s, -1)
                p = s.sub_(lse[..., None]).exp_()
                got = {"lse": lse}
                o = one("o")[:, r] if "o" in x else torch.matmul(p, v)
                got["o"] = o
                if first or second:
                    dor = do[:, r].contiguous()
                    dp = torch.matmul(dor, vT)
                    d = (o * dor).sum(-1, keepdim=True)
                    ds = (dp - d).mul_(p).mul_(scale)
                    dsT = t(ds)
                if first:
                    got["dq"] = torch.matmul(ds, k)
                    got["dk"] = torch.matmul(dsT, q[:, r])
                    got["dv"] = torch.matmul(t(p), dor)
                if second:
                    tqr = tq[:, r].contiguous()
                    dds = (torch.matmul(tqr, kT) + torch.matmul(q[:, r], tkT)).mul_(scale)
                    dd = (dds * p).sum(-1, keepdim=True)
                    dp2 = torch.matmul(dor, tvT) - dp * dd - dds * d + dp * dds
                    bst = (dp2 * p).sum(-1, keepdim=True)
                    ds2 = dp2.sub_(bst).mul_(p).mul_(scale)
                    ddp = dds.sub_(dd).mul_(p)
                    got["dq2"] = torch.matmul(ds, tk) + torch.matmul(ds2, k)
                    got["dk2"] = torch.matmul(dsT, tqr) + torch.matmul(t(ds2), q[:, r])
                    got["dv2"] = torch.matmul(t(ddp), dor)
                    got["ddo"] = torch.matmul(p, tv) + torch.matmul(ddp, v)
                for w in wanted:
                    if w == "lse":
                        out[w][b, hq, r] = got[w]
                    elif w in query_side:
                        out[w][b, r, hq] = got[w].transpose(0, 1)
                    else:
                        sums[w] += got[w]
            for w, m in sums.items():
                out[w][b, :, hk0:hk1] = m.unflatten(0, (hk1 - hk0, group)).sum(1).transpose(0, 1)
    return tuple(out[w] for w in wanted)
