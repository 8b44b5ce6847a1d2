"""Stage 1 at D = 128 with two waves per 32 queries (fhog_bwdbwd_fused_pair.hip).

Sizes where it can go wrong: one row, a tile and its neighbours, ragged last
tiles, half-empty and empty 64- and 128-query blocks, rows that see no key,
grouped heads, a grid whose block order the launch folds (257 to 512 workgroups
of 64 queries) and one that takes 128-query workgroups (more). dQ2, ddO and the row
statistics against the closed form in fp64, at the tolerances of
tests/helpers.py; a sequence inside a large grid gives the bits it gives alone in
a small one.
"""

from __future__ import annotations

import pytest
import torch

from helpers import DEGENERATE_FLOOR, TOL, default_scale, make_inputs, rel_err
from test_gpu_bwd_pair import SHAPES, _probs

pytestmark = pytest.mark.gpu

D = 128
# grids of 128-query workgroups, which compute a power-of-two scale in another instance
LARGE = [s for s in SHAPES if s[0].startswith("over_")]
SCALES = {"default": None, "pow2": 0.125, "negative": -0.11}


def _inputs(shape, dtype, scale, device):
    name, B, Nq, Nk, H, Hk, causal = shape
    x = make_inputs(B, Nq, Nk, H, D, dtype, seed=43, kv_heads=Hk, device=device)
    o = torch.empty_like(x["q"])
    lse = torch.empty((B, H, Nq), device=device)
    f = lambda t, b, j: t[b, :, j].double().contiguous()
    probs = {}
    for b in range(B):
        for h in range(H):
            p, l64 = _probs(f(x["q"], b, h), f(x["k"], b, h * Hk // H), scale, causal)
            o[b, :, h] = (p @ f(x["v"], b, h * Hk // H)).to(dtype)
            lse[b, h] = l64.float()
            if b in (0, B - 1):
                probs[b, h] = p
    return x, o, lse, probs


def _run(x, o, lse, causal, scale, b=slice(None)):
    from flash_hog import _hip

    c = lambda t: t[b].contiguous()
    dq2, _, _, ddo, stats = _hip.attention_bwdbwd(c(x["q"]), c(x["k"]), c(x["v"]), c(o), c(x["do"]), c(x["ddq"]),
                                                  c(x["ddk"]), c(x["ddv"]), c(lse), causal, scale, return_stats=True)
    torch.cuda.synchronize()
    return (dq2, ddo, *stats)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("shape,scale", [(s, "default") for s in SHAPES] + [(SHAPES[4], "pow2"), (SHAPES[6], "negative")]
                         + [(s, "pow2") for s in LARGE],
                         ids=[s[0] for s in SHAPES] + ["pow2_scale", "negative_scale"]
                         + ["pow2_scale_" + s[0] for s in LARGE])
def test_stage1_pair(shape, scale, dtype, cuda_device):
    name, B, Nq, Nk, H, Hk, causal = shape
    print("[case] stage 1 at D = 128, two waves per 32 queries:", name, scale, dtype, flush=True)
    scale = SCALES[scale] or default_scale(D)
    x, o, lse, probs = _inputs(shape, dtype, scale, cuda_device)
    got = _run(x, o, lse, causal, scale)
    f = lambda t, b, j: t[b, :, j].double().contiguous()
    t = lambda m: m.t().contiguous()
    for b in sorted({0, B - 1}):
        alone = _run(x, o, lse, causal, scale, slice(b, b + 1))
        for a, r in zip(got, alone):
            assert torch.equal(a[b:b + 1], r)
        for h in range(H):
            hk = h * Hk // H
            k, v, ddk, ddv = (f(x[i], b, hk) for i in ("k", "v", "ddk", "ddv"))
            p, do, q, ddq = probs[b, h], f(x["do"], b, h), f(x["q"], b, h), f(x["ddq"], b, h)
            d = (f(o, b, h) * do).sum(-1, keepdim=True)
            dp = do @ t(v)
            dds = scale * (ddq @ t(k) + q @ t(ddk))
            dd = (dds * p).sum(-1, keepdim=True)
            dp2 = do @ t(ddv) - dp * dd - dds * d + dp * dds
            bst = (dp2 * p).sum(-1, keepdim=True)
            dq2 = scale * (p * (dp - d)) @ ddk + scale * (p * (dp2 - bst)) @ k
            ddo = p @ ddv + (p * (dds - dd)) @ v
            for a, r, label in ((got[0][b, :, h], dq2, "dq2"), (got[1][b, :, h], ddo, "ddo"),
                                (got[2][b, h], d[:, 0], "D"), (got[3][b, h], dd[:, 0], "dD"),
                                (got[4][b, h], bst[:, 0], "B")):
                err = rel_err(a, r, DEGENERATE_FLOOR)
                assert err < TOL[dtype], f"{label} batch {b} head {h}: {err:.2e}"
