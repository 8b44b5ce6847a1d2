"""Stage 2 with two waves per 32 keys (fhog_bwdbwd_pair.hip).

It serves fp32 and 2-byte head dims 128 and 256 always, and 2-byte D = 64 on
small grids or with FLASH_HOG_STAGE2=pair. The sizes are those where
test_gpu_bwd_pair.py's kernel, which splits its work the same way, can go
wrong (one row, tile edges, half-empty and empty key blocks, grouped heads, the
folded block order), with a power-of-two scale and another one for bf16.
dK2 and dV2 are checked against the closed form in fp64 (the oracle's
equations, tests/helpers.py tolerances); at D = 64 they must be
bwdbwd_k_kernel's bits.
"""

from __future__ import annotations

import pytest
import torch

from helpers import DEGENERATE_FLOOR, TOL, default_scale, make_inputs, rel_err
from test_gpu_bwd_pair import KINDS, SHAPES, _probs

pytestmark = pytest.mark.gpu

SCALES = {"default": None, "pow2": 0.125, "negative": -0.11}


@pytest.mark.parametrize("dtype,D", KINDS, ids=[f"{str(t).split('.')[1]}_d{d}" for t, d in KINDS])
@pytest.mark.parametrize("shape,scale", [(s, "default") for s in SHAPES] + [(SHAPES[4], "pow2"), (SHAPES[6], "negative")],
                         ids=[s[0] for s in SHAPES] + ["pow2_scale", "negative_scale"])
def test_stage2_pair(shape, scale, dtype, D, cuda_device, monkeypatch):
    from flash_hog import _hip

    name, B, Nq, Nk, H, Hk, causal = shape
    print("[case] stage 2, two waves per 32 keys:", name, scale, dtype, D, flush=True)
    scale = SCALES[scale] or default_scale(D)
    x = make_inputs(B, Nq, Nk, H, D, dtype, seed=37, kv_heads=Hk, device=cuda_device)
    o = torch.empty_like(x["q"])
    lse = torch.empty((B, H, Nq), device=cuda_device)
    f = lambda t, b, j: t[b, :, j].double().contiguous()
    probs = {}
    for b in range(B):
        for h in range(H):
            p, l64 = _probs(f(x["q"], b, h), f(x["k"], b, h * Hk // H), scale, causal)
            o[b, :, h] = (p @ f(x["v"], b, h * Hk // H)).to(dtype)
            lse[b, h] = l64.float()
            if b in (0, B - 1):
                probs[b, h] = p
    args = (x["q"], x["k"], x["v"], o, x["do"], x["ddq"], x["ddk"], x["ddv"], lse, causal, scale)
    monkeypatch.setenv("FLASH_HOG_STAGE2", "pair")
    got = _hip.attention_bwdbwd(*args)
    torch.cuda.synchronize()
    if D == 64 and dtype is not torch.float32:
        monkeypatch.setenv("FLASH_HOG_STAGE2", "compiled")
        want = _hip.attention_bwdbwd(*args)
        for a, r, label in zip(got, want, ("dq2", "dk2", "dv2", "ddo")):
            assert torch.equal(a, r), label
        return
    grp = H // Hk
    t = lambda m: m.t().contiguous()
    for b in sorted({0, B - 1}):
        for hk in range(Hk):
            k, v, ddk, ddv = (f(x[i], b, hk) for i in ("k", "v", "ddk", "ddv"))
            dk2 = dv2 = 0.0
            for h in range(hk * grp, (hk + 1) * grp):
                p, do, q, ddq = probs[b, h], f(x["do"], b, h), f(x["q"], b, h), f(x["ddq"], b, h)
                d = (f(o, b, h) * do).sum(-1, keepdim=True)
                dp = do @ t(v)
                dds = scale * (ddq @ t(k) + q @ t(ddk))
                dd = (dds * p).sum(-1, keepdim=True)
                dp2 = do @ t(ddv) - dp * dd - dds * d + dp * dds
                ds2 = scale * p * (dp2 - (dp2 * p).sum(-1, keepdim=True))
                dk2 = dk2 + t(scale * p * (dp - d)) @ ddq + t(ds2) @ q
                dv2 = dv2 + t(p * (dds - dd)) @ do
            for a, r, label in ((got[1], dk2, "dk2"), (got[2], dv2, "dv2")):
                err = rel_err(a[b, :, hk], r, DEGENERATE_FLOOR)
                assert err < TOL[dtype], f"{label} batch {b} head {hk}: {err:.2e}"
