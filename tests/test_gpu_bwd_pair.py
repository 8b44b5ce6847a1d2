"""The first backward's kernels with two waves per 32 rows: dK/dV per 32 keys
(fhog_bwd_pair.h) and dQ per 32 queries (fhog_bwd_qpair.hip).

The first serves fp32 and 2-byte head dims 128 and 256 always, and 2-byte
D = 64 on small grids or with FLASH_HOG_BWD=pair; the second fp32 and head dim
256 always, and 2-byte 64 and 128 on small grids or with FLASH_HOG_BWDQ=pair.
Sizes are where they can go wrong: one row, one tile and its neighbours, a
ragged last tile on either side, blocks of 64 that are half empty or see
nothing, grouped heads, and grids above the sizes where the launch folds the
block order (257 to 512 workgroups on 256 CUs) and takes more waves per SIMD, with
a mask and without (over 512 and over 1024 workgroups). Against the closed form in fp64 at the tolerances of
tests/helpers.py (fp32 products here sum at most 1300 terms). They must give
the bits of bwd_k_kernel (D = 64) and bwd_q_kernel (2-byte D = 64 and 128).
"""

from __future__ import annotations

import pytest
import torch

from helpers import DEGENERATE_FLOOR, TOL, default_scale, make_inputs, rel_err

pytestmark = pytest.mark.gpu

# id, batch, n_q, n_k, heads, kv_heads, causal (C ABI code)
SHAPES = [
    ("one_row", 1, 1, 1, 1, 1, 1),
    ("tile_minus_1", 1, 31, 31, 2, 1, 1),
    ("tile_plus_1", 1, 33, 65, 2, 2, 0),
    ("half_block", 2, 96, 96, 4, 2, 1),
    ("ragged_gqa", 1, 130, 77, 4, 1, 0),
    ("empty_blocks", 1, 64, 300, 2, 2, 1),
    ("bottom_right_long_q", 1, 300, 100, 2, 2, 2),
    ("folded_order", 37, 450, 450, 1, 1, 1),
    ("over_1024_workgroups", 26, 600, 600, 4, 4, 1),
    ("over_512_workgroups_no_mask", 15, 600, 600, 4, 4, 0),
    ("over_1024_workgroups_no_mask", 26, 600, 600, 4, 4, 0),
]
KINDS = [(torch.bfloat16, 64), (torch.bfloat16, 128), (torch.float16, 256), (torch.float32, 64), (torch.float32, 128)]


def _probs(q, k, scale, causal):
    s = scale * (q @ k.t().contiguous())
    if causal:
        off = k.shape[0] - q.shape[0] if causal == 2 else 0
        i = torch.arange(q.shape[0], device=q.device)[:, None]
        s = s.masked_fill(torch.arange(k.shape[0], device=q.device)[None, :] > i + off, float("-inf"))
    lse = torch.logsumexp(s, -1)
    lse = torch.where(torch.isneginf(lse), float("inf"), lse)  # rows without keys: P = 0
    return torch.exp(s - lse[:, None]), lse


@pytest.mark.parametrize("dtype,D", KINDS, ids=[f"{str(t).split('.')[1]}_d{d}" for t, d in KINDS])
@pytest.mark.parametrize("shape", SHAPES, ids=[s[0] for s in SHAPES])
def test_bwd_pair(shape, dtype, D, cuda_device, monkeypatch):
    from flash_hog import _hip

    name, B, Nq, Nk, H, Hk, causal = shape
    print("[case] first backward, two waves per 32 keys:", name, dtype, D, flush=True)
    scale = default_scale(D)
    x = make_inputs(B, Nq, Nk, H, D, dtype, seed=31, kv_heads=Hk, device=cuda_device)
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
    args = (x["q"], x["k"], x["v"], o, x["do"], lse, causal, scale)
    monkeypatch.setenv("FLASH_HOG_BWD", "pair")
    monkeypatch.setenv("FLASH_HOG_BWDQ", "pair")
    got = _hip.attention_bwd(*args)
    torch.cuda.synchronize()
    if D <= 128 and dtype is not torch.float32:
        monkeypatch.setenv("FLASH_HOG_BWD", "compiled")
        monkeypatch.setenv("FLASH_HOG_BWDQ", "compiled")
        want = _hip.attention_bwd(*args)
        for a, r, label in zip(got, want, ("dq", "dk", "dv", "D")):
            assert torch.equal(a, r), label
    grp = H // Hk
    for b in sorted({0, B - 1}):
        for hk in range(Hk):
            dk = dv = 0.0
            for h in range(hk * grp, (hk + 1) * grp):
                p, do = probs[b, h], f(x["do"], b, h)
                d = (f(o, b, h) * do).sum(-1, keepdim=True)
                ds = scale * p * (do @ f(x["v"], b, hk).t().contiguous() - d)
                for a, r, label in ((got[0][b, :, h], ds @ f(x["k"], b, hk), "dq"), (got[3][b, h], d[:, 0], "D")):
                    err = rel_err(a, r, DEGENERATE_FLOOR)
                    assert err < TOL[dtype], f"{label} batch {b} head {h}: {err:.2e}"
                dk = dk + ds.t().contiguous() @ f(x["q"], b, h)
                dv = dv + p.t().contiguous() @ do
            for a, r, label in ((got[1], dk, "dk"), (got[2], dv, "dv")):
                err = rel_err(a[b, :, hk], r, DEGENERATE_FLOOR)
                assert err < TOL[dtype], f"{label} batch {b} head {hk}: {err:.2e}"
