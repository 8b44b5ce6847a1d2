"""The forward with two waves per 32 queries (fhog_fwd_pair.hip) at D = 256.

Every 2-byte D = 256 forward runs it. The sizes are test_gpu_bwd_pair.py's: one row,
tile edges, half-empty and empty 64-query blocks, rows that see no key, grouped heads,
and grids whose block order the launch folds (257 to 512 workgroups) or not (more).
O and L against the closed form in fp64 on the first and last sequence, at the
tolerances of tests/helpers.py, L to 1e-3 of max(1, max|L|); a sequence inside a large
grid gives the bits it gives alone. One case has a negative scale.
"""

from __future__ import annotations

import pytest
import torch

from helpers import DEGENERATE_FLOOR, TOL, default_scale, make_inputs, rel_err
from test_gpu_bwd_pair import SHAPES, _probs

pytestmark = pytest.mark.gpu

D = 256


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("shape,scale", [(s, None) for s in SHAPES] + [(SHAPES[7], -0.07)],
                         ids=[s[0] for s in SHAPES] + ["folded_negative_scale"])
def test_fwd_pair_d256(shape, scale, dtype, cuda_device):
    from flash_hog import _hip

    name, B, Nq, Nk, H, Hk, causal = shape
    print("[case] forward at D = 256, two waves per 32 queries:", name, scale, dtype, flush=True)
    scale = scale or default_scale(D)
    x = make_inputs(B, Nq, Nk, H, D, dtype, seed=47, kv_heads=Hk, device=cuda_device)
    o, lse = _hip.attention_fwd(x["q"], x["k"], x["v"], causal, scale)
    torch.cuda.synchronize()
    for b in sorted({0, B - 1}):
        c = lambda t: t[b:b + 1].contiguous()
        o1, lse1 = _hip.attention_fwd(c(x["q"]), c(x["k"]), c(x["v"]), causal, scale)
        torch.cuda.synchronize()
        assert torch.equal(o[b:b + 1], o1) and torch.equal(lse[b:b + 1], lse1)
        for h in range(H):
            f = lambda t, j: t[b, :, j].double().contiguous()
            p, want = _probs(f(x["q"], h), f(x["k"], h * Hk // H), scale, causal)
            err = rel_err(o[b, :, h], p @ f(x["v"], h * Hk // H), DEGENERATE_FLOOR)
            assert err < TOL[dtype], f"O batch {b} head {h}: {err:.2e}"
            seen = torch.isfinite(want)
            assert torch.equal(lse[b, h][~seen].double(), want[~seen])
            if seen.any():
                err = (lse[b, h][seen].double() - want[seen]).abs().max() / want[seen].abs().max().clamp(min=1.0)
                assert err < 1e-3, f"L batch {b} head {h}: {err:.2e}"
