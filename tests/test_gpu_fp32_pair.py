"""fp32's kernels with two waves per 32 queries give the bits of the ones with one.

launch_fwd and launch_bwdbwd choose between fwd_kernel and fwd_pair_kernel
(fhog_fwd_pair.hip), and between bwdbwd_q_kernel and bwdbwd_qpair_kernel
(fhog_bwdbwd_qpair.hip), by the size of the grid; FLASH_HOG_FWD and
FLASH_HOG_STAGE1 = pair or compiled force one. The sizes are one row, a tile and
its neighbours, ragged last tiles, half-empty and empty 64-query blocks, rows
that see no key, grouped heads, and a grid whose block order the launch folds.
That the bits are right is the parity suites' matter, which run small grids, the
pair kernels, and full-size ones.
"""

from __future__ import annotations

import pytest
import torch

from helpers import default_scale, make_inputs
from test_gpu_bwd_pair import SHAPES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("scale", [None, -0.11])
@pytest.mark.parametrize("shape", SHAPES, ids=[s[0] for s in SHAPES])
def test_fp32_pair_kernels_match(shape, scale, D, cuda_device, monkeypatch):
    from flash_hog import _hip

    name, B, Nq, Nk, H, Hk, causal = shape
    print("[case] fp32, two waves per 32 queries:", name, D, flush=True)
    scale = scale or default_scale(D)
    x = make_inputs(B, Nq, Nk, H, D, torch.float32, seed=41, kv_heads=Hk, device=cuda_device)
    out = {}
    for which in ("compiled", "pair"):
        monkeypatch.setenv("FLASH_HOG_FWD", which)
        monkeypatch.setenv("FLASH_HOG_STAGE1", which)
        o, lse = _hip.attention_fwd(x["q"], x["k"], x["v"], causal, scale)
        dq2, dk2, dv2, ddo, stats = _hip.attention_bwdbwd(x["q"], x["k"], x["v"], o, x["do"], x["ddq"], x["ddk"],
                                                          x["ddv"], lse, causal, scale, return_stats=True)
        torch.cuda.synchronize()
        out[which] = (o, lse, dq2, dk2, dv2, ddo, *stats)
    for a, r, label in zip(out["pair"], out["compiled"], ("o", "lse", "dq2", "dk2", "dv2", "ddo", "D", "dD", "B")):
        assert torch.equal(a, r), label
        assert not torch.isnan(a).any(), label
