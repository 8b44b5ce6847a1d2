"""Block orders of the causal kernels that keep one workgroup per CU or per slot.

bwdbwd_q32_kernel (stage 1), bwdbwd_k_kernel (stage 2) and bwd_k64_kernel choose
the order of their blocks by the size of the grid: one block per workgroup, blocks
dealt over several rounds, or mirrored blocks folded into one item. Every order
runs every block once with the same arithmetic, so a sequence's results must have
the same bits alone and inside a batch whose grid takes another order. The
batches below give, with 128-row blocks on 256 CUs, three blocks per head in
1.5 rounds, four in 1.25 rounds of folded items, four in exactly one and two of
them, and nine blocks in 4.5 rounds; in stage 2, at two workgroups per CU, three
and four blocks mirrored in one round (an odd count has a middle block that is its
own mirror), eight unmirrored although they would fill two, and 32 mirrored in
half a round.
"""

from __future__ import annotations

import pytest
import torch

from helpers import default_scale, make_inputs

pytestmark = pytest.mark.gpu

# name, batch, n_q, n_k, heads, causal
GRIDS = [
    ("three_blocks_ragged", 43, 300, 300, 3, 1),
    ("four_blocks_uneven_rounds", 40, 512, 512, 4, 1),
    ("four_blocks_whole_round", 32, 512, 512, 4, 1),
    ("three_blocks_mirrored", 64, 330, 330, 4, 1),
    ("four_blocks_two_rounds", 64, 512, 512, 4, 1),
    ("eight_blocks_two_rounds", 64, 1000, 1000, 4, 1),
    ("many_blocks_one_per_cu", 4, 4000, 4000, 4, 1),
    ("nine_blocks_bottom_right", 8, 1100, 1170, 16, 2),
    ("rows_without_keys", 24, 700, 500, 6, 2),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("grid", GRIDS, ids=[g[0] for g in GRIDS])
def test_results_do_not_depend_on_the_grid(grid, dtype, cuda_device, monkeypatch):
    from flash_hog import _hip

    name, B, Nq, Nk, H, causal = grid
    print("[case] causal grid:", name, dtype, flush=True)
    monkeypatch.setenv("FLASH_HOG_STAGE1", "q32")
    monkeypatch.setenv("FLASH_HOG_STAGE2", "compiled")
    monkeypatch.setenv("FLASH_HOG_BWD", "k64")
    scale = default_scale(64)
    x = make_inputs(B, Nq, Nk, H, 64, dtype, seed=41, device=cuda_device)

    def run(sl):
        y = {k: v[sl].contiguous() for k, v in x.items()}
        o, lse = _hip.attention_fwd(y["q"], y["k"], y["v"], causal, scale)
        first = _hip.attention_bwd(y["q"], y["k"], y["v"], o, y["do"], lse, causal, scale)
        second = _hip.attention_bwdbwd(y["q"], y["k"], y["v"], o, y["do"], y["ddq"], y["ddk"], y["ddv"], lse, causal,
                                       scale)
        torch.cuda.synchronize()
        return [*first, *second]

    whole = run(slice(None))
    for b in (0, B // 2, B - 1):
        for i, (w, a) in enumerate(zip(whole, run(slice(b, b + 1)))):
            assert torch.isfinite(a.float()).all(), (b, i)
            assert torch.equal(w[b : b + 1], a), (b, i)
