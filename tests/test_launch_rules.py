"""The launch rules of csrc/fhog_grid.h, compiled for the host.

The rules are plain C++: a few C wrappers around them are built with the host
compiler and called here with the sizes of 256 CUs, so that a rule can be checked
without a GPU. Each row names a call and the kernel or block order that was
measured the faster one there; the times stand beside the rules.
"""

from __future__ import annotations

import random

import pytest

from rules_host import CUS, load, one_wave_order, stage2_order


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    return load(tmp_path_factory.mktemp("rules"))


def dkdv(r, causal, nq, nk, npairs):
    if r.bwd_pair(causal, nq, nk, npairs, CUS):
        return "pair"
    return "k64" if r.bwd_k64(causal, nq, nk, npairs, CUS) else "compiled"


def dq(r, causal, nq, nk, npairs, d=64):
    if r.bwd_qpair(causal, nq, nk, npairs, d, CUS):
        return "pair"
    return "q64" if r.bwd_q64(causal, nq, nk, npairs, CUS) else "compiled"


# batch, length, heads (square, top-left causal): dK/dV, dQ, stage 2, its block order
SQUARES = [
    (1, 1024, 12, "pair", "pair", "pair", None),
    (1, 4096, 12, "pair", "compiled", "pair", None),
    (2, 2048, 12, "pair", "compiled", "pair", None),
    (2, 2048, 16, "k64", "q64", "k", 0),
    (4, 2048, 16, "k64", "q64", "k", 2),
    (1, 16384, 8, "k64", "q64", "k", 2),
    (8, 2048, 16, "k64", "q64", "k", 0),
    (1, 32768, 8, "k64", "q64", "k", 0),
    (1, 8192, 8, "k64", "q64", "k", 1),
    (4, 2048, 8, "k64", "q64", "k", 0),
    (3, 2048, 12, "k64", "compiled", "k", 0),
]


@pytest.mark.parametrize("row", SQUARES, ids=lambda r: "b%d_n%d_h%d" % r[:3])
def test_squares(rules, row):
    batch, n, heads, want_kv, want_q, want_2, order = row
    np_ = batch * heads
    assert dkdv(rules, 1, n, n, np_) == want_kv
    assert dq(rules, 1, n, n, np_) == want_q
    assert ("pair" if rules.stage2_pair(1, n, n, np_, CUS) else "k") == want_2
    if order is not None:
        assert stage2_order(rules, 1, n, n, np_) == order


def test_folded_ranks_are_a_permutation(rules):
    for nb in range(1, 70):
        for npairs in (1, 3, 8, 12, 37, 64, 300):
            f = rules.fold(1, nb, npairs, CUS)
            assert sorted(r if r < f else nb - 1 - (r - f) for r in range(nb)) == list(range(nb))


def test_chunks_cover_every_pair(rules):
    for npairs in (1, 7, 64, 500, 5000):
        for nranks in (1, 2, 9, 64, 700):
            for resident in (0, CUS, 2 * CUS):
                assert 1 <= rules.chunk(npairs, nranks, resident) <= max(npairs, 8)


def test_blocks_see(rules):
    """blocks_see against a count block by block."""
    lengths = (1, 31, 64, 65, 127, 128, 200, 256, 384, 500, 512, 1000)
    for nq in lengths:
        for nk in lengths:
            for causal in (0, 1, 2):
                coff = nk - nq if causal == 2 else 0
                for rows in (64, 128, 256):
                    if causal:
                        by_query = [min(nk, max(0, q0 + rows + coff)) for q0 in range(0, nq, rows)]
                        by_key = [nq - min(nq, max(0, k0 - coff)) for k0 in range(0, nk, rows)]
                    else:
                        by_query, by_key = [nk] * -(-nq // rows), [nq] * -(-nk // rows)
                    assert rules.sees(causal, nq, nk, rows, 0) == sum(by_query), (causal, nq, nk, rows)
                    assert rules.sees(causal, nq, nk, rows, 1) == sum(by_key), (causal, nq, nk, rows)


def test_near_square(rules):
    for parts in (3, 4, 16):
        assert rules.near_square(1, 700, 700, parts) and rules.near_square(2, 700, 700, parts)
        assert rules.near_square(1, 300, 5000, parts)  # top-left: keys past the last query are seen by none
        assert rules.near_square(2, 5000, 300, parts)  # bottom-right: the first queries see nothing
        assert rules.near_square(1, 480 + 480 // parts, 480, parts)
        assert not rules.near_square(1, 481 + 480 // parts, 480, parts)
        assert not rules.near_square(2, 480, 481 + 480 // parts, parts)
        assert not rules.near_square(0, 700, 700, parts)


# n_q, n_k, causal, whether stage 1 at D = 64 takes the fused kernel
STAGE1 = [
    (256, 256, 1, True), (384, 384, 1, True), (448, 448, 1, True), (1, 1, 1, True), (448, 512, 2, True),
    (400, 500, 2, True), (32, 512, 2, True), (200, 512, 1, True), (512, 200, 2, True),
    (512, 512, 1, False), (500, 500, 1, False), (513, 513, 1, False), (256, 512, 2, False), (128, 512, 2, False),
    (512, 128, 1, False), (512, 256, 1, False), (512, 448, 1, False), (256, 128, 1, False), (384, 512, 2, False),
    (256, 256, 0, False), (64, 600, 2, False),
]


@pytest.mark.parametrize("row", STAGE1, ids=str)
def test_stage1_fused(rules, row):
    nq, nk, causal, want = row
    assert bool(rules.stage1_fused(causal, nq, nk)) == want


# batch, n_q, n_k, heads, causal: the dQ kernel
DQ = [
    (64, 512, 1024, 12, 2, "compiled"), (32, 512, 4096, 12, 2, "compiled"),
    (8, 512, 8192, 16, 2, "q64"),
    (64, 512, 640, 12, 2, "compiled"), (64, 256, 512, 12, 2, "compiled"), (128, 512, 512, 12, 1, "compiled"),
    (1, 512, 512, 12, 1, "pair"), (2, 512, 2048, 12, 2, "pair"), (1, 512, 4096, 12, 1, "pair"),
    (2, 512, 4096, 12, 2, "compiled"), (16, 443, 4058, 2, 2, "compiled"), (1, 8192, 8192, 2, 1, "compiled"),
    (16, 4096, 512, 12, 2, "q64"), (32, 2048, 512, 12, 2, "q64"),
    (32, 1024, 512, 16, 1, "q64"), (32, 1024, 512, 8, 1, "q64"), (32, 1500, 1500, 12, 1, "compiled"),
]


@pytest.mark.parametrize("row", DQ, ids=str)
def test_dq(rules, row):
    batch, nq, nk, heads, causal, want = row
    assert dq(rules, causal, nq, nk, batch * heads) == want
    small = -(-nq // 64) * batch * heads <= CUS
    assert (dq(rules, causal, nq, nk, batch * heads, 128) == "pair") == small


# batch, n_q, n_k, heads, causal: whether dK/dV's 256-row kernel may run
K64 = [
    (32, 2117, 2117, 16, 1, True), (8, 3200, 3200, 12, 1, True), (4, 4096, 1024, 12, 1, True),
    (32, 2048, 1024, 12, 1, True), (32, 1280, 1024, 12, 1, True), (2, 8192, 4096, 12, 1, True),
    (64, 1030, 1030, 12, 1, False), (64, 1000, 1000, 12, 1, False), (64, 512, 256, 16, 1, False),
    (64, 600, 600, 16, 0, False), (8, 2048, 2048, 10, 0, False), (8, 2048, 2048, 16, 0, True),
]


@pytest.mark.parametrize("row", K64, ids=str)
def test_k64(rules, row):
    batch, nq, nk, heads, causal, want = row
    assert bool(rules.bwd_k64(causal, nq, nk, batch * heads, CUS)) == want


# batch, n_q, n_k, heads, causal: the dK/dV kernel
DKDV = [
    (8, 8192, 1024, 16, 1, "k64"), (16, 4096, 512, 16, 1, "k64"),
    (32, 1280, 1024, 12, 1, "k64"), (32, 1024, 512, 16, 1, "k64"), (32, 768, 1024, 12, 2, "k64"),
    (64, 768, 512, 12, 1, "compiled"), (64, 400, 600, 12, 2, "pair"), (64, 256, 512, 12, 2, "pair"),
    (32, 2048, 512, 12, 2, "pair"), (128, 512, 512, 12, 1, "pair"), (32, 1024, 1024, 16, 1, "pair"),
    (64, 1000, 1000, 12, 1, "pair"), (32, 1100, 1100, 16, 1, "compiled"),
    (2, 8192, 2048, 12, 1, "k64"), (4, 4096, 1024, 12, 1, "k64"), (1, 1024, 4096, 12, 2, "k64"),
    (2, 3072, 2048, 12, 1, "pair"), (2, 8192, 2048, 8, 1, "pair"),
    (16, 512, 4096, 12, 1, "k64"), (32, 512, 2048, 12, 1, "k64"), (32, 1024, 2048, 12, 1, "k64"),
]


@pytest.mark.parametrize("row", DKDV, ids=str)
def test_dkdv(rules, row):
    batch, nq, nk, heads, causal, want = row
    assert dkdv(rules, causal, nq, nk, batch * heads) == want


def test_dkdv_short_squares(rules):
    """Square causal problems of up to 1024 tokens run the pair kernel on any grid."""
    for n in range(1, 1025):
        assert rules.bwd_pair(1, n, n, 4000, CUS) and rules.bwd_pair(2, n, n, 4000, CUS), n


# batch, n_q, n_k, heads, causal: waves per SIMD of dK/dV's pair kernel, 2-byte D = 64
DKDV_WAVES = [
    (1, 4096, 4096, 12, 1, 2), (2, 2048, 2048, 12, 2, 2), (2, 2048, 2048, 16, 1, 4), (2, 2176, 2048, 12, 1, 2),
    (2, 2560, 2048, 12, 1, 4), (2, 4096, 2048, 12, 1, 4), (2, 1024, 2048, 12, 2, 4), (2, 4096, 2048, 8, 1, 2),
    (2, 2048, 2048, 12, 0, 4), (1, 2048, 2048, 16, 0, 2),
]


@pytest.mark.parametrize("row", DKDV_WAVES, ids=str)
def test_dkdv_waves(rules, row):
    batch, nq, nk, heads, causal, want = row
    assert rules.bwd_waves(causal, nq, nk, batch * heads, 64, 2, CUS) == want


# batch, n_q, n_k, heads, causal: whether stage 2 at D = 64 takes its pair kernel
STAGE2 = [
    (2, 2048, 2048, 12, 1, True), (2, 2560, 2048, 12, 1, True), (2, 1792, 2048, 12, 2, True),
    (2, 4096, 2048, 8, 1, True), (1, 8192, 2048, 12, 1, True),
    (2, 3072, 2048, 12, 1, False), (2, 8192, 2048, 12, 1, False), (2, 1024, 2048, 12, 2, False),
    (1, 1024, 8192, 6, 2, False), (2, 4096, 2048, 10, 1, False), (2, 2048, 2048, 16, 1, False),
    (1, 2048, 2048, 8, 0, True), (1, 2048, 2048, 12, 0, False),
]


@pytest.mark.parametrize("row", STAGE2, ids=str)
def test_stage2_pair(rules, row):
    batch, nq, nk, heads, causal, want = row
    assert bool(rules.stage2_pair(causal, nq, nk, batch * heads, CUS)) == want


# batch, n_q, n_k, heads, causal: `pairs` of stage 2's one-wave kernel
STAGE2_ORDER = [
    (1, 8192, 8192, 8, 1, 1), (2, 4096, 4096, 8, 1, 1), (1, 8192, 8192, 8, 2, 1), (1, 6144, 8192, 8, 1, 1),
    (2, 16384, 4096, 8, 1, 0), (2, 5120, 4096, 8, 1, 0), (2, 2048, 4096, 8, 2, 0), (4, 512, 4096, 4, 2, 0),
    (1, 9216, 8192, 8, 1, 0), (2, 4096, 4096, 9, 1, 0), (2, 4096, 4096, 15, 1, 1), (4, 2048, 2048, 15, 1, 1),
    (7, 1200, 2500, 7, 2, 0), (31, 4096, 2048, 2, 1, 0), (31, 2400, 2048, 2, 1, 1),
    (4, 2048, 2048, 14, 1, 0), (4, 2048, 2048, 17, 1, 0), (4, 2048, 2048, 16, 1, 2), (3, 2048, 2048, 12, 1, 0),
    # several whole rounds: neither order chunked, the single blocks only, both
    (128, 256, 256, 16, 1, 1), (64, 512, 512, 8, 1, 1), (16, 1024, 1024, 16, 1, 0), (8, 2048, 2048, 16, 1, 0),
    (192, 256, 256, 16, 1, 1), (96, 384, 384, 16, 1, 1), (128, 512, 512, 12, 1, 0), (96, 512, 512, 16, 1, 0),
    (64, 768, 768, 16, 1, 0), (1, 32768, 32768, 8, 1, 0),
    (384, 256, 256, 16, 1, 1), (160, 512, 512, 16, 1, 1), (96, 1024, 1024, 16, 1, 1), (64, 1536, 1536, 16, 1, 1),
    (64, 2048, 2048, 16, 1, 0),
    # half of the key blocks and more see no query
    (9, 2325, 16384, 4, 1, 1), (13, 1664, 11392, 8, 1, 1),
    (16, 512, 4096, 12, 1, 1), (32, 1024, 2048, 12, 1, 1), (8, 1024, 2048, 16, 1, 0), (32, 1500, 2048, 12, 1, 0),
    (4, 2048, 2048, 8, 1, 0), (1, 8192, 8192, 8, 0, 0),
]


@pytest.mark.parametrize("row", STAGE2_ORDER, ids=str)
def test_stage2_order(rules, row):
    batch, nq, nk, heads, causal, want = row
    assert stage2_order(rules, causal, nq, nk, batch * heads) == want


def test_folded_percent(rules):
    """Against the two blocks on each CU of a folded grid of two workgroups per CU."""
    for nq in (64, 512, 1024, 4096):
        for nk in (64, 512, 1024, 4096):
            for causal in (1, 2):
                coff = nk - nq if causal == 2 else 0
                see = sorted((min(nk, max(0, q0 + 64 + coff)) for q0 in range(0, nq, 64)), reverse=True)
                busiest = max(a + b for a, b in zip(see, reversed(see)))
                want = 100 * (busiest - (64 if nq > 64 else 0)) / max(see)  # a block's own 64 rows
                got = rules.folded_percent(causal, nq, nk)
                assert abs(got - want) <= 100 * 128 / max(see) or nq == 64, (nq, nk, causal, got, want)
    assert rules.folded_percent(0, 512, 512) == 200


# batch, n_q, n_k, heads, head_dim, causal: whether the fp32 forward takes its pair kernel
FORWARD = [
    (2, 2048, 2048, 8, 64, 1, True), (4, 2048, 2048, 8, 64, 1, True), (4, 2048, 2048, 16, 64, 1, False),
    (4, 1024, 2048, 8, 64, 2, True), (4, 1536, 1024, 8, 64, 1, True), (8, 1024, 1152, 8, 64, 2, True),
    (4, 512, 2048, 8, 64, 2, True), (1, 4096, 512, 4, 64, 1, True),
    (8, 512, 4096, 8, 64, 2, False), (16, 512, 4096, 8, 64, 2, False), (4, 2048, 1024, 4, 64, 1, False),
    (8, 1024, 1280, 8, 64, 2, False), (4, 4096, 2048, 4, 64, 1, False),
    (3, 2048, 2048, 8, 128, 1, True), (8, 512, 4096, 8, 128, 2, True), (4, 1024, 2048, 8, 128, 2, True),
    (4, 1280, 1024, 8, 128, 1, True), (4, 1536, 1024, 8, 128, 1, False), (6, 1024, 2048, 8, 128, 2, False),
    (4, 2048, 1024, 4, 128, 1, False), (4, 2048, 2048, 8, 128, 1, False),
    (1, 2048, 2048, 8, 64, 0, True), (2, 2048, 2048, 8, 64, 0, False),
]


@pytest.mark.parametrize("row", FORWARD, ids=str)
def test_forward(rules, row):
    batch, nq, nk, heads, d, causal, want = row
    assert bool(rules.fwd_pair(causal, nq, nk, batch * heads, d, CUS)) == want


# batch, n_q, n_k, heads, causal: whether the fp32 stage 1 takes its pair kernel
STAGE1_FP32 = [
    (2, 2048, 2048, 8, 1, True), (4, 768, 1024, 10, 2, True), (4, 1280, 1024, 6, 1, True), (4, 512, 512, 8, 2, True),
    (1, 2048, 1024, 8, 1, True), (1, 2048, 2048, 8, 0, True),
    (8, 512, 4096, 8, 2, False), (4, 2048, 1024, 4, 1, False), (4, 1536, 1024, 5, 1, False),
    (4, 2048, 2048, 8, 1, False), (2, 2048, 2048, 8, 0, False),
]


@pytest.mark.parametrize("row", STAGE1_FP32, ids=str)
def test_stage1_fp32(rules, row):
    batch, nq, nk, heads, causal, want = row
    assert bool(rules.stage1_qpair(causal, nq, nk, batch * heads, CUS)) == want


# batch, n_q, n_k, heads, causal: whether stage 1's 32-query kernel deals its blocks
DEAL = [
    (1, 512, 512, 12, 1, True), (4, 1024, 1024, 12, 1, True), (24, 1024, 1024, 12, 1, True),
    (1, 8192, 8192, 12, 1, True), (8, 1500, 1500, 12, 1, True), (3, 2048, 2048, 12, 1, True),
    (40, 1024, 1024, 12, 1, False), (2, 2048, 2048, 12, 1, False), (1, 4096, 4096, 12, 1, False),
    (32, 1024, 1024, 12, 1, False), (4, 2048, 2048, 16, 1, False),
    (7, 1024, 8192, 12, 2, True), (12, 600, 3000, 12, 2, True), (6, 4096, 1024, 12, 1, True),
    (13, 900, 2000, 12, 2, True), (1, 8192, 4096, 12, 1, True), (24, 2048, 1024, 12, 2, True),
    (9, 1500, 3000, 10, 2, True), (9, 3000, 1500, 10, 1, True), (32, 2048, 512, 12, 2, True),
    (35, 1664, 768, 16, 2, False), (66, 1152, 128, 4, 2, False), (487, 681, 681, 1, 1, False),
    (16, 640, 640, 16, 1, False),
    (28, 1024, 4096, 12, 2, False), (4, 1024, 4096, 10, 2, False), (4, 1024, 8192, 12, 2, False),
    (3, 1024, 8192, 16, 2, False), (2, 5000, 1000, 12, 1, False), (32, 1024, 4096, 12, 2, False),
    (3, 2048, 2048, 12, 0, False),
]


@pytest.mark.parametrize("row", DEAL, ids=str)
def test_deal(rules, row):
    batch, nq, nk, heads, causal, want = row
    assert bool(rules.q32_deal(causal, nq, nk, batch * heads, CUS)) == want


# batch, n_q, n_k, rows blocked, heads, causal: `pairs` of the kernels with 256-row blocks
ONE_WAVE_ORDER = [
    (4, 2048, 2048, 2048, 16, 1, 1), (8, 2048, 2048, 2048, 12, 1, 0), (16, 1536, 1536, 1536, 16, 1, 1),
    (2, 2048, 2048, 2048, 16, 1, 0), (24, 2048, 2048, 2048, 16, 1, 1), (4, 2048, 2048, 2048, 16, 0, 0),
]


@pytest.mark.parametrize("row", ONE_WAVE_ORDER, ids=str)
def test_one_wave_order(rules, row):
    batch, nq, nk, n, heads, causal, want = row
    assert one_wave_order(rules, causal, nq, nk, n, batch * heads) == want


def _walk(causal, nq, nk, npairs):
    """The most keys that a workgroup sweeps in the folded and in the dealt list, walked as the kernel does."""
    coff = nk - nq if causal == 2 else 0
    nqb = -(-nq // 128)
    npr = (nqb + 1) // 2
    keys = [min(nk, max(0, (i + 1) * 128 + coff)) for i in range(nqb)]
    item = [keys[nqb - 1 - r] + (keys[r] if 2 * r + 1 != nqb else 0) for r in range(npr)]
    n = npairs * npr
    folded = max(sum(item[i % npr] for i in range(w, n, CUS)) for w in range(min(CUS, n)))
    n = npairs * nqb
    grid = min(CUS, n)
    dealt = [0] * grid
    for k in range(-(-n // grid)):
        for w in range(grid):
            i = k * grid + (((grid // 8 - 1 - w // 8) * 8 + w % 8 if grid % 8 == 0 else grid - 1 - w) if k % 2 else w)
            if i < n:
                dealt[w] += keys[nqb - 1 - i // npairs]
    return folded, max(dealt)


def test_q32_load(rules):
    """The estimate of the rule is the walk's: exactly for folded lists of up to 4096 steps, to the
    reversed groups of eight workgroups (a block more or less in the last round) for dealt ones."""
    rng = random.Random(3)
    for _ in range(300):
        causal, nq, npairs = rng.choice((1, 2)), rng.randint(1, 40) * 128, rng.randint(1, 400)
        nk = nq if rng.random() < 0.3 else rng.randint(1, 40) * 128
        if npairs * nq // 128 <= CUS:
            continue
        folded, dealt = _walk(causal, nq, nk, npairs)
        got = rules.q32_folded(causal, nq, nk, npairs, CUS), rules.q32_dealt(causal, nq, nk, npairs, CUS)
        npr = (nq // 128 + 1) // 2
        if npr * (-(-npairs * npr // CUS)) <= 4096:
            assert got[0] == folded, (causal, nq, nk, npairs)
        assert abs(got[0] - folded) <= 0.05 * folded + nq, (causal, nq, nk, npairs, got, folded)
        assert abs(got[1] - dealt) <= 0.05 * dealt + 128, (causal, nq, nk, npairs, got, dealt)


# batch, n_q, n_k, heads, causal: pairs of waves per workgroup of the D = 128 stage 1
STAGE1_PAIRS = [
    (1, 1024, 1024, 8, 1, 2), (1, 2048, 2048, 8, 0, 2), (64, 64, 64, 16, 1, 2), (16, 300, 300, 12, 1, 2),
    (64, 128, 128, 16, 1, 2), (84, 1288, 169, 8, 2, 2), (23, 327, 100, 8, 1, 2),
    (64, 256, 256, 16, 1, 4), (32, 512, 512, 16, 1, 4), (2, 2048, 2048, 32, 1, 4), (2, 8192, 8192, 16, 1, 4),
    (4, 2048, 2048, 16, 0, 4), (64, 256, 256, 16, 0, 4), (64, 256, 1024, 8, 2, 4),
]


@pytest.mark.parametrize("row", STAGE1_PAIRS, ids=str)
def test_stage1_pairs(rules, row):
    batch, nq, nk, heads, causal, want = row
    assert rules.stage1_pairs(causal, nq, nk, batch * heads, CUS) == want
