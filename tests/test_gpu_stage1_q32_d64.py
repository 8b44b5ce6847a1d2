"""The 32-query stage 1 at D = 64 (fhog_bwdbwd_q32.hip) on every small case.

Short causal problems run the fused kernel by default (stage1_fused_rule), so
the small causal cases of the parity, scale, single-key and random-sweep suites
would not reach the 32-query kernel; here they run again with
FLASH_HOG_STAGE1=q32, at the same tolerances.
"""

from __future__ import annotations

import pytest
import torch

import test_gpu_parity as parity
import test_gpu_sweep as sweep

pytestmark = pytest.mark.gpu


@pytest.fixture
def q32(monkeypatch):
    monkeypatch.setenv("FLASH_HOG_STAGE1", "q32")


def _two_byte_d64(cases, dim, dtype):
    return [c for c in cases if c[dim] == 64 and c[dtype] in (torch.bfloat16, torch.float16)]


CASES = _two_byte_d64(parity.CASES, 6, 7)
SCALE_CASES = _two_byte_d64(parity.SCALE_CASES, 6, 7)
SINGLE_KEY_CASES = _two_byte_d64(parity.SINGLE_KEY_CASES, 6, 7)
PROBLEMS = _two_byte_d64(sweep.PROBLEMS, 6, 7)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_q32_bwdbwd_matches_oracle(case, cuda_device, q32):
    parity.test_bwdbwd_matches_oracle(case, cuda_device)


@pytest.mark.parametrize("case", SCALE_CASES, ids=[c[0] for c in SCALE_CASES])
def test_q32_other_scales(case, cuda_device, q32):
    parity.test_all_kernels_other_scales(case, cuda_device)


@pytest.mark.parametrize("case", SINGLE_KEY_CASES, ids=[c[0] for c in SINGLE_KEY_CASES])
def test_q32_single_key_rows_are_exact(case, cuda_device, q32):
    parity.test_single_key_rows_are_exact(case, cuda_device)


@pytest.mark.parametrize("problem", PROBLEMS, ids=[p[0] for p in PROBLEMS])
def test_q32_random_problem(problem, cuda_device, q32):
    sweep.test_random_problem_all_kernels(problem, cuda_device)
