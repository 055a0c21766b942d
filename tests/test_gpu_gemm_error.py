"""The wide GEMM's error against 64 bits (mmfw.hip.inc) is no larger than that of the 64-row passes of the other
forms (option mmfw=0) on the same inputs: f32 activations and f32 activations rounded to bf16, the row tiles and
slices that the shape gets and every number of row tiles."""
import numpy as np
import pytest

from gllm_amd.synth import random_activations, random_weight

pytestmark = pytest.mark.gpu

Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14

# Root mean squares over 1e5 outputs and more, which share rows of weights and of activations: their ratio is good to about 1 %.
SPREAD = 1.03


@pytest.fixture(scope="module")
def torch():
    import torch
    return torch


def errors(torch, dtype, m, n, k, bf16, tiles):
    """Relative error of the 64-row passes, then of the wide GEMM for each entry of `tiles` (0: by the shape)."""
    from gllm_amd.backend import ACT_BF16, ACT_F32_SPLIT, HipBackend
    w = torch.from_numpy(random_weight(dtype, n, k, seed=m + n).view(np.uint8).reshape(-1)).cuda()
    x = torch.from_numpy(random_activations(m, k, seed=k)).cuda()
    plain = HipBackend(0)
    deq = torch.zeros(n, k, device="cuda")
    plain.dequantize(w, deq, dtype)
    want = (x.bfloat16() if bf16 else x).double() @ deq.double().t()
    found = []
    for options in [{"mmfw": 0}] + [{"mmfw_mt": t, "mmfw_min_m": 9} for t in tiles]:
        hip, y = HipBackend(0, options=options), torch.full((m, n), float("nan"), device="cuda")
        hip.quantized_matmul(w, x, y, dtype, m, n, k, act_mode=ACT_BF16 if bf16 else ACT_F32_SPLIT)
        found.append(float((y.double() - want).norm() / want.norm()))
    return found


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("m, n, k", [(64, 2000, 2048), (200, 14336, 1024), (130, 1000, 1280)])
def test_q6_k(torch, m, n, k, bf16):
    before, *here = errors(torch, Q6_K, m, n, k, bf16, (0, 1, 2, 3, 4))
    print(f"q6_k {m} {n} {k} bf16={bf16}: {before:.3e} here {[f'{e:.3e}' for e in here]}", flush=True)
    assert max(here) <= SPREAD * before


@pytest.mark.parametrize("dtype", [Q6_K, Q8_0])
@pytest.mark.parametrize("m, n, k", [(200, 14336, 4096), (2048, 4096, 14336), (300, 28672, 2560)])
def test_long_rows(torch, dtype, m, n, k):
    """Many blocks in one slice of K: their sums are taken in runs."""
    for bf16 in (False, True):
        before, *here = errors(torch, dtype, m, n, k, bf16, (0, 1, 2, 3))
        print(f"{dtype} {m} {n} {k} bf16={bf16}: {before:.3e} here {[f'{e:.3e}' for e in here]}", flush=True)
        assert max(here) <= SPREAD * before


@pytest.mark.parametrize("dtype", [Q4_K, Q5_K])
@pytest.mark.parametrize("m, n, k", [(64, 2000, 2048), (512, 14336, 4096), (1024, 4096, 14336)])
def test_q4_k_q5_k(torch, dtype, m, n, k):
    """Up to three row tiles with sums of their own for the lo plane's products, four with those ahead of the others."""
    before, *here = errors(torch, dtype, m, n, k, False, (0, 1, 2, 3, 4))
    print(f"{dtype} {m} {n} {k}: {before:.3e} here {[f'{e:.3e}' for e in here]}", flush=True)
    assert max(here) <= SPREAD * before
