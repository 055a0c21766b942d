"""GPU parity of the GEMM for more than 32 activation rows (mmfw.hip.inc: gq_mmf_*_w1 .. _w4 and
their one-plane forms) at the sizes where it can go wrong: the edges of its tiles of 32 to 128
activation rows and 256 weight rows, slices of K, the short last group of a Q8_0 row, rows of zeros
and non-finite rows, 16-bit elements against f32, passes of fewer rows than the call has."""
import numpy as np
import pytest

from gllm_amd.synth import random_activations, random_weight
from tests.test_gpu_parity import check_close, gpu_matmul

pytestmark = pytest.mark.gpu

Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14
ALL = [Q4_K, Q5_K, Q6_K, Q8_0]


@pytest.fixture(scope="module")
def torch():
    import torch
    return torch


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("tiles, ksplit", [(1, 0), (1, 3), (2, 1), (3, 2), (4, 1), (4, 5)])
def test_tile_edges(torch, oracle, dtype, tiles, ksplit):
    from gllm_amd.backend import ACT_BF16, HipBackend
    from oracle import npref
    hip = HipBackend(0, options={"mmfw_mt": tiles, "mmfw_ksplit": ksplit})
    for m, n, k in ((33, 257, 1280), (32 * tiles + 1, 40, 256), (131, 300, 768 + 64), (128, 255, 1504)):
        for bf16 in (False, True):
            print(f"wide gemm dtype={dtype} tiles={tiles} ksplit={ksplit} m={m} n={n} k={k} bf16={bf16}", flush=True)
            w, x = random_weight(dtype, n, k, seed=m + n), random_activations(m, k, seed=k + m)
            x[m - 1] = 0.0
            want = oracle.quantized_matmul(w, npref.bf16_rne(x) if bf16 else x, dtype, m, n, k, acc=oracle.ACC_F64, threads=16)
            got = gpu_matmul(hip, torch, w, x, dtype, m, n, k, **({"act_mode": ACT_BF16} if bf16 else {}))
            assert hip.last_kernel_name() == "gq_mmf_reduce" or "_w" in hip.last_kernel_name(), hip.last_kernel_name()
            check_close(got, want, f"dtype={dtype} m={m} n={n} k={k} bf16={bf16}")


@pytest.mark.parametrize("dtype", ALL)
def test_non_finite_rows_stay_in_their_rows(torch, oracle, dtype):
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0)
    m, n, k = 70, 300, 1024
    w, x = random_weight(dtype, n, k, seed=1), random_activations(m, k, seed=2)
    want = oracle.quantized_matmul(w, x, dtype, m, n, k, acc=oracle.ACC_F64, threads=16)
    x[3, 700], x[65, 0] = np.inf, np.nan
    got = gpu_matmul(hip, torch, w, x, dtype, m, n, k)
    assert not np.isfinite(got[[3, 65]]).any()
    keep = np.delete(np.arange(m), [3, 65])
    check_close(got[keep], want[keep], f"dtype={dtype}")


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("elem", ["float16", "bfloat16"])
def test_one_plane_gives_the_bits_of_two(torch, dtype, elem):
    """16-bit activations leave nothing for the lo plane: y is the rounded f32 result, bit for bit,
    for values over the whole range of the element type."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0, options={"mmfw_mt": 2, "mmfw_ksplit": 2})
    m, n, k = 67, 270, 1024
    t = getattr(torch, elem)
    w = torch.from_numpy(random_weight(dtype, n, k, seed=5)).cuda()
    x = torch.from_numpy(random_activations(m, k, seed=6)).cuda()
    x *= torch.exp2(torch.randint(-20, 3, x.shape, device="cuda").float())
    x16 = x.to(t)
    y16, y32 = torch.zeros(m, n, dtype=t, device="cuda"), torch.zeros(m, n, device="cuda")
    hip.quantized_matmul(w, x16, y16, dtype, m, n, k)
    hip.quantized_matmul(w, x16.float(), y32, dtype, m, n, k)
    torch.cuda.synchronize()
    assert torch.equal(y16.view(torch.int16), y32.to(t).view(torch.int16))


@pytest.mark.parametrize("dtype", [Q4_K, Q8_0])
def test_passes_of_fewer_rows(torch, dtype):
    """The entry point with scratch of a fixed size takes a prompt in passes: the same bits."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0)
    m, n, k = 700, 520, 14336
    w = torch.from_numpy(random_weight(dtype, n, k, seed=7)).cuda()
    x = torch.from_numpy(random_activations(m, k, seed=8)).cuda()
    want, got = torch.zeros(m, n, device="cuda"), torch.full((m, n), float("nan"), device="cuda")
    hip.quantized_matmul(w, x, want, dtype, m, n, k)
    hip.quantized_matmul_noalloc(w, x, got, dtype, m, n, k)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
