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


@pytest.mark.parametrize("dtype", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("tiles", [1, 2])
@pytest.mark.parametrize("blocks", [1, 3, 4, 5, 8, 9])
def test_weights_in_units(torch, oracle, dtype, tiles, blocks):
    """Whole rows of one or two blocks of K at a time: an odd block left over, one block in all, rows past the last one, a last
    block that K does not fill; a matrix that ends with its allocation."""
    from gllm_amd.backend import ACT_BF16, HipBackend
    from oracle import npref
    hip = HipBackend(0, options={"mmfw_mt": tiles, "mmfw_ksplit": 1})
    for m, n, k in ((33, 257, 256 * blocks), (40, 1, 256 * blocks - 192)):
        for bf16 in (False, True):
            print(f"units dtype={dtype} tiles={tiles} m={m} n={n} k={k} bf16={bf16}", flush=True)
            w, x = random_weight(dtype, n, k, seed=m + n), random_activations(m, k, seed=k + m)
            want = oracle.quantized_matmul(w, npref.bf16_rne(x) if bf16 else x, dtype, m, n, k, acc=oracle.ACC_F64, threads=16)
            got = gpu_matmul(hip, torch, w, x, dtype, m, n, k, **({"act_mode": ACT_BF16} if bf16 else {}))
            check_close(got, want, f"dtype={dtype} m={m} n={n} k={k} bf16={bf16}")


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("elem", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("slices, blocks", [(1, 1), (1, 2), (1, 3), (1, 4), (1, 5), (2, 2), (2, 3), (3, 3), (3, 4)])
def test_images_made_by_the_workgroup(torch, dtype, elem, slices, blocks):
    """Short slices of K, whose workgroups prepare their activations themselves: the bits of the launch that prepares them, with
    blocks that K does not fill, a slice shorter than the rest, rows past the last, rows of zeros, tiny, huge and non-finite ones,
    several matrices; blocks that do not fit take the launch."""
    from gllm_amd.backend import HipBackend
    t = getattr(torch, elem)
    hips = [HipBackend(0, options={"mmfw_mt": 1, "mmfw_ksplit": slices, "mmfw_min_m": 9, "mmfw_own": v}) for v in (1, 0)]
    k = 256 * slices * blocks - (256 if slices > 1 and blocks > 1 else 0)
    for m, cut in ((33, 0), (9, 32 if dtype == Q8_0 and k > 256 else 0), (64, 224 if dtype == Q8_0 and k > 256 else 0)):
        x = torch.from_numpy(random_activations(m, k - cut, seed=k + m)).cuda()
        x[0] = 0.0
        x[1] *= 1e-30
        x[2] *= 2.0 ** 100
        x[3, 5], x[m - 1, 0] = float("nan"), float("inf")
        x = x.to(t)
        sizes = (257, 64, 1)
        ws = [torch.from_numpy(random_weight(dtype, n, k - cut, seed=n)).cuda() for n in sizes]
        outs = []
        for hip in hips:
            print(f"own images dtype={dtype} {elem} slices={slices} blocks={blocks} m={m} k={k - cut}", flush=True)
            ys = [torch.full((m, n), 7.0, device="cuda", dtype=t) for n in sizes]
            own = hip is hips[0] and blocks <= (4 if elem != "float32" else 2 if dtype == Q8_0 else 3)  # (slices: test_host_routes.py)
            hip.quantized_matmul(ws[0], x, ys[0], dtype, m, sizes[0], k - cut)
            assert slices > 1 or ("_w1_own" in hip.last_kernel_name()) == own, hip.last_kernel_name()
            hip.quantized_matmul_batch([(w, x, y, dtype, m, y.shape[1], k - cut) for w, y in list(zip(ws, ys))[1:]])
            assert slices > 1 or ("_w1_own" in hip.last_kernel_name()) == own, hip.last_kernel_name()
            torch.cuda.synchronize()
            outs.append(ys)
        for a, b in zip(*outs):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("elem", ["float32", "bfloat16"])
def test_outputs_over_the_activations(torch, dtype, elem):
    """A square matmul in place, of a size whose workgroups make their images themselves where the outputs lie elsewhere: the same
    bits."""
    from gllm_amd.backend import HipBackend
    t, hip = getattr(torch, elem), HipBackend(0, options={"mmfw_mt": 1, "mmfw_ksplit": 1})
    for m, k in ((64, 512), (200, 512)):
        print(f"in place dtype={dtype} {elem} m={m} k={k}", flush=True)
        w = torch.from_numpy(random_weight(dtype, k, k, seed=k)).cuda()
        x = torch.from_numpy(random_activations(m, k, seed=m)).cuda().to(t)
        y = torch.zeros_like(x)
        hip.quantized_matmul(w, x, y, dtype, m, k, k)
        assert "_own" in hip.last_kernel_name(), hip.last_kernel_name()
        hip.quantized_matmul(w, x, x, dtype, m, k, k)
        assert "_own" not in hip.last_kernel_name(), hip.last_kernel_name()
        torch.cuda.synchronize()
        assert torch.equal(x, y)


@pytest.mark.parametrize("dtype", [Q4_K, Q5_K])
@pytest.mark.parametrize("tiles", [2, 3, 4])
@pytest.mark.parametrize("run", [2, 3, 16])
def test_runs_of_weight_tiles(torch, dtype, tiles, run):
    """A workgroup takes several weight tiles one after the other, across matrices and up to a ragged last one: the bits of a
    tile per workgroup, for the shortest rows that allow it and longer ones."""
    from gllm_amd.backend import HipBackend
    one, several = (HipBackend(0, options={"mmfw_mt": tiles, "mmfw_ksplit": 1, "mmfw_run": r}) for r in (1, run))
    for m, k in ((65, 1024), (130, 1536 - 64), (200, 1280)):  # (the last: an odd number of blocks)
        x = torch.from_numpy(random_activations(m, k, seed=k)).cuda().to(torch.bfloat16)
        ws = [torch.from_numpy(random_weight(dtype, n, k, seed=n)).cuda() for n in (513, 256, 300)]
        outs = []
        for hip in (one, several):
            print(f"runs dtype={dtype} tiles={tiles} run={run} m={m} k={k}", flush=True)
            y = [torch.full((m, n), float("nan"), device="cuda", dtype=torch.bfloat16) for n in (513, 256, 300)]
            hip.quantized_matmul_batch([(w, x, o, dtype, m, o.shape[1], k) for w, o in zip(ws, y)])
            single = torch.full((m, 513), float("nan"), device="cuda", dtype=torch.bfloat16)
            hip.quantized_matmul(ws[0], x, single, dtype, m, 513, k)
            torch.cuda.synchronize()
            outs.append(y + [single])
        for a, b in zip(*outs):
            assert torch.equal(a, b) and bool(torch.isfinite(a.float()).all())


@pytest.mark.parametrize("tiles", [1, 2, 3])
@pytest.mark.parametrize("tail", [1, 3, 4, 5, 7, 8])
def test_q8_0_short_last_groups(torch, oracle, tiles, tail):
    """Quants are read ahead of a unit into a last group that holds `tail` blocks, windowed to end with the row."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0, options={"mmfw_mt": tiles, "mmfw_ksplit": 1})
    for m, n, groups in ((33, 257, 1), (97, 3, 3)):
        k = 256 * groups + 32 * tail
        print(f"q8_0 tail={tail} tiles={tiles} m={m} n={n} k={k}", flush=True)
        w, x = random_weight(Q8_0, n, k, seed=m + n), random_activations(m, k, seed=k + m)
        want = oracle.quantized_matmul(w, x, Q8_0, m, n, k, acc=oracle.ACC_F64, threads=16)
        check_close(gpu_matmul(hip, torch, w, x, Q8_0, m, n, k), want, f"m={m} n={n} k={k}")


@pytest.mark.parametrize("ksplit", [2, 4, 5, 8, 9, 15])
@pytest.mark.parametrize("m, n", [(33, 33), (34, 1), (35, 257), (36, 260)])
def test_sums_of_slices_at_any_place(torch, oracle, ksplit, m, n):
    """The sums over K slices go by fours of the m x n outputs in a row, wherever they start and end: outputs at every
    alignment of their type, a last few that are no four, nothing written around them; 16-bit outputs are the rounded f32 ones."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0, options={"mmfw_mt": 1, "mmfw_ksplit": ksplit})
    k = 256 * 15
    w, x = random_weight(Q4_K, n, k, seed=n), random_activations(m, k, seed=m).astype(np.float16).astype(np.float32)
    want = oracle.quantized_matmul(w, x, Q4_K, m, n, k, acc=oracle.ACC_F64, threads=16)
    wd, xd, f32 = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(), None
    for t in (torch.float32, torch.float16):
        for offset in ((0, 1, 3) if t is torch.float32 else (0, 2, 6)):  # (outputs are four-byte aligned)
            print(f"slices={ksplit} m={m} n={n} {t} offset={offset}", flush=True)
            buf = torch.full((offset + m * n + 64,), 7.0, dtype=t, device="cuda")
            hip.quantized_matmul(wd, xd.to(t), buf[offset:offset + m * n].view(m, n), Q4_K, m, n, k)
            torch.cuda.synchronize()
            got = buf[offset:offset + m * n].cpu().view(m, n)
            assert bool(torch.all(buf[:offset] == 7.0)) and bool(torch.all(buf[offset + m * n:] == 7.0))
            if f32 is None:
                check_close(got.numpy(), want, f"slices={ksplit} m={m} n={n}")
                f32 = got
            assert torch.equal(got, f32.to(t))


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
    """16-bit activations leave nothing for the lo plane: with the same tiles and slices y is the rounded f32 result, bit for
    bit, for values over 23 powers of two."""
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


@pytest.mark.parametrize("t_gu, t_dn, hidden, ffn, experts, top_k, tokens, elem", [
    (Q4_K, Q6_K, 512, 256, 4, 2, 70, "float32"),     # jobs of one and two tiles
    (Q5_K, Q4_K, 768, 520, 3, 2, 200, "bfloat16"),   # of four tiles and a fifth; a ragged ffn
    (Q8_0, Q8_0, 288, 352, 2, 1, 190, "float16"),    # short last groups; four tiles in two halves
    (Q6_K, Q5_K, 256, 256, 40, 8, 45, "float32"),    # few rows per tile
])
def test_experts_with_many_tokens(torch, oracle, t_gu, t_dn, hidden, ffn, experts, top_k, tokens, elem):
    """moe_matvec through the GEMM (from `moe_wide_min` pairs per expert up) against the oracle, with an
    expert nobody chose, routes dropped (length below top_k) and separate gate and up tensors."""
    from gllm_amd.backend import HipBackend
    from gllm_amd.ggml import row_bytes
    hip = HipBackend(0, options={"moe_wide_min": 1})
    rng = np.random.default_rng(tokens)
    gate = random_weight(t_gu, experts * ffn, hidden, seed=1)
    up = random_weight(t_gu, experts * ffn, hidden, seed=2)
    down = random_weight(t_dn, experts * hidden, ffn, seed=3)
    t = getattr(torch, elem)
    x = torch.from_numpy(random_activations(tokens, hidden, seed=4) * 1e-3).to(t)
    expert = np.stack([rng.permutation(max(1, experts - 1))[np.arange(top_k) % max(1, experts - 1)] for _ in range(tokens)]).astype(np.int32)
    weight = rng.uniform(0.1, 1.0, (tokens, top_k)).astype(np.float32)
    length = np.full(tokens, top_k, np.int32)
    length[::7] = max(1, top_k - 1)
    out = torch.full((tokens, hidden), float("nan"), dtype=t, device="cuda")
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    print(f"wide experts {t_gu}/{t_dn} hidden={hidden} ffn={ffn} tokens={tokens} {elem}", flush=True)
    hip.moe_matvec(dev(gate), t_gu, dev(down), t_dn, x.cuda(), out, hidden, ffn, experts, dev(expert), dev(weight), dev(length), up=dev(up))
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    xf = x.float().numpy()
    want = np.zeros((tokens, hidden), np.float64)
    gb, db = ffn * row_bytes(t_gu, hidden), hidden * row_bytes(t_dn, ffn)
    for e in range(experts):
        pairs = [(a, i) for a in range(tokens) for i in range(length[a]) if expert[a, i] == e]
        if not pairs:
            continue
        rows = oracle.ffn_swiglu(gate[e * gb:(e + 1) * gb], up[e * gb:(e + 1) * gb], t_gu, down[e * db:(e + 1) * db], t_dn,
                                 np.ascontiguousarray(xf[[a for a, _ in pairs]]), len(pairs), hidden, ffn, acc=oracle.ACC_F64, threads=16)
        for (a, i), r in zip(pairs, rows.reshape(len(pairs), hidden)):
            want[a] += weight[a, i] * r.astype(np.float64)
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert rel <= {"float32": 1e-5, "float16": 1e-3, "bfloat16": 5e-3}[elem], rel


def test_router_walks_from_the_first_token_without_a_place(torch, oracle):
    """Ranks in parallel up to the first token that loses all its choices, the serial walk from there:
    capacities from none to plenty, top_k that does not divide 64, more tokens than a wave's run."""
    from gllm_amd.backend import HipBackend
    from tests.test_gpu_route import check_against_oracle, route
    hip = HipBackend(0)
    rng = np.random.default_rng(5)
    for tokens, experts, top_k in ((65, 8, 2), (300, 16, 3), (777, 5, 5), (130, 128, 8), (1000, 600, 7), (90, 4, 8)):
        logits = rng.standard_normal((tokens, experts)).astype(np.float32)
        logits[:, 0] += 2.0  # a favourite
        for factor in (0.0, 0.4, 1.0, 1.25, 3.0, 1e9):
            print(f"route tokens={tokens} experts={experts} top_k={top_k} capacity={factor}", flush=True)
            got = route(hip, torch, logits, top_k, capacity_factor=factor)
            check_against_oracle(oracle, got, logits, top_k, factor, f"{tokens} {experts} {top_k} {factor}")


def element_bar(elem):
    """The rounding of the output to its type (2^-11, 2^-9 of a value at most), over the f32 bar."""
    return {"float32": 1e-5, "float16": 1e-3, "bfloat16": 5e-3}[elem]


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("elem", ["float32", "float16", "bfloat16"])
def test_nine_to_32_rows(torch, oracle, dtype, elem):
    """One row tile, where the streamed GEMMs do not take the call: few weight rows, Q6_K and Q8_0."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0)
    t = getattr(torch, elem)
    for m, n, k in ((9, 257, 1280), (16, 1000, 2080 if dtype == Q8_0 else 2048), (31, 40, 256), (32, 513, 4864)):
        print(f"one tile dtype={dtype} {elem} m={m} n={n} k={k}", flush=True)
        w, x = random_weight(dtype, n, k, seed=m + n), torch.from_numpy(random_activations(m, k, seed=k + m) * 1e-2).to(t)
        y = torch.full((m, n), float("nan"), dtype=t, device="cuda")
        hip.quantized_matmul(torch.from_numpy(w.view(np.uint8).reshape(-1)).cuda(), x.cuda(), y, dtype, m, n, k)
        assert hip.last_kernel_name() == "gq_mmf_reduce" or "_w1" in hip.last_kernel_name(), hip.last_kernel_name()
        want = oracle.quantized_matmul(w, x.float().numpy(), dtype, m, n, k, acc=oracle.ACC_F64, threads=16)
        rel = np.linalg.norm(y.float().cpu().numpy() - want) / np.linalg.norm(want)
        assert rel <= element_bar(elem), f"m={m} n={n} k={k}: {rel}"


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("m, elem", [(9, "float32"), (16, "bfloat16"), (33, "float16"), (100, "float32")])
def test_projections_as_one_launch(torch, oracle, dtype, m, elem):
    """Independent batch entries over the same rows: two and three of them (a fourth starts the next group), rows
    that fill no tile, an entry that waits for the ones before it, one with other activations; entries that write
    the same output stay apart and in order."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0)
    t, k = getattr(torch, elem), 1280
    sizes = [300, 40, 257, 33, 256, 70]
    host_x = [torch.from_numpy(random_activations(m, k, seed=s + m) * 1e-2).to(t) for s in (1, 2)]
    xs = [x.cuda() for x in host_x]
    which = [0, 0, 0, 0, 1, 1]
    ws = [random_weight(dtype, n, k, seed=n) for n in sizes]
    dev = [torch.from_numpy(w.view(np.uint8).reshape(-1)).cuda() for w in ws]
    ys = [torch.full((m, n), float("nan"), dtype=t, device="cuda") for n in sizes]
    entries = [(d, xs[i], y, dtype, m, n, k) for d, i, y, n in zip(dev, which, ys, sizes)]
    print(f"group dtype={dtype} m={m} {elem}", flush=True)
    hip.run_batch(hip.make_batch(entries, after_previous=lambda i: i == 2))
    torch.cuda.synchronize()
    for w, i, y, n in zip(ws, which, ys, sizes):
        want = oracle.quantized_matmul(w, host_x[i].float().numpy(), dtype, m, n, k, acc=oracle.ACC_F64, threads=16)
        rel = np.linalg.norm(y.float().cpu().numpy() - want) / np.linalg.norm(want)
        assert rel <= element_bar(elem), f"n={n}: {rel}"
    # the second writes over the first: not one launch, whose tiles would finish in any order
    twice = torch.full((m, 300), float("nan"), dtype=t, device="cuda")
    w2 = torch.from_numpy(random_weight(dtype, 300, k, seed=99).view(np.uint8).reshape(-1)).cuda()
    alone = torch.full((m, 300), float("nan"), dtype=t, device="cuda")
    hip.quantized_matmul(w2, xs[0], alone, dtype, m, 300, k)
    hip.run_batch(hip.make_batch([(dev[0], xs[0], twice, dtype, m, 300, k), (w2, xs[0], twice, dtype, m, 300, k)]))
    torch.cuda.synchronize()
    assert torch.equal(twice, alone)


def test_group_under_capture_keeps_to_the_reserved_scratch(torch):
    """What was reserved entry by entry serves the captured batch; replays, with eager work between them, give the
    results of the single calls (of the eager batch, bit for bit: test_captured_group_gives_the_eager_bits)."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0)
    m, k, sizes = 24, 1024, [512, 128, 128]
    x = torch.from_numpy(random_activations(m, k, seed=3)).cuda()
    dev = [torch.from_numpy(random_weight(Q4_K, n, k, seed=n + i).view(np.uint8).reshape(-1)).cuda() for i, n in enumerate(sizes)]
    ys = [torch.zeros(m, n, device="cuda") for n in sizes]
    batch = hip.make_batch([(d, x, y, Q4_K, m, n, k) for d, y, n in zip(dev, ys, sizes)])
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        hip.reserve_matmul(Q4_K, m, max(sizes), k)
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            hip.run_batch(batch)
    torch.cuda.synchronize()
    plain = HipBackend(0)
    for trial in range(3):
        x.copy_(torch.from_numpy(random_activations(m, k, seed=10 + trial)))
        for y in ys:
            y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for d, y, n in zip(dev, ys, sizes):
            want = torch.zeros(m, n, device="cuda")
            plain.quantized_matmul(d, x, want, Q4_K, m, n, k)
            torch.cuda.synchronize()
            # two orders of the same f32 sums
            assert float((y - want).norm() / want.norm()) <= 1e-6


@pytest.mark.parametrize("dtype", ALL)
def test_five_to_eight_rows(torch, oracle, dtype):
    """Long rows of more activation rows than one pass of the int8 kernels takes; a group of
    projections, and the feed-forward block, of as many rows."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0)
    passes = {Q4_K: 8, Q5_K: 7, Q6_K: 6, Q8_0: 6}[dtype]
    n, k = 4801, 10240 + 256  # (48 M weights and more)
    w = random_weight(dtype, n, k, seed=5)
    wd = torch.from_numpy(w.view(np.uint8).reshape(-1)).cuda()
    for elem in ("float32", "bfloat16"):
        t = getattr(torch, elem)
        for m in (4, 5, 6, 7, 8):
            print(f"few rows dtype={dtype} {elem} m={m}", flush=True)
            x = torch.from_numpy(random_activations(m, k, seed=m) * 1e-2).to(t)
            y = torch.full((m, n), float("nan"), dtype=t, device="cuda")
            hip.quantized_matmul(wd, x.cuda(), y, dtype, m, n, k)
            wide = m > passes
            assert (hip.last_kernel_name() == "gq_mmf_reduce" or "_w1" in hip.last_kernel_name()) == wide, hip.last_kernel_name()
            want = oracle.quantized_matmul(w, x.float().numpy(), dtype, m, n, k, acc=oracle.ACC_F64, threads=16)
            rel = np.linalg.norm(y.float().cpu().numpy() - want) / np.linalg.norm(want)
            assert rel <= element_bar(elem), f"m={m}: {rel}"
            hidden, ffn = 512, 768
            g, u, d = (random_weight(dtype, a, b, seed=i) for i, (a, b) in enumerate(((ffn, hidden), (ffn, hidden), (hidden, ffn))))
            xf = torch.from_numpy(random_activations(m, hidden, seed=m) * 1e-2).to(t)
            out = torch.full((m, hidden), float("nan"), dtype=t, device="cuda")
            dev = [torch.from_numpy(a.view(np.uint8).reshape(-1)).cuda() for a in (g, u, d)]
            hip.ffn_swiglu(dev[0], dev[1], dtype, dev[2], dtype, xf.cuda(), out, m, hidden, ffn)
            want = oracle.ffn_swiglu(g, u, dtype, d, dtype, xf.float().numpy(), m, hidden, ffn, acc=oracle.ACC_F64, threads=16)
            rel = np.linalg.norm(out.float().cpu().numpy() - want.reshape(m, hidden)) / np.linalg.norm(want)
            assert rel <= element_bar(elem), f"ffn m={m}: {rel}"
            ys = [torch.full((m, r), float("nan"), dtype=t, device="cuda") for r in (ffn, ffn)]
            xg = xf.cuda()
            hip.run_batch(hip.make_batch([(dev[0], xg, ys[0], dtype, m, ffn, hidden), (dev[1], xg, ys[1], dtype, m, ffn, hidden)]))
            for wi, yi in zip((g, u), ys):
                want = oracle.quantized_matmul(wi, xf.float().numpy(), dtype, m, ffn, hidden, acc=oracle.ACC_F64, threads=16)
                rel = np.linalg.norm(yi.float().cpu().numpy() - want) / np.linalg.norm(want)
                assert rel <= element_bar(elem), f"group m={m}: {rel}"


@pytest.mark.parametrize("dtype", ALL)
def test_projections_of_two_to_four_long_rows(torch, oracle, dtype):
    """Rows beyond what the streamed launch over several matrices takes: the GEMM from three rows on, in 16 bits from two."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0)
    k, sizes = 4352, [300, 40, 257]
    ws = [random_weight(dtype, n, k, seed=n) for n in sizes]
    dev = [torch.from_numpy(w.view(np.uint8).reshape(-1)).cuda() for w in ws]
    for elem in ("float32", "float16"):
        t = getattr(torch, elem)
        for m in (1, 2, 3, 4):
            print(f"long rows dtype={dtype} {elem} m={m}", flush=True)
            x = torch.from_numpy(random_activations(m, k, seed=m) * 1e-2).to(t)
            xd, ys = x.cuda(), [torch.full((m, n), float("nan"), dtype=t, device="cuda") for n in sizes]
            hip.run_batch(hip.make_batch([(d, xd, y, dtype, m, n, k) for d, y, n in zip(dev, ys, sizes)]))
            grouped = hip.last_kernel_name() == "gq_mmf_reduce"
            assert grouped == (m >= (2 if elem == "float16" else 3)), hip.last_kernel_name()
            for w, y, n in zip(ws, ys, sizes):
                want = oracle.quantized_matmul(w, x.float().numpy(), dtype, m, n, k, acc=oracle.ACC_F64, threads=16)
                rel = np.linalg.norm(y.float().cpu().numpy() - want) / np.linalg.norm(want)
                assert rel <= element_bar(elem), f"m={m} n={n}: {rel}"


def captured(torch, hip, stream, call, outputs):
    """The call captured on `stream`, replayed three times with eager work between: its outputs of every replay."""
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
        call()
    found = []
    for _ in range(3):
        for y in outputs:
            y.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        found.append([y.clone() for y in outputs])
    return found


@pytest.mark.parametrize("dtype, n, k, first, elem", [
    (Q4_K, 2000, 2048, 64, "float32"), (Q6_K, 14336, 1024, 512, "float32"), (Q8_0, 1280, 5120, 2048, "float32"), (Q5_K, 700, 1024, 33, "bfloat16")])
def test_capture_of_any_rows_behind_one_call(torch, dtype, n, k, first, elem):
    """A call of 33 rows and more, or a reserved one, leaves scratch for any number of rows: fewer, more (in passes), of the
    other element types, over other weight rows.  The captured call gives the eager bits."""
    from gllm_amd.backend import HipBackend
    plain, t = HipBackend(0), getattr(torch, elem)
    w = torch.from_numpy(random_weight(dtype, n, k, seed=5).view(np.uint8).reshape(-1)).cuda()
    x = torch.from_numpy(random_activations(2100, k, seed=6)).cuda()
    for reserve in (True, False):
        hip, stream = HipBackend(0), torch.cuda.Stream()
        with torch.cuda.stream(stream):
            if reserve:
                hip.reserve_matmul(dtype, first, n, k)
            else:
                y = torch.zeros(first, n, dtype=t, device="cuda")
                hip.quantized_matmul(w, x[:first].to(t), y, dtype, first, n, k)
        for m in (12, 33, 64, 65, 100, 129, 192, 700, 2100):
            for e in {torch.float32, t}:
                print(f"capture dtype={dtype} first={first} reserve={reserve} m={m} {e}", flush=True)
                xm, y, want = x[:m].to(e), torch.zeros(m, n, dtype=e, device="cuda"), torch.zeros(m, n, dtype=e, device="cuda")
                plain.quantized_matmul(w, xm, want, dtype, m, n, k)
                for got, in captured(torch, hip, stream, lambda: hip.quantized_matmul(w, xm, y, dtype, m, n, k), [y]):
                    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("m, elem", [(2, "bfloat16"), (4, "float32"), (24, "float32"), (24, "float16"), (70, "float32")])
def test_captured_group_gives_the_eager_bits(torch, dtype, m, elem):
    """Reserved entry by entry, a batch of projections is captured as the one launch that it is eagerly."""
    from gllm_amd.backend import HipBackend
    t, k, sizes = getattr(torch, elem), 4352, [512, 128, 130]
    x = torch.from_numpy(random_activations(m, k, seed=3)).cuda().to(t)
    dev = [torch.from_numpy(random_weight(dtype, n, k, seed=n + i).view(np.uint8).reshape(-1)).cuda() for i, n in enumerate(sizes)]
    ys, want = ([torch.zeros(m, n, dtype=t, device="cuda") for n in sizes] for _ in range(2))
    plain, hip, stream = HipBackend(0), HipBackend(0), torch.cuda.Stream()
    plain.run_batch(plain.make_batch([(d, x, y, dtype, m, n, k) for d, y, n in zip(dev, want, sizes)]))
    eager = plain.last_kernel_name()
    with torch.cuda.stream(stream):
        for n in sizes:
            hip.reserve_matmul(dtype, m, n, k)
    batch = hip.make_batch([(d, x, y, dtype, m, n, k) for d, y, n in zip(dev, ys, sizes)])
    print(f"captured group dtype={dtype} m={m} {elem}", flush=True)
    for got in captured(torch, hip, stream, lambda: hip.run_batch(batch), ys):
        assert hip.last_kernel_name() == eager
        assert all(torch.equal(g.view(torch.uint8), a.view(torch.uint8)) for g, a in zip(got, want))


def rounded_f32_call(torch, hip, w, x16, dtype, m, n, k):
    """The call over 16-bit elements, and the f32 call on the widened activations rounded to them."""
    y16, y32 = torch.zeros(m, n, dtype=x16.dtype, device="cuda"), torch.zeros(m, n, device="cuda")
    hip.quantized_matmul(w, x16, y16, dtype, m, n, k)
    hip.quantized_matmul(w, x16.float(), y32, dtype, m, n, k)
    torch.cuda.synchronize()
    return y16.view(torch.int16), y32.to(x16.dtype).view(torch.int16)


@pytest.mark.parametrize("dtype, n, k, rows", [
    (Q4_K, 4096, 4096, (33, 48, 100, 200)), (Q8_0, 4999, 2880, (77, 40)), (Q6_K, 4096, 4096, (20, 128, 77)), (Q5_K, 700, 14336, (33, 64, 300)),
    (Q8_0, 2000, 8192, (17, 64, 130)), (Q6_K, 3000, 11008, (9, 33, 257))])
@pytest.mark.parametrize("elem", ["float16", "bfloat16"])
def test_element_types_have_the_slices_of_the_f32_call(torch, dtype, n, k, rows, elem):
    """Tiles and slices as the shape gets them: the 16-bit call is the rounded f32 call, bit for bit."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0)
    w = torch.from_numpy(random_weight(dtype, n, k, seed=5).view(np.uint8).reshape(-1)).cuda()
    x = torch.from_numpy(random_activations(max(rows), k, seed=6)).cuda().to(getattr(torch, elem))
    for m in rows:
        print(f"slices dtype={dtype} m={m} n={n} k={k} {elem}", flush=True)
        got, want = rounded_f32_call(torch, hip, w, x[:m].contiguous(), dtype, m, n, k)
        assert torch.equal(got, want)


@pytest.mark.parametrize("t_gu, t_dn", [(Q4_K, Q6_K), (Q5_K, Q6_K), (Q6_K, Q6_K), (Q8_0, Q8_0)])
@pytest.mark.parametrize("hidden, ffn", [(1024, 1280), (4096, 8192)])
def test_feed_forward_of_16_bit_elements_is_the_rounded_f32_block(torch, t_gu, t_dn, hidden, ffn):
    """Whatever kernels the rows and the size take: the int8 kernels and the GEMM for 5 to 8 rows, the GEMM beyond."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0)
    g, u, d = (torch.from_numpy(random_weight(t, a, b, seed=i).view(np.uint8).reshape(-1)).cuda()
               for i, (t, a, b) in enumerate(((t_gu, ffn, hidden), (t_gu, ffn, hidden), (t_dn, hidden, ffn))))
    for m in (1, 4, 5, 6, 7, 8, 9, 24, 70):
        for t in (torch.float16, torch.bfloat16):
            print(f"ffn {t_gu}/{t_dn} {hidden} {ffn} m={m} {t}", flush=True)
            x = (torch.from_numpy(random_activations(m, hidden, seed=m)) * 1e-2).cuda().to(t)
            out, full = torch.zeros(m, hidden, dtype=t, device="cuda"), torch.zeros(m, hidden, device="cuda")
            hip.ffn_swiglu(g, u, t_gu, d, t_dn, x, out, m, hidden, ffn)
            hip.ffn_swiglu(g, u, t_gu, d, t_dn, x.float(), full, m, hidden, ffn)
            torch.cuda.synchronize()
            assert torch.equal(out.view(torch.int16), full.to(t).view(torch.int16))


@pytest.mark.parametrize("dtype, m, k, sizes, one", [
    (Q4_K, 5, 512, [8192, 4096], True), (Q4_K, 5, 512, [8192, 4097], False), (Q6_K, 8, 256, [4096, 4096, 4096], True), (Q6_K, 8, 256, [4096, 4096, 4097], False),
    (Q5_K, 3, 4352, [9216, 9216], True), (Q5_K, 3, 4352, [9216, 9217], False), (Q4_K, 16, 4096, [16384, 16384], True), (Q4_K, 16, 4096, [16384, 16385], False),
    (Q8_0, 9, 4096, [16384, 16385], True)])
def test_lines_of_the_launch_over_several_matrices(torch, dtype, m, k, sizes, one):
    """On both sides of the most weight rows that the GEMM takes as one launch."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0)
    x = torch.from_numpy(random_activations(m, k, seed=3)).cuda()
    dev = [torch.from_numpy(random_weight(dtype, n, k, seed=n + i).view(np.uint8).reshape(-1)).cuda() for i, n in enumerate(sizes)]
    ys, alone = ([torch.full((m, n), float("nan"), device="cuda") for n in sizes] for _ in range(2))
    print(f"lines dtype={dtype} m={m} k={k} {sizes}", flush=True)
    for d, y, n in zip(dev, alone, sizes):
        hip.quantized_matmul(d, x, y, dtype, m, n, k)
    hip.run_batch(hip.make_batch([(d, x, y, dtype, m, n, k) for d, y, n in zip(dev, ys, sizes)]))
    torch.cuda.synchronize()
    for a, b in zip(ys, alone):
        if one:
            assert float((a - b).norm() / b.norm()) <= 4e-6 # (the int8 kernels' 1.2e-6, twice, over the GEMM's)
        else:
            assert torch.equal(a, b)


@pytest.mark.parametrize("elem", ["float32", "bf16 mode", "float16", "bfloat16"])
@pytest.mark.parametrize("tiles, runs", [(2, 0), (3, 0), (4, 0), (0, 0), (0, 1)])
def test_weights_decoded_first(torch, elem, tiles, runs):
    """Q6_K weights that are decoded ahead of the GEMM: the bits of the GEMM that unpacks them, with one block of K, blocks that K does
    not fill, long rows added up in runs, weight rows that are no whole tiles or records, several matrices, one that goes in slabs,
    rows of zeros and non-finite ones."""
    from gllm_amd.backend import ACT_BF16, ACT_F32_SPLIT, HipBackend
    mode = ACT_BF16 if elem == "bf16 mode" else ACT_F32_SPLIT
    t = torch.float32 if elem == "bf16 mode" else getattr(torch, elem)
    options = {"mmfw_ksplit": 1, "mmfw_mt": tiles, "mmfw_min_m": 9}
    hips = [HipBackend(0, options={**options, "mmfx_min_m": v}) for v in (33, 0)]
    shapes = [(129, 257, 14336)] if runs else [(33, 257, 256), (131, 1, 512), (97, 1000, 832), (300, 545, 2304)]
    if tiles == 0 and not runs:
        shapes.append((64, 80000, 1024))  # more than 128 MiB of decoded weights
    for m, n, k in shapes:
        x = torch.from_numpy(random_activations(m, k, seed=k + m)).cuda()
        x[0] = 0.0
        x[1] *= 1e-30
        x[3, 5], x[m - 1, 0] = float("nan"), float("inf")
        x = x.to(t)
        sizes = (n, n // 3 + 1, 40)
        ws = [torch.from_numpy(random_weight(Q6_K, s, k, seed=s)).cuda() for s in sizes]
        outs = []
        for hip in hips:
            print(f"decoded weights {elem} tiles={tiles} m={m} n={n} k={k}", flush=True)
            ys = [torch.full((m, s), 7.0, device="cuda", dtype=t) for s in (n,) + sizes]
            hip.quantized_matmul(ws[0], x, ys[0], Q6_K, m, n, k, mode)
            assert hip.last_kernel_name().endswith("_dec") == (hip is hips[0]), hip.last_kernel_name()
            if mode == ACT_F32_SPLIT and n < 80000:
                hip.quantized_matmul_batch([(w, x, y, Q6_K, m, y.shape[1], k) for w, y in zip(ws, ys[1:])])
                assert hip.last_kernel_name().endswith("_dec") == (hip is hips[0]), hip.last_kernel_name()
            torch.cuda.synchronize()
            outs.append(ys)
        for a, b in zip(*outs):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_weights_decoded_first_in_a_graph(torch):
    """A captured block decodes where the scratch has room for it, also behind calls that outgrow that scratch, and gives the eager
    bits on every replay."""
    from gllm_amd.backend import HipBackend
    hip = HipBackend(0, options={"mmfx_min_m": 64})
    m, hidden, ffn = 96, 512, 1024
    weights = [torch.from_numpy(random_weight(Q6_K, n, k, seed=n + i)).cuda() for i, (n, k) in enumerate(((ffn, hidden), (ffn, hidden), (hidden, ffn)))]
    x = torch.from_numpy(random_activations(m, hidden, seed=5)).cuda()
    want, got = torch.zeros(m, hidden, device="cuda"), torch.zeros(m, hidden, device="cuda")
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        call = lambda y: hip.ffn_swiglu(weights[0], weights[1], Q6_K, weights[2], Q6_K, x, y, m, hidden, ffn)
        call(want)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call(got)
        more = torch.zeros(4 * m, hidden, device="cuda")
        for i in range(4):
            got.fill_(7.0)
            graph.replay()
            hip.ffn_swiglu(weights[0], weights[1], Q6_K, weights[2], Q6_K, more, torch.zeros_like(more), 4 * m, hidden, ffn)
            stream.synchronize()
            assert torch.equal(want, got), i
