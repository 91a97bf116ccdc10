"""GEMMs whose rows the DMA kernel cannot read as they are (K % 128 != 0, or
operands off by a word) run on zero-padded copies: accumulators against exact
int64 sums around the 128-byte stage, for int8 and int4 weights. The copies live
in a workspace of the stream: two host threads on one stream do not mix theirs,
and a captured GEMM does not use it (it takes the other kernel): against the
eager bits, with graphs replayed on several streams at once."""
import threading

import numpy as np
import pytest
import torch

from brain_amd import ops
from oracle import oracle as o

pytestmark = pytest.mark.gpu


def words(rng, rows, kw):
    return torch.from_numpy(rng.integers(-2 ** 31, 2 ** 31, (rows, kw), dtype=np.int64).astype(np.int32)).cuda()


def int8_of(t):
    return t.contiguous().cpu().numpy().view(np.int8).astype(np.int64)


def int4_of(t):
    w = t.cpu().numpy().view(np.uint32)
    n = np.stack([(w >> (4 * b)) & 15 for b in range(8)], -1).reshape(w.shape[0], -1).astype(np.int64)
    return np.where(n > 7, n - 16, n)


@pytest.mark.parametrize("m,k,n", [(33, 4, 1), (33, 124, 65), (64, 128, 64), (65, 132, 130), (200, 1000, 257),
                                   (333, 2900, 111), (40, 6148, 70), (300, 516, 1030)])
@pytest.mark.parametrize("off", [0, 1])
def test_padded_i8_accumulators(gpu, m, k, n, off):
    rng = np.random.default_rng(m + k + n)
    x = words(rng, 1, m * k // 4 + off).view(-1)[off:].view(m, k // 4)  # off: not 16-byte aligned
    w = words(rng, n, k // 4)
    one = torch.ones(max(m, n), device="cuda")
    got = ops.matmul_i8(x, w, one[:m], one[:n], None, torch.int32, "dyn").cpu().numpy()
    assert np.array_equal(got, int8_of(x) @ int8_of(w).T)


@pytest.mark.parametrize("m,k,n", [(33, 8, 1), (33, 120, 65), (64, 128, 64), (65, 136, 130), (200, 1000, 257),
                                   (512, 2048, 300), (300, 6976, 70), (40, 4096, 129), (1030, 256, 520)])
def test_q4_accumulators(gpu, m, k, n):
    rng = np.random.default_rng(m + k + n + 7)
    x, w = words(rng, m, k // 4), words(rng, n, k // 8)
    one = torch.ones(max(m, n), device="cuda")
    got = ops.matmul_q4(x, w, one[:m], one[:n], None, torch.int32, "dyn").cpu().numpy()
    assert np.array_equal(got, int8_of(x) @ int4_of(w).T)


def gpu_words(g, rows, kw):
    return torch.randint(-2 ** 31, 2 ** 31, (rows, kw), device="cuda", generator=g, dtype=torch.int64).to(torch.int32)


def gpu_int4(w):
    n = torch.stack([(w >> (4 * b)) & 15 for b in range(8)], -1).reshape(w.shape[0], -1)
    return torch.where(n > 7, n - 16, n)


@pytest.mark.parametrize("m,k,n", [
    (8192, 256, 1108), (6144, 128, 257),     # expanded to int8
    (4096, 256, 21000), (5000, 136, 17001),  # column ranges of 256x256 tiles and a rest
    (300, 131200, 64), (70, 262272, 65),     # K split so that 16 q fit an i32 sum
    (300, 9952, 151936),                     # padded copies in two column ranges
    (1152, 10240, 3840),                     # 256x256 tiles split over K
    (1000, 640, 4000), (1000, 640, 2100), (1000, 648, 3990),  # 128x128 and 64x128 tiles; padded
])
def test_q4_large_accumulators(gpu, m, k, n):
    g = torch.Generator(device="cuda")
    g.manual_seed(m + k + n)
    x, w = gpu_words(g, m, k // 4), gpu_words(g, n, k // 8)
    one = torch.ones(max(m, n), device="cuda")
    got = ops.matmul_q4(x, w, one[:m], one[:n], None, torch.int32, "dyn")
    rows = torch.arange(m, device="cuda") if m * n * k < 2 ** 36 else torch.randperm(m, device="cuda", generator=g)[:64]
    xr = x[rows].view(torch.int8).double()
    for n0 in range(0, n, 16384):  # exact: sums below 2^53
        assert torch.equal(got[rows, n0:n0 + 16384].double(), xr @ gpu_int4(w[n0:n0 + 16384]).double().t())


@pytest.mark.parametrize("reserve", [False, True])
@pytest.mark.parametrize("q4", [False, True])
def test_ragged_capture(gpu, q4, reserve):
    m, k, n = 150, 1000, 420
    rng = np.random.default_rng(5)
    x, w = words(rng, m, k // 4), words(rng, n, k // (8 if q4 else 4))
    sx, sw = torch.rand(m, device="cuda"), torch.rand(n, device="cuda")
    mm = ops.matmul_q4 if q4 else ops.matmul_i8
    eager = mm(x, w, sx, sw, None, torch.float32, "dyn").clone()
    out = torch.empty(m, n, device="cuda")
    cap = torch.cuda.Stream()
    if reserve:
        ops.reserve_workspace(m, k, n, cap)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=cap):
        mm(x, w, sx, sw, None, torch.float32, "dyn", out=out)
    for _ in range(3):
        out.fill_(0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


def ragged(m, k, n, q4, seed):
    rng = np.random.default_rng(seed)
    x, w = words(rng, m, k // 4), words(rng, n, k // (8 if q4 else 4))
    one = torch.ones(max(m, n), device="cuda")
    want = torch.from_numpy((int8_of(x) @ (int4_of(w) if q4 else int8_of(w)).T).astype(np.int32)).cuda()
    mm = ops.matmul_q4 if q4 else ops.matmul_i8
    return (lambda: mm(x, w, one[:m], one[:n], None, torch.int32, "dyn")), want


@pytest.mark.parametrize("m,k,n", [(65, 1000, 257), (40, 6152, 64)])  # unsplit; split over K
def test_two_threads_on_one_stream(gpu, m, k, n):
    work = [ragged(m, k, n, q4, seed) for seed, q4 in enumerate((False, True, False, True))]
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream()
    start, bad = threading.Barrier(len(work)), []

    def run(call, want):
        with torch.cuda.stream(stream):
            start.wait()
            outs = [call() for _ in range(50)]
            torch.cuda.synchronize()
            bad.extend(i for i, out in enumerate(outs) if not torch.equal(out, want))

    threads = [threading.Thread(target=run, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_two_graphs_of_one_capture_stream(gpu):
    m, k, n = 65, 1000, 257
    cap = torch.cuda.Stream()
    work = [ragged(m, k, n, q4, 11 + q4) for q4 in (False, True)] + [ragged(m, k, n, False, 13)]
    torch.cuda.synchronize()
    graphs = []
    with torch.cuda.stream(cap):
        for call, want in work:
            assert torch.equal(call(), want)  # the stream's workspace is large enough
    for call, _ in work[:2]:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=cap):
            graphs.append((g, call()))
    s0, s1 = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(20):
        for _, out in graphs:
            out.fill_(0)
        torch.cuda.synchronize()
        for s, (g, _) in zip((s0, s1), graphs):
            with torch.cuda.stream(s):
                g.replay()
        with torch.cuda.stream(cap):  # eager work that does use the workspace
            assert torch.equal(work[2][0](), work[2][1])
        torch.cuda.synchronize()
        for (_, out), (_, want) in zip(graphs, work):
            assert torch.equal(out, want)


def test_capture_after_a_larger_ragged_call(gpu):
    """33x2692x1024 does not split K, its padded K = 2816 does: captured without
    a reserve after an eager call that left a larger padded copy, it runs."""
    cap = torch.cuda.Stream()
    call, want = ragged(33, 2692, 1024, False, 3)
    large, _ = ragged(1056, 2692, 1024, False, 4)  # padded, unsplit: no slabs are left behind
    torch.cuda.synchronize()
    with torch.cuda.stream(cap):
        large()
    cap.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=cap):
        out = call()
    for _ in range(3):
        out.fill_(0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_captured_q4_splits_from_256_rows_only(gpu):
    """int4 weights under capture with the slabs reserved: from 256 rows K is
    split (K % 128 == 0 on the DMA tiles, else on the register-staged ones),
    below it is not. Exact sums either way."""
    for m, k, n in ((256, 8160, 1024), (256, 8192, 1024), (200, 8192, 1024)):
        cap = torch.cuda.Stream()
        call, want = ragged(m, k, n, True, m + k)
        ops.reserve_workspace(m, k, n, cap)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=cap):
            out = call()
        for _ in range(3):
            out.fill_(0)
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want), (m, k, n)
