"""Weight-only antiquant matmul captured in a HIP graph: every replay, with eager work and synchronisations between
the replays, equals the eager call bit for bit (the decode-loop use of the entry point; it records no memset, no
allocation and no host synchronisation, so the calls capture as plain kernel nodes)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import seeded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w_type", ["int4", "int8"])
@pytest.mark.parametrize("M", [1, 16, 32, 64])
def test_antiquant_matmul_graph_replays(ascq_gpu, w_type, M):
    rng = seeded(4000 + M)
    K, N, g = 1024, 1008, 128
    at = ascq_gpu.INT8 if w_type == "int8" else ascq_gpu.INT4
    wb = K * N // (1 if w_type == "int8" else 2)
    w = torch.from_numpy(rng.integers(0, 256, wb, dtype=np.uint8)).cuda()
    wp = ascq_gpu.weight_pack(w, at, K, N)
    scale = torch.from_numpy(np.exp(rng.uniform(np.log(1e-3), np.log(1e-1), (K // g, N))).astype(np.float16)).cuda()
    offset = torch.from_numpy(rng.uniform(-8, 8, (K // g, N)).astype(np.float16)).cuda()
    xs = [torch.from_numpy(rng.standard_normal((M, K)).astype(np.float16)).cuda() for _ in range(2)]
    ys = [torch.empty((M, N), dtype=torch.float16, device="cuda") for _ in range(2)]
    eager = [ascq_gpu.antiquant_matmul(xs[i], wp, at, scale, offset, g, N) for i in range(2)]
    torch.cuda.synchronize()

    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(st):
        with torch.cuda.graph(graph, stream=st):
            for i in range(2):
                ascq_gpu.antiquant_matmul(xs[i], wp, at, scale, offset, g, N, out=ys[i])
    torch.cuda.current_stream().wait_stream(st)
    for rep in range(4):
        for y in ys:
            y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for i in range(2):
            assert torch.equal(ys[i], eager[i]), f"replay {rep}, call {i} differs from the eager result"
        # eager work between replays, on the same buffers the graph reads
        ascq_gpu.antiquant_matmul(xs[1], wp, at, scale, offset, g, N, out=ys[0])
        torch.cuda.synchronize()
    del graph


@pytest.mark.parametrize("fp8", [False, True])
def test_eager_packed_call_leaves_a_captured_graph_alone(ascq_gpu, fp8):
    """A decode call whose K-split partials lie in the handle's workspace, captured; then eager calls of the same handle
    with a misaligned A, which is packed: every replay between them equals the eager result (integer-valued operands,
    exact sums)"""
    ascq = ascq_gpu
    M, N, K = 16, 4096, 8192
    g = torch.Generator().manual_seed(11)
    A, B = torch.randint(-4, 5, (M, K), generator=g), torch.randint(-4, 5, (N, K), generator=g)
    A2 = torch.randint(-4, 5, (M, K), generator=g)
    dt = torch.float8_e4m3fn if fp8 else torch.int8
    code = lambda t: t.float().to(dt).cuda()  # noqa: E731
    ref, ref2 = A.float() @ B.float().t(), A2.float() @ B.float().t()
    mm = ascq.Matmul(ascq.FP8_E4M3, ascq.FP8_E4M3, ascq.F32) if fp8 else ascq.Matmul(ascq.INT8, ascq.INT8, ascq.INT32)
    mm.SetOrgShape(M, N, K)
    a, b = code(A), code(B)
    buf = torch.zeros(M * K + 16, dtype=torch.uint8, device="cuda")
    buf[3:3 + M * K] = code(A2).view(torch.uint8).reshape(-1)
    mm.SetTensorA(a)
    mm.SetTensorB(b, True)
    out = torch.zeros((M, N), dtype=torch.float32 if fp8 else torch.int32, device="cuda")
    out2 = torch.zeros_like(out)
    mm.IterateAll(out)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(st), torch.cuda.graph(graph, stream=st):
        mm.IterateAll(out)
    torch.cuda.current_stream().wait_stream(st)
    mm.SetTensorA(buf[3:3 + M * K])
    for _ in range(3):
        out2.zero_()
        mm.IterateAll(out2)
        assert torch.equal(out2.cpu().float(), ref2)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.cpu().float(), ref)


def test_packed_calls_beside_a_capture_and_on_two_streams(ascq_gpu):
    """Calls whose operands are packed: the first call of a new handle on another stream while a capture is running leaves
    the capture valid, and one handle used on two streams without waits between them computes both products"""
    ascq = ascq_gpu
    M, N, K = 300, 2000, 3001
    g = torch.Generator().manual_seed(12)
    A = [torch.randint(-4, 5, (M, K), generator=g) for _ in range(2)]
    B = torch.randint(-4, 5, (K, N), generator=g)
    ref = [x.float() @ B.float() for x in A]
    a, b = [x.to(torch.int8).cuda() for x in A], B.to(torch.int8).cuda()

    def handle():
        mm = ascq.Matmul(ascq.INT8, ascq.INT8, ascq.INT32)
        mm.SetOrgShape(M, N, K)
        mm.SetTensorA(a[0])
        mm.SetTensorB(b)
        return mm

    out = [torch.zeros((M, N), dtype=torch.int32, device="cuda") for _ in range(2)]
    warm = handle()
    warm.IterateAll(out[0])
    x = torch.ones(64, device="cuda")
    st, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    fresh = handle()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(st), torch.cuda.graph(graph, stream=st):
        x.add_(1.0)
        fresh.IterateAll(out[1], stream=other)
    other.synchronize()
    assert torch.equal(out[1].cpu().float(), ref[0])
    for rep in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert bool((x == 2.0 + rep).all())
    for o in out:
        o.zero_()
    torch.cuda.synchronize()
    for i, s in enumerate((st, other)):
        warm.SetTensorA(a[i])
        warm.IterateAll(out[i], stream=s)
    torch.cuda.synchronize()
    for i in range(2):
        assert torch.equal(out[i].cpu().float(), ref[i])
