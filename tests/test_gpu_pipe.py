"""GPU parity of the pipelined GEMM tiles (gemm_pipe.h) at sizes the dispatch gives to each tile shape: partial last tiles
in M and N, K tails of 16-byte chunks, odd stage counts, both B layouts, vector and element-wise stores.  int8: bit-exact
against the oracle.  fp8: integer-valued codes (-4 .. 4) make every sum exact in fp32, so f32 C equals the fp64 product
and bf16 C its one rounding."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle_lib as O
from conftest import seeded

pytestmark = pytest.mark.gpu

# (M, N, K): the tile pick_pipe_tile chooses
SHAPES = [
    (77, 377, 64),       # 64 x 128, one partial stage
    (65, 4100, 336),     # 64 x 128, three stages, the last of 80 bytes
    (3353, 536, 272),    # 128 x 128
    (4127, 932, 416),    # 128 x 192
    (1607, 3736, 528),   # 128 x 256
    (3457, 1732, 64),    # 64 x 128, seven rounds of one partial stage
    (3273, 1816, 144),   # 64 x 128
    (3585, 2180, 144),   # 192 x 256
    (4436, 1288, 144),   # 256 x 192
    (3301, 3804, 80),    # 256 x 256
]


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _bits(t):
    return t.cpu().view(torch.int16).numpy().view(np.uint16)


# odd N (odd pitches of C, a [K, N] B packed), and K of every remainder class of a chunk (operands packed): few rows too
# aligned calls with few tiles or few stages, on the 32 x 32 and 64 x 64 tiles (which of the two layouts: in the comments)
FEW = [
    (70, 528, 528),       # both: 32 x 32 (int8); 64 x 64 (fp8, [N, K])
    (70, 4112, 1040),     # [N, K]: 64 x 64, 66 tiles of 64 x 128
    (130, 8000, 528),     # [N, K]: 64 x 64, 189 of them (int8)
    (300, 6032, 272),     # both: 64 x 64 (int8)
    (65, 1040, 4112),     # [N, K]: 64 x 64, rows off 128 bytes
    (40, 4624, 6160),     # [K, N]: 64 x 64 (few_long_kn), K its least
    (130, 2576, 8208),    # [K, N]: 64 x 64
    (33, 2064, 10256),    # [K, N]: 32 x 32 (int8)
    (300, 848, 12304),    # [K, N]: 64 x 64
]
RAGGED = [(130, 1001, 2048), (300, 5003, 1040), (130, 1004, 2047), (1, 1030, 1009), (20, 515, 77), (33, 601, 1), (70, 130, 4095)]


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES + RAGGED + FEW)
def test_int8_pipe(ascq_gpu, oracle, M, N, K, trans_b):
    rng = seeded(M + N + K + trans_b)
    A = rng.integers(-128, 128, (M, K), dtype=np.int8)
    B = rng.integers(-128, 128, (N, K) if trans_b else (K, N), dtype=np.int8)
    bias = rng.integers(-(1 << 20), 1 << 20, N, dtype=np.int32)
    words = np.exp(rng.uniform(np.log(2.0 ** -20), np.log(2.0 ** -8), N)).astype(np.float32).view(np.uint32).astype(np.uint64)
    acc = O.matmul_i8(A, B, bias, False, trans_b)
    a, b, bi, w = _dev(A), _dev(B), _dev(bias), _dev(words.view(np.int64))
    for c_type, dt, ref in [(ascq_gpu.F16, torch.float16, O.mm_dequant(acc, O.F16, qvec=words)),
                            (ascq_gpu.BF16, torch.bfloat16, O.mm_dequant(acc, O.BF16, qvec=words)),
                            (ascq_gpu.INT32, torch.int32, acc),
                            (ascq_gpu.INT8, torch.int8, O.mm_requant(acc, qvec=words | np.uint64(1 << 46)))]:
        mm = ascq_gpu.Matmul(ascq_gpu.INT8, ascq_gpu.INT8, c_type, ascq_gpu.INT32)
        mm.SetOrgShape(M, N, K)
        if c_type != ascq_gpu.INT32:
            mm.SetQuantVector(_dev((words | np.uint64(1 << 46)).view(np.int64)) if c_type == ascq_gpu.INT8 else w)
        mm.SetTensorA(a)
        mm.SetTensorB(b, trans_b)
        mm.SetBias(bi)
        out = torch.zeros(M * N + 16, dtype=dt, device="cuda")  # the 16 past the end must stay zero
        mm.IterateAll(out)
        torch.cuda.synchronize()
        got = out[:M * N].view(M, N)
        assert not bool(out[M * N:].any()), c_type
        if dt in (torch.float16, torch.bfloat16):
            np.testing.assert_array_equal(_bits(got), ref)
        else:
            np.testing.assert_array_equal(got.cpu().numpy(), ref.view(np.int8) if dt == torch.int8 else ref)


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES + RAGGED + FEW)
def test_fp8_pipe(ascq_gpu, M, N, K, trans_b):
    g = torch.Generator().manual_seed(M + N + K + trans_b)
    A = torch.randint(-4, 5, (M, K), generator=g)
    B = torch.randint(-4, 5, (N, K) if trans_b else (K, N), generator=g)
    bias = torch.randint(-8, 9, (N,), generator=g).float()
    ref = A.double() @ (B.double().t() if trans_b else B.double()) + bias.double()
    a, b = A.float().to(torch.float8_e4m3fn).cuda(), B.float().to(torch.float8_e5m2).cuda()
    for c_type, dt in [(ascq_gpu.F32, torch.float32), (ascq_gpu.BF16, torch.bfloat16)]:
        mm = ascq_gpu.Matmul(ascq_gpu.FP8_E4M3, ascq_gpu.FP8_E5M2, c_type, ascq_gpu.F32)
        mm.SetOrgShape(M, N, K)
        mm.SetTensorA(a)
        mm.SetTensorB(b, trans_b)
        mm.SetBias(bias.cuda())
        out = torch.zeros(M * N + 16, dtype=dt, device="cuda")
        mm.IterateAll(out)
        torch.cuda.synchronize()
        assert not bool(out[M * N:].any()), c_type
        assert torch.equal(out[:M * N].view(M, N).cpu(), ref.float().to(dt)), c_type


def test_ragged_without_a_workspace(ascq_gpu, oracle):
    """Under stream capture a handle without a workspace allocates none: the any-alignment tiles, the same bits; and an
    operand that follows NaN bytes of another buffer (fp8) reads none of them"""
    M, N, K = 70, 200, 1003
    rng = seeded(5)
    A = rng.integers(-128, 128, (M, K), dtype=np.int8)
    B = rng.integers(-128, 128, (K, N), dtype=np.int8)
    a, b = _dev(A), _dev(B)
    mm = ascq_gpu.Matmul(ascq_gpu.INT8, ascq_gpu.INT8, ascq_gpu.INT32)
    mm.SetOrgShape(M, N, K)
    mm.SetTensorA(a)
    mm.SetTensorB(b)
    out = torch.zeros((M, N), dtype=torch.int32, device="cuda")
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(st), torch.cuda.graph(graph, stream=st):
        mm.IterateAll(out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), O.matmul_i8(A, B, None))
    mm.IterateAll(out.zero_())  # eager: the packed form
    np.testing.assert_array_equal(out.cpu().numpy(), O.matmul_i8(A, B, None))

    buf = torch.full((M * K + 64,), 0x7F, dtype=torch.uint8, device="cuda")  # e4m3 NaN around A
    buf[1:1 + M * K] = torch.ones(M * K).to(torch.float8_e4m3fn).view(torch.uint8).cuda()
    ones = torch.ones((K, N)).to(torch.float8_e4m3fn).cuda()
    f8 = ascq_gpu.Matmul(ascq_gpu.FP8_E4M3, ascq_gpu.FP8_E4M3, ascq_gpu.F32)
    f8.SetOrgShape(M, N, K)
    f8.SetTensorA(buf[1:1 + M * K])
    f8.SetTensorB(ones)
    y = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    f8.IterateAll(y)
    assert bool((y == K).all())


# (M, N, K): more than 128 tiles of 64 x 128, the tile pick_pipe_tile chooses; odd and even counts of half stages
MX_SHAPES = [(513, 1900, 640), (1100, 2100, 384), (3353, 536, 640), (4127, 932, 896), (1607, 3736, 1152), (3457, 1732, 128),
             (3273, 1816, 384), (3301, 3804, 128), (3394, 2308, 384), (4430, 1288, 384)]
E2M1 = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64)


@pytest.mark.parametrize("pairs", [False, True])
@pytest.mark.parametrize("M,N,K", MX_SHAPES)
def test_mxfp4_pipe(ascq_gpu, M, N, K, pairs):
    """Elements of at most two significant bits and block scales of 2^-2 .. 2^2: products are multiples of 2^-6 and the
    sums (at most 2^18 in magnitude here) are exact in fp32, so f32 C equals the fp64 product, bf16 C its rounding"""
    g = torch.Generator().manual_seed(M + N + K + pairs)
    A = torch.randint(0, 256, (M, K // 2), generator=g, dtype=torch.uint8)
    B = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8)
    sA = torch.randint(125, 130, (M, K // 32), generator=g, dtype=torch.uint8)
    sB = torch.randint(125, 130, (N, K // 32), generator=g, dtype=torch.uint8)

    def decode(x, s):
        v = torch.stack([E2M1[(x & 15).long()], E2M1[(x >> 4).long()]], -1).reshape(x.shape[0], -1)
        return v * torch.exp2(s.double() - 127).repeat_interleave(32, 1)

    ref = decode(A, sA) @ decode(B, sB).t()
    assert float(ref.abs().max()) < 2.0 ** 18
    to_pairs = lambda s: s.reshape(s.shape[0], -1, 2).permute(1, 0, 2).contiguous()  # noqa: E731
    for c_type, dt in [(ascq_gpu.F32, torch.float32), (ascq_gpu.BF16, torch.bfloat16)]:
        mm = ascq_gpu.Matmul(ascq_gpu.FP4_E2M1, ascq_gpu.FP4_E2M1, c_type, 0, ascq_gpu.E8M0)
        mm.SetOrgShape(M, N, K)
        mm.SetTensorA(A.cuda())
        mm.SetTensorB(B.cuda(), True)
        mm.SetTensorScaleA(to_pairs(sA).cuda() if pairs else sA.cuda(), pairs)
        mm.SetTensorScaleB(to_pairs(sB).cuda() if pairs else sB.cuda(), not pairs)
        out = torch.zeros(M * N + 16, dtype=dt, device="cuda")
        mm.IterateAll(out)
        torch.cuda.synchronize()
        assert not bool(out[M * N:].any()), c_type
        assert torch.equal(out[:M * N].view(M, N).cpu(), ref.float().to(dt)), c_type
