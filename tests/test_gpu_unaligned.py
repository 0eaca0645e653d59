"""GPU parity of operands off their alignment (K not a multiple of 16, operands at any byte offset) against the oracle: the
any-alignment MFMA tiles of the quantized group matmul, and for the int8 and fp8 Matmul both forms -- packed to aligned
rows first (room == "own": the handle's own, the call made twice, since a first call may go without), and the any-alignment
tiles (room == "none": a caller's workspace too small for packing); and ASCQ_LOG=1 naming the generic kernel a launch falls
back to.

Each operand is placed at a byte offset inside a larger device buffer whose other bytes hold 0x5A, so bytes read past
K, past a row or past the operand would enter the sums unless the kernel zeroes them.  int8: int32 accumulators,
bit-exact outputs.  fp8: integer-valued codes (-4 .. 4) give exact sums, so f32 C is bit-exact as well."""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

import oracle_lib as O
from conftest import seeded

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parents[1]
FILL = 0x5A


def _dev_at(a, off):
    """a (int8 / uint8) on the device at byte offset `off` of a buffer filled with FILL"""
    a = np.ascontiguousarray(a)
    buf = torch.full((a.nbytes + off + 64,), FILL, dtype=torch.uint8, device="cuda")
    buf[off:off + a.nbytes] = torch.from_numpy(a.view(np.uint8).reshape(-1)).cuda()
    t = buf[off:off + a.nbytes]
    return (t.view(torch.int8) if a.dtype == np.int8 else t).view(a.shape)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _bits(t):
    return t.view(torch.int16).numpy().view(np.uint16)


@pytest.mark.parametrize("w_trans", [False, True])
@pytest.mark.parametrize("K,N,x_off,w_off", [(100, 160, 0, 0), (333, 150, 3, 5), (17, 162, 1, 0), (1, 64, 0, 7),
                                             (256, 160, 4, 2), (1000, 704, 1, 1)])
def test_group_matmul_any_alignment(ascq_gpu, oracle, w_trans, K, N, x_off, w_off):
    """K % 16 != 0 and / or X, W at odd byte offsets: the any-alignment tiles, bit-exact, rows outside the groups
    untouched"""
    rng = seeded(900 + K + N + x_off + 2 * w_off + w_trans)
    counts = np.array([97, 0, 140, 33], np.int64) if K < 1000 else np.array([400, 1, 333, 290], np.int64)
    G = len(counts)
    M = int(counts.sum()) + 5
    x = rng.integers(-128, 128, (M, K), dtype=np.int8)
    w = rng.integers(-128, 128, (G, N, K) if w_trans else (G, K, N), dtype=np.int8)
    pts = np.exp(rng.uniform(np.log(1e-3), np.log(1e-1), M)).astype(np.float32)
    scale = np.exp(rng.uniform(np.log(1e-4), np.log(1e-2), (G, N))).astype(np.float32)
    gl = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    y = torch.full((M, N), 3.0, dtype=torch.bfloat16, device="cuda")
    ascq_gpu.quant_group_matmul(_dev_at(x, x_off), _dev(pts), _dev_at(w, w_off), _dev(scale), _dev(gl), 0, w_trans,
                                torch.bfloat16, out=y)
    y0 = torch.full((M, N), 3.0, dtype=torch.bfloat16).view(torch.int16).numpy().view(np.uint16).copy()
    ref = O.group_matmul(x, pts, w, scale, gl, 0, G, M, K, N, O.BF16, w_trans, y=y0)
    np.testing.assert_array_equal(_bits(y.cpu()), ref)


def _no_room(mm):
    """a caller's workspace that holds what the call cannot do without, but no room to pack operands"""
    mm.SetWorkspace(torch.empty(256, dtype=torch.uint8, device="cuda"), 256)


def _int8_mm(ascq, A, B, bias, words, trans_a, trans_b, a_off, b_off, M, N, K, single=None, room="own"):
    mm = ascq.Matmul(ascq.INT8, ascq.INT8, ascq.F16, ascq.INT32)
    mm.SetOrgShape(M, N, K)
    if single is not None:
        mm.SetSingleShape(*single)
    mm.SetQuantVector(_dev(words.view(np.int64)))
    mm.SetTensorA(_dev_at(A, a_off), trans_a)
    mm.SetTensorB(_dev_at(B, b_off), trans_b)
    mm.SetBias(_dev(bias))
    if room == "none":
        _no_room(mm)
    first = None
    for _ in range(2 if room == "own" else 1):
        c = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
        mm.IterateAll(c)
        torch.cuda.synchronize()
        bits = _bits(c.cpu())
        assert first is None or np.array_equal(first, bits)
        first = bits
    mm.End()
    return first


@pytest.mark.parametrize("room", ["own", "none"])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("shape,a_off,b_off", [((77, 200, 99), 0, 0), ((300, 132, 1037), 3, 1), ((5, 7, 3), 1, 2),
                                               ((1030, 1100, 333), 2, 0), ((2100, 2080, 77), 0, 3),
                                               ((2100, 2080, 205), 1, 3)])
def test_int8_matmul_any_alignment(ascq_gpu, oracle, trans_b, shape, a_off, b_off, room):
    """int8 Matmul, DEQF16 C with int32 bias and per-channel words, K % 16 != 0 and / or A, B at odd byte offsets: packed from
    K = 192 on where there is room, else 64 x 64 and, for 2100 x 2080, 128 x 128 any-alignment tiles; bit-exact"""
    M, N, K = shape
    rng = seeded(M + N + K + a_off + trans_b)
    A = rng.integers(-128, 128, (M, K), dtype=np.int8)
    Bkn = rng.integers(-128, 128, (K, N), dtype=np.int8)
    bias = rng.integers(-(1 << 20), 1 << 20, N, dtype=np.int32)
    sc = np.exp(rng.uniform(np.log(2.0 ** -20), np.log(2.0 ** -8), N)).astype(np.float32)
    words = sc.view(np.uint32).astype(np.uint64)
    got = _int8_mm(ascq_gpu, A, np.ascontiguousarray(Bkn.T) if trans_b else Bkn, bias, words, False, trans_b, a_off,
                   b_off, M, N, K, room=room)
    ref = O.mm_dequant(O.matmul_i8(A, Bkn, bias), O.F16, qvec=words)
    np.testing.assert_array_equal(got, ref)


def test_int8_matmul_any_alignment_trans_a_single_shape(ascq_gpu, oracle):
    """A given [K, M] (transposed into the workspace, rows of K = 150 bytes) and a SetSingleShape block with k = 131"""
    rng = seeded(77)
    M, N, K = 200, 180, 150
    A = rng.integers(-128, 128, (M, K), dtype=np.int8)
    Bkn = rng.integers(-128, 128, (K, N), dtype=np.int8)
    bias = rng.integers(-(1 << 20), 1 << 20, N, dtype=np.int32)
    words = np.full(N, np.float32(2.0 ** -12).view(np.uint32), np.uint64)
    got = _int8_mm(ascq_gpu, np.ascontiguousarray(A.T), Bkn, bias, words, True, False, 1, 0, M, N, K)
    np.testing.assert_array_equal(got, O.mm_dequant(O.matmul_i8(A, Bkn, bias), O.F16, qvec=words))
    sm, sn, sk = 130, 100, 131
    got = _int8_mm(ascq_gpu, A, Bkn, bias, words, False, False, 3, 1, M, N, K, single=(sm, sn, sk))
    ref = O.mm_dequant(O.matmul_i8(np.ascontiguousarray(A[:sm, :sk]), np.ascontiguousarray(Bkn[:sk, :sn]), bias[:sn]),
                       O.F16, qvec=words[:sn])
    np.testing.assert_array_equal(got[:sm, :sn], ref)
    assert np.isnan(got[sm:].view(np.float16)).all() and np.isnan(got[:, sn:].view(np.float16)).all()


def _fp8_of(v):
    return torch.from_numpy(np.ascontiguousarray(v)).float().to(torch.float8_e4m3fn).view(torch.uint8).numpy()


def _fp8_codes(rng, shape, t8):
    v = rng.integers(-4, 5, shape).astype(np.float32)
    return torch.from_numpy(v).to(t8).view(torch.uint8).numpy()


@pytest.mark.parametrize("room", ["own", "none"])
@pytest.mark.parametrize("fa,fb", [(O.FP8_E4M3, O.FP8_E4M3), (O.FP8_E5M2, O.FP8_E4M3)])
@pytest.mark.parametrize("shape,a_off,b_off", [((96, 160, 150), 0, 0), ((300, 200, 77), 5, 3),
                                               ((2100, 2080, 40), 1, 0), ((96, 160, 250), 3, 0), ((2100, 2080, 203), 1, 2)])
def test_fp8_matmul_any_alignment(ascq_gpu, oracle, fa, fb, shape, a_off, b_off, room):
    """fp8 A [M, K], B [N, K] with K % 16 != 0 and / or at odd byte offsets, f32 bias, f32 C: integer-valued codes,
    exact sums, bit-exact; packed from K = 192 on where there is room, else the 64 x 64 and (2100 x 2080) 128 x 128
    any-alignment tiles"""
    M, N, K = shape
    rng = seeded(M + K + fa + 3 * fb + a_off)
    tt = {O.FP8_E4M3: torch.float8_e4m3fn, O.FP8_E5M2: torch.float8_e5m2}
    A = _fp8_codes(rng, (M, K), tt[fa])
    Bt = _fp8_codes(rng, (N, K), tt[fb])
    bias = rng.integers(-64, 65, N).astype(np.float32)
    mm = ascq_gpu.Matmul(fa, fb, ascq_gpu.F32, ascq_gpu.F32)
    mm.SetOrgShape(M, N, K)
    mm.SetTensorA(_dev_at(A, a_off))
    mm.SetTensorB(_dev_at(Bt, b_off), True)
    mm.SetBias(_dev(bias))
    if room == "none":
        _no_room(mm)
    ref, _, _, _ = O.matmul_fp8(A, Bt, fa, fb, bias=bias, out_type=O.F32, trans_b=True)
    for _ in range(2 if room == "own" else 1):
        c = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
        mm.IterateAll(c)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(c.cpu().numpy(), ref)
    mm.End()


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("kind", ["int8", "fp8"])
def test_packed_calls(ascq_gpu, oracle, kind, trans_b):
    """One handle whose operands are packed, through what can change between its calls: other pointers at other offsets, a
    single shape and back, A given [K, M] with an odd K (a copy in the workspace is packed), enAtomic, a caller's workspace
    of the reported size, End and a smaller shape.  Integer-valued operands, exact sums"""
    ascq = ascq_gpu
    M, N, K = 150, 333, 1201
    rng = seeded(60 + trans_b)
    fp8 = kind == "fp8"
    code = _fp8_of if fp8 else (lambda v: v)
    ints = lambda *shape: rng.integers(-4, 5, shape, dtype=np.int8)  # noqa: E731
    A, A2, B, B2 = ints(M, K), ints(M, K), ints(K, N), ints(K, N)
    lay = lambda b: np.ascontiguousarray(b.T) if trans_b else b  # noqa: E731
    prod = lambda a, b: a.astype(np.int32) @ b.astype(np.int32)  # noqa: E731
    dt = torch.float32 if fp8 else torch.int32
    t = ascq.FP8_E4M3 if fp8 else ascq.INT8
    mm = ascq.Matmul(t, t, ascq.F32 if fp8 else ascq.INT32)

    def run(want, op=0, c0=0, calls=1, block=None):
        m, n = block or (M, N)
        c = torch.full((M, N), c0, dtype=dt, device="cuda")
        for _ in range(calls):
            mm.IterateAll(c, op)
        got = c.cpu().numpy()
        np.testing.assert_array_equal(got[:m, :n], want.astype(got.dtype))
        assert (got[m:] == c0).all() and (got[:, n:] == c0).all()

    mm.SetOrgShape(M, N, K)
    mm.SetTensorA(_dev_at(code(A), 0))
    mm.SetTensorB(_dev_at(code(lay(B)), 1), trans_b)
    run(prod(A, B))
    run(prod(A, B))
    mm.SetTensorA(_dev_at(code(A2), 5))
    run(prod(A2, B))
    mm.SetTensorB(_dev_at(code(lay(B2)), 0), trans_b)
    run(prod(A2, B2))
    mm.SetSingleShape(70, 130, 501)
    run(prod(A2[:70, :501], B2[:501, :130]), block=(70, 130))
    mm.SetSingleShape(M, N, K)
    run(3 + 2 * prod(A2, B2), op=ascq.ATOMIC_ADD, c0=3, calls=2)
    mm.SetTensorA(_dev_at(code(np.ascontiguousarray(A.T)), 3), True)
    run(prod(A, B2))
    run(prod(A, B2))
    mm.SetTensorA(_dev_at(code(A), 0))
    nbytes = mm.WorkspaceSize()
    assert nbytes >= M * K
    ws = torch.full((nbytes + 64,), FILL, dtype=torch.uint8, device="cuda")
    mm.SetWorkspace(ws[:nbytes], nbytes)
    run(prod(A, B2))
    assert bool((ws[nbytes:] == FILL).all()) and not bool((ws[:nbytes] == FILL).all())
    mm.SetWorkspace(None, 0)
    mm.End()
    m, n, k = 33, 65, 257
    mm.SetOrgShape(m, n, k)
    mm.SetTensorA(_dev_at(code(np.ascontiguousarray(A[:m, :k])), 0))
    mm.SetTensorB(_dev_at(code(lay(B[:k, :n])), 0), trans_b)
    c = torch.zeros((m, n), dtype=dt, device="cuda")
    mm.IterateAll(c)
    np.testing.assert_array_equal(c.cpu().numpy().astype(np.int32), prod(A[:m, :k], B[:k, :n]))


@pytest.mark.parametrize("room", ["own", "none"])
@pytest.mark.parametrize("fa,fb", [(O.FP8_E4M3, O.FP8_E4M3), (O.FP8_E5M2, O.FP8_E4M3), (O.FP8_E4M3, O.FP8_E5M2)])
@pytest.mark.parametrize("M,N,K,a_off,b_off", [(70, 200, 1003, 0, 0), (600, 100, 333, 1, 0), (33, 68, 512, 3, 0), (5, 66, 1024, 0, 2),
                                               (1, 1, 17, 0, 0), (520, 272, 272, 1, 0)])
def test_fp8_kn_off_alignment_sums_in_fp32(ascq_gpu, fa, fb, M, N, K, a_off, b_off, room):
    """fp8 B [K, N] with a ragged K or N or off its alignment, f32 C: one product of 1 and small ones of 2^-15 in every group of
    16 K.  fp32 sums keep them all (exactly: multiples of 2^-15 below 2^9); the fp8 MFMAs would drop them.  With 16-byte
    multiples from 512 rows on (the last case) the call is on the fp8 MFMAs, aligned or not: their bound of 2^-13"""
    t8 = {O.FP8_E4M3: torch.float8_e4m3fn, O.FP8_E5M2: torch.float8_e5m2}
    a, b = torch.full((M, K), 2.0 ** -8), torch.full((K, N), 2.0 ** -7)
    a[:, ::16], b[::16] = 1.0, 1.0
    want = a.double() @ b.double()
    mm = ascq_gpu.Matmul(fa, fb, ascq_gpu.F32)
    mm.SetOrgShape(M, N, K)
    code = lambda x, t: x.to(t).view(torch.uint8).numpy()  # noqa: E731
    mm.SetTensorA(_dev_at(code(a, t8[fa]), a_off))
    mm.SetTensorB(_dev_at(code(b, t8[fb]), b_off))
    if room == "none":
        _no_room(mm)
    for _ in range(2):
        c = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
        mm.IterateAll(c)
        if M >= 512 and K % 16 == 0 and N % 16 == 0:
            assert float((c.cpu().double() - want).abs().max()) <= 2.0 ** -13 * K
        else:
            assert torch.equal(c.cpu().double(), want)


def test_fp8_kn_off_alignment_special_values(ascq_gpu):
    """NaN and infinities (e5m2) of operands that are decoded to bf16 rows, and of the bytes around them"""
    M, N, K = 40, 50, 77
    g = torch.Generator().manual_seed(9)
    a, b = torch.randn((M, K), generator=g).to(torch.float8_e5m2), torch.randn((K, N), generator=g).to(torch.float8_e5m2)
    a[3, 5], a[7, 76], b[20, 9], b[76, 49] = float("nan"), float("inf"), float("-inf"), float("nan")
    buf = torch.full((M * K + 33,), 0x7F, dtype=torch.uint8, device="cuda")
    buf[1:1 + M * K] = a.view(torch.uint8).reshape(-1).cuda()
    mm = ascq_gpu.Matmul(ascq_gpu.FP8_E5M2, ascq_gpu.FP8_E5M2, ascq_gpu.F32)
    mm.SetOrgShape(M, N, K)
    mm.SetTensorA(buf[1:1 + M * K])
    mm.SetTensorB(b.cuda())
    c = torch.zeros((M, N), device="cuda")
    mm.IterateAll(c)
    want = a.float() @ b.float()
    got = c.cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    f = want.isfinite()
    np.testing.assert_allclose(got[f].numpy(), want[f].numpy(), rtol=1e-5, atol=1e-4)


_LOG_SCRIPT = r"""
import sys
sys.path.insert(0, {pkg!r})
import numpy as np, torch, ascq
dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
rng = np.random.default_rng(5)
# group matmul, K = 100: the any-alignment tiles (no fallback)
x = rng.integers(-8, 8, (64, 100), dtype=np.int8)
w = rng.integers(-8, 8, (2, 100, 96), dtype=np.int8)
ascq.quant_group_matmul(dev(x), dev(np.ones(64, np.float32)), dev(w), dev(np.ones((2, 96), np.float32)),
                        dev(np.array([0, 30, 64], np.int64)), 0, False, torch.bfloat16)
torch.cuda.synchronize()
print("step group done", file=sys.stderr, flush=True)
# fp8 Matmul with B given [K, N], K = 40 and a workspace without room to pack the operands: the generic kernel
mm = ascq.Matmul(ascq.FP8_E4M3, ascq.FP8_E4M3, ascq.F32)
mm.SetOrgShape(32, 32, 40)
mm.SetWorkspace(dev(np.zeros(16, np.uint8)), 16)
mm.SetTensorA(dev(np.full((32, 40), 0x38, np.uint8)))
mm.SetTensorB(dev(np.full((40, 32), 0x38, np.uint8)), False)
c = torch.empty((32, 32), dtype=torch.float32, device="cuda")
mm.IterateAll(c)
mm.End()
torch.cuda.synchronize()
assert (c == 40.0).all(), c
print("step fp8 done", file=sys.stderr, flush=True)
"""


def test_fallback_logged_under_ascq_log():
    """ASCQ_LOG=1: a launch that takes a generic kernel prints 'ascq: fallback: <kernel> (<reason>)' on stderr;
    the any-alignment tiles print nothing.  One child process (the level is read once per process)."""
    code = _LOG_SCRIPT.format(pkg=str(ROOT / "asc-devkit_clone_amd"))
    env = dict(os.environ, ASCQ_LOG="1")
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=240)
    assert r.returncode == 0, r.stderr[-2000:]
    lines = [ln for ln in r.stderr.splitlines() if ln.startswith("ascq:")]
    assert lines == ["ascq: fallback: gemm_f8_generic_kernel (B given [K, N] with K not a multiple of 16 or operands "
                     "not aligned)"], r.stderr[-2000:]


@pytest.mark.parametrize("where", ["owned", "reported", "scratch"])
@pytest.mark.parametrize("org,single,b_off", [((1000, 4096, 8200), (16, 4096, 8192), 0), ((16, 8192, 8192), (16, 4096, 8192), 4),
                                              ((128, 4096, 8192), (40, 4096, 8192), 1)])
@pytest.mark.parametrize("fp8", [False, True])
def test_packed_operands_beside_split_partials(ascq_gpu, oracle, fp8, org, single, b_off, where):
    """B [N, K] rows off their alignment (packed), an org shape without the K split across workgroups and a single shape
    with it: the split's partials and the packed operands are both in use.  Integer-valued operands, exact sums"""
    ascq = ascq_gpu
    (M, N, K), (m, n, k) = org, single
    rng = seeded(M + K + b_off)
    A = rng.integers(-4, 5, (M, K), dtype=np.int8)
    B = rng.integers(-4, 5, (N, K), dtype=np.int8)
    ref = torch.from_numpy(A[:m, :k]).float() @ torch.from_numpy(B[:n, :k]).float().t()  # (below 2^18: exact)
    code = (lambda v: torch.from_numpy(v).float().to(torch.float8_e4m3fn).view(torch.uint8).numpy()) if fp8 else (lambda v: v)
    mm = ascq.Matmul(ascq.FP8_E4M3, ascq.FP8_E4M3, ascq.F32) if fp8 else ascq.Matmul(ascq.INT8, ascq.INT8, ascq.INT32)
    mm.SetOrgShape(M, N, K)
    mm.SetSingleShape(m, n, k)
    mm.SetTensorA(_dev(code(A)))
    mm.SetTensorB(_dev_at(code(B), b_off), True)
    if where == "reported":
        nbytes = mm.WorkspaceSize()
        mm.SetWorkspace(torch.empty(nbytes, dtype=torch.uint8, device="cuda"), nbytes)
    c = torch.zeros((M, N), dtype=torch.float32 if fp8 else torch.int32, device="cuda")
    for _ in range(3):
        c.zero_()
        (mm.IterateAllNoAlloc if where == "scratch" else mm.IterateAll)(c)
        assert torch.equal(c[:m, :n].cpu().float(), ref)
    assert not bool(c[m:].any()) and not bool(c[:, n:].any())
