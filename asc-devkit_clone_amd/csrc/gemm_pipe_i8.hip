// gemm_pipe_i8.hip -- the int8 Matmul on the pipelined tiles of gemm_pipe.h: the GEMM and epilogues of gemm_i8.hip for
// A [M, K] with 16-byte-aligned rows and B [N, K] the same, or B [K, N] with 4-byte-aligned rows (whose range
// is rounded up to whole dwords: they lie in the row's pitch).
#include "common.h"
#include "gemm_pipe.h"
#include "launch.h"

namespace ascq {

template <int BM, int BN, int WM, int WN, bool BTR>
__global__ __launch_bounds__(WM * WN * 64, 2) void gemm_i8_pipe_kernel(GemmI8Args p)
{
    using T = GemmPipe<BM, BN, WM, WN, OP_I8, 0, BTR>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    int tm, tn;
    pipe_tile((int)blockIdx.x, (int)((p.M + BM - 1) / BM), (int)((p.N + BN - 1) / BN), tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int rows = (int)(p.M - m0 < BM ? p.M - m0 : BM), cols = (int)(p.N - n0 < BN ? p.N - n0 : BN);
    PipeArgs c{};
    c.a = make_rsrc4(p.A, (uint32_t)(p.lda * (p.M - 1) + (p.K + 15) / 16 * 16));  // (whole chunks: within the pitch)
    c.b = make_rsrc4(p.B, (uint32_t)(BTR ? p.ldb * (p.K - 1) + (p.N + 3) / 4 * 4 : p.ldb * (p.N - 1) + p.K));
    c.lda = (uint32_t)p.lda;
    c.ldb = (uint32_t)p.ldb;
    c.a0 = (uint32_t)(m0 * p.lda);
    c.b0 = (uint32_t)(BTR ? n0 : n0 * p.ldb);
    c.kbytes = (int32_t)p.K;
    ColLds col;
    col.request(smem + T::LDS_BYTES, T::NW, p.bias, 0u, p.qvec, p.qscalar, n0, cols);
    typename T::acc_t acc[T::FM][T::FN];
    T::run(c, smem, acc);

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave / WN, wn = wave % WN;
    // acc + bias (int32, wrapping), then x M1
    auto sum = [](int32_t a, const ColWords& w, int e) { return (int32_t)((uint32_t)a + w.bias[e]); };
    auto value = [&](int32_t a, const ColWords& w, int e) { return (float)sum(a, w, e) * w.m1[e]; };
    auto word = [](const ColWords& w, int e) { return w.lo[e] | ((uint64_t)w.hi[e] << 32); };
    if (p.epi == EPI_REQ4) {  // (V)REQ4: int4 codes, two per byte
        const TileOut o4 = tile_out_int4(p.C, m0, n0, p.ldc, rows, cols);
        ct_store<T, OUT_I4>(o4, ((uintptr_t)p.C | (uintptr_t)o4.pitch) % 4 == 0, cols, acc, wm, wn, lane, col,
                            [&](int32_t a, const ColWords& w, int e) { return requant4(value(a, w, e), word(w, e)); });
        return;
    }
    const int esize = p.epi == EPI_I32 ? 4 : (p.epi == EPI_REQ8 ? 1 : 2);
    const TileOut out = tile_out(p.C, m0, n0, p.ldc, rows, cols, esize);
    const bool vec = ((uintptr_t)p.C | (uintptr_t)out.pitch) % 4 == 0;
    if (p.atomic != C_STORE) {  // enAtomic: int32 / f16 / bf16 C (the host layer refuses the others)
        // (the parked accumulators overwrite the main loop's ring, not the column words behind it)
        auto v = [&](int cl, uint32_t a) { return (int32_t)(a + col.bias(cl)); };
        auto f = [&](int cl, uint32_t a) { return (float)v(cl, a) * quant_pre_m1(col.word(cl)); };
        if (p.epi == EPI_I32)
            atomic_epilogue<T, DT_INT32>(smem, acc, out, rows, cols, p.atomic,
                                         [&](int cl, uint32_t a) { return (uint32_t)v(cl, a); });
        else if (p.epi == EPI_DEQ_F16)
            atomic_epilogue<T, DT_F16>(smem, acc, out, rows, cols, p.atomic,
                                       [&](int cl, uint32_t a) { return (uint32_t)f32_to_f16_sat(f(cl, a)); });
        else
            atomic_epilogue<T, DT_BF16>(smem, acc, out, rows, cols, p.atomic,
                                        [&](int cl, uint32_t a) { return (uint32_t)f32_to_bf16_sat(f(cl, a)); });
        return;
    }
    if (p.epi == EPI_I32)
        ct_store<T, OUT_4>(out, true, cols, acc, wm, wn, lane, col,
                           [&](int32_t a, const ColWords& w, int e) { return (uint32_t)sum(a, w, e); });
    else if (p.epi == EPI_DEQ_F16) ct_store<T, OUT_F16>(out, vec, cols, acc, wm, wn, lane, col, value);
    else if (p.epi == EPI_DEQ_BF16) ct_store<T, OUT_BF16>(out, vec, cols, acc, wm, wn, lane, col, value);
    else
        ct_store<T, OUT_1>(out, vec, cols, acc, wm, wn, lane, col, [&](int32_t a, const ColWords& w, int e) {
            return (uint32_t)requant8(value(a, w, e), word(w, e));
        });
}

template <int BM, int BN, int WM, int WN, bool BTR>
static hipError_t launch_i8_pipe(const GemmI8Args& a, hipStream_t st)
{
    using T = GemmPipe<BM, BN, WM, WN, OP_I8, 0, BTR>;
    constexpr int LDS = (int)T::LDS_BYTES + ColLds::BYTES;
    const int tiles = (int)(((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN));
    const hipError_t e = ensure_dynamic_lds<gemm_i8_pipe_kernel<BM, BN, WM, WN, BTR>>(LDS);
    if (e != hipSuccess) return e;
    launch_k((gemm_i8_pipe_kernel<BM, BN, WM, WN, BTR>), dim3(tiles), dim3(T::NT), LDS, st, a);
    return hipGetLastError();
}

template <bool BTR>
static hipError_t launch_i8_pipe_layout(const GemmI8Args& a, hipStream_t st)
{
    switch (pick_pipe_tile(a.M, a.N, a.K)) {
    case PIPE_256x256: return launch_i8_pipe<256, 256, 2, 4, BTR>(a, st);
    case PIPE_192x256: return launch_i8_pipe<192, 256, 2, 4, BTR>(a, st);
    case PIPE_256x192: return launch_i8_pipe<256, 192, 4, 2, BTR>(a, st);
    case PIPE_128x256: return launch_i8_pipe<128, 256, 2, 4, BTR>(a, st);
    case PIPE_128x192: return launch_i8_pipe<128, 192, 4, 2, BTR>(a, st);
    case PIPE_128x128: return launch_i8_pipe<128, 128, 2, 2, BTR>(a, st);
    default: return launch_i8_pipe<64, 128, 2, 2, BTR>(a, st);
    }
}

hipError_t launch_gemm_i8_pipe(const GemmI8Args& a, hipStream_t st)
{
    return a.trans_b ? launch_i8_pipe_layout<false>(a, st) : launch_i8_pipe_layout<true>(a, st);
}

}  // namespace ascq
