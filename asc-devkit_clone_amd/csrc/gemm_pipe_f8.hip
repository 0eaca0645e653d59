// gemm_pipe_f8.hip -- the fp8 Matmul on the pipelined tiles of gemm_pipe.h: the GEMM and epilogues of gemm_f8.hip for
// A [M, K] with 16-byte-aligned rows and B [N, K] the same, or B [K, N] with 4-byte-aligned rows; K a multiple of 16.
#include "common.h"
#include "gemm_pipe.h"
#include "launch.h"

namespace ascq {

template <int BM, int BN, int WM, int WN, int FMT, bool BTR>
__global__ __launch_bounds__(WM * WN * 64, 2) void gemm_f8_pipe_kernel(GemmF8Args p)
{
    using T = GemmPipe<BM, BN, WM, WN, OP_F8, FMT, BTR>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem_f8[];
    int tm, tn;
    pipe_tile((int)blockIdx.x, (int)((p.M + BM - 1) / BM), (int)((p.N + BN - 1) / BN), tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int rows = (int)(p.M - m0 < BM ? p.M - m0 : BM), cols = (int)(p.N - n0 < BN ? p.N - n0 : BN);
    PipeArgs c{};
    c.a = make_rsrc4(p.A, (uint32_t)(p.lda * (p.M - 1) + p.K));
    c.b = make_rsrc4(p.B, (uint32_t)(BTR ? p.ldb * (p.K - 1) + (p.N + 3) / 4 * 4 : p.ldb * (p.N - 1) + p.K));
    c.lda = (uint32_t)p.lda;
    c.ldb = (uint32_t)p.ldb;
    c.a0 = (uint32_t)(m0 * p.lda);
    c.b0 = (uint32_t)(BTR ? n0 : n0 * p.ldb);
    c.kbytes = (int32_t)p.K;
    ColLds col;  // (without a quant word the sums are multiplied by 1)
    col.request(smem_f8 + T::LDS_BYTES, T::NW, p.bias, 0x80000000u, p.use_quant ? p.qvec : nullptr,
                p.use_quant ? p.qscalar : 0x3F800000u, n0, cols);
    typename T::acc_t acc[T::FM][T::FN];
    T::run(c, smem_f8, acc);

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave / WN, wn = wave % WN;
    auto value = [](float v, const ColWords& w, int e) { return (v + __uint_as_float(w.bias[e])) * w.m1[e]; };
    if (p.c_type == DT_INT4) {  // (V)QF322S4_PRE
        const TileOut o4 = tile_out_int4(p.C, m0, n0, p.ldc, rows, cols);
        ct_store<T, OUT_I4>(o4, ((uintptr_t)p.C | (uintptr_t)o4.pitch) % 4 == 0, cols, acc, wm, wn, lane, col,
                       [&](float a, const ColWords& w, int e) {
                           return requant4(value(a, w, e), w.lo[e] | ((uint64_t)w.hi[e] << 32));
                       });
        return;
    }
    const int esize = p.c_type == DT_F32 ? 4 : ((p.c_type == DT_F16 || p.c_type == DT_BF16) ? 2 : 1);
    const TileOut out = tile_out(p.C, m0, n0, p.ldc, rows, cols, esize);
    const bool vec = ((uintptr_t)p.C | (uintptr_t)out.pitch) % 4 == 0;
    auto at = [&](int cl, uint32_t a) { return (__uint_as_float(a) + __uint_as_float(col.bias(cl))) * quant_pre_m1(col.word(cl)); };
    if (p.atomic != C_STORE) {  // enAtomic: f32 / f16 / bf16 C (the host layer refuses the others)
        // (the parked accumulators overwrite the main loop's ring, not the column words behind it)
        if (p.c_type == DT_F32)
            atomic_epilogue<T, DT_F32>(smem_f8, acc, out, rows, cols, p.atomic,
                                       [&](int cl, uint32_t a) { return __float_as_uint(at(cl, a)); });
        else if (p.c_type == DT_F16)
            atomic_epilogue<T, DT_F16>(smem_f8, acc, out, rows, cols, p.atomic,
                                       [&](int cl, uint32_t a) { return (uint32_t)f32_to_f16_sat(at(cl, a)); });
        else
            atomic_epilogue<T, DT_BF16>(smem_f8, acc, out, rows, cols, p.atomic,
                                        [&](int cl, uint32_t a) { return (uint32_t)f32_to_bf16_sat(at(cl, a)); });
        return;
    }
    if (p.c_type == DT_F32)
        ct_store<T, OUT_4>(out, true, cols, acc, wm, wn, lane, col,
                           [&](float a, const ColWords& w, int e) { return __float_as_uint(value(a, w, e)); });
    else if (p.c_type == DT_F16) ct_store<T, OUT_F16>(out, vec, cols, acc, wm, wn, lane, col, value);
    else if (p.c_type == DT_BF16) ct_store<T, OUT_BF16>(out, vec, cols, acc, wm, wn, lane, col, value);
    else  // the 1-byte C types in the rolled epilogue (the hifloat8 encoder alone is ~30 instructions per element)
        rolled_epilogue<T>(smem_f8, acc, rows, cols, [&](int rr, int cc, uint32_t a) {
            __builtin_amdgcn_raw_buffer_store_b8(byte_out(at(cc, a), col.word(cc), p.c_type), out.r,
                                                 (uint32_t)rr * out.pitch + (uint32_t)cc, 0, 0);
        });
}

template <int BM, int BN, int WM, int WN, int FMT, bool BTR>
static hipError_t launch_f8_pipe(const GemmF8Args& a, hipStream_t st)
{
    using T = GemmPipe<BM, BN, WM, WN, OP_F8, FMT, BTR>;
    constexpr int LDS = (int)T::LDS_BYTES + ColLds::BYTES;
    const int tiles = (int)(((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN));
    const hipError_t e = ensure_dynamic_lds<gemm_f8_pipe_kernel<BM, BN, WM, WN, FMT, BTR>>(LDS);
    if (e != hipSuccess) return e;
    launch_k((gemm_f8_pipe_kernel<BM, BN, WM, WN, FMT, BTR>), dim3(tiles), dim3(T::NT), LDS, st, a);
    return hipGetLastError();
}

template <int FMT, bool BTR>
static hipError_t launch_f8_pipe_layout(const GemmF8Args& a, hipStream_t st)
{
    // (f32 C combined by enAtomic is bound by the exchanges of a CU: the smallest tiles, M = 1000, N = 2052, K = 272: 55 us
    // on 128 x 128)
    const bool f32_atomic = a.atomic != C_STORE && a.c_type == DT_F32 && !(a.M >= 1024 && a.N >= 1024);
    switch (f32_atomic ? PIPE_64x128 : pick_pipe_tile(a.M, a.N, a.K)) {
    case PIPE_256x256: return launch_f8_pipe<256, 256, 2, 4, FMT, BTR>(a, st);
    case PIPE_192x256: return launch_f8_pipe<192, 256, 2, 4, FMT, BTR>(a, st);
    case PIPE_256x192: return launch_f8_pipe<256, 192, 4, 2, FMT, BTR>(a, st);
    case PIPE_128x256: return launch_f8_pipe<128, 256, 2, 4, FMT, BTR>(a, st);
    case PIPE_128x192: return launch_f8_pipe<128, 192, 4, 2, FMT, BTR>(a, st);
    case PIPE_128x128: return launch_f8_pipe<128, 128, 2, 2, FMT, BTR>(a, st);
    default: return launch_f8_pipe<64, 128, 2, 2, FMT, BTR>(a, st);
    }
}
template <int FMT>
static hipError_t launch_f8_pipe_fmt(const GemmF8Args& a, hipStream_t st)
{
    return a.trans_b ? launch_f8_pipe_layout<FMT, false>(a, st) : launch_f8_pipe_layout<FMT, true>(a, st);
}

hipError_t launch_gemm_f8_pipe(const GemmF8Args& a, hipStream_t st)
{
    switch (a.fmt_a | (a.fmt_b << 3)) {
    case F8F6F4_E4M3 | (F8F6F4_E4M3 << 3): return launch_f8_pipe_fmt<F8F6F4_E4M3 | (F8F6F4_E4M3 << 3)>(a, st);
    case F8F6F4_E5M2 | (F8F6F4_E5M2 << 3): return launch_f8_pipe_fmt<F8F6F4_E5M2 | (F8F6F4_E5M2 << 3)>(a, st);
    case F8F6F4_E4M3 | (F8F6F4_E5M2 << 3): return launch_f8_pipe_fmt<F8F6F4_E4M3 | (F8F6F4_E5M2 << 3)>(a, st);
    case F8F6F4_E5M2 | (F8F6F4_E4M3 << 3): return launch_f8_pipe_fmt<F8F6F4_E5M2 | (F8F6F4_E4M3 << 3)>(a, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace ascq
