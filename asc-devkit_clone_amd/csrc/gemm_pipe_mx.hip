// gemm_pipe_mx.hip -- the MX-FP4 Matmul (E2M1 elements, E8M0 block scales) above decode size on the pipelined tiles of
// gemm_pipe.h: A [M, K / 2] and B [N, K / 2] with K a multiple of 128, the scales rearranged stage-major first.
#include "common.h"
#include "gemm_pipe.h"
#include "launch.h"

namespace ascq {

// stages of a problem: 256 fp4 (8 scale blocks) each
__host__ __device__ static inline int64_t pipe_mx_stages(int64_t K) { return (K + 255) / 256; }

template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(WM * WN * 64, 2) void mx_pipe_kernel(MxGemmArgs p, const uint8_t* __restrict__ sa_sm,
                                                                  const uint8_t* __restrict__ sb_sm)
{
    using T = GemmPipe<BM, BN, WM, WN, OP_MXFP4>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem_mx[];
    int tm, tn;
    pipe_tile((int)blockIdx.x, (int)((p.M + BM - 1) / BM), (int)((p.N + BN - 1) / BN), tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN, KB = p.K / 2;
    const int rows = (int)(p.M - m0 < BM ? p.M - m0 : BM), cols = (int)(p.N - n0 < BN ? p.N - n0 : BN);
    PipeArgs c{};
    c.a = make_rsrc4(p.A, (uint32_t)(p.M * KB));
    c.b = make_rsrc4(p.B, (uint32_t)(p.N * KB));
    c.lda = c.ldb = (uint32_t)KB;
    c.a0 = (uint32_t)(m0 * KB);
    c.b0 = (uint32_t)(n0 * KB);
    c.kbytes = (int32_t)KB;
    // (one resource over both scale copies; rows past an operand's last read other scales, for rows that are dropped)
    c.aux = make_rsrc4(sa_sm, (uint32_t)(sb_sm - sa_sm) + (uint32_t)(p.N * 8 * pipe_mx_stages(p.K)));
    c.sa_off = (uint32_t)m0 * 8u;
    c.sa_stride = (uint32_t)p.M * 8u;
    c.sb_off = (uint32_t)(sb_sm - sa_sm) + (uint32_t)n0 * 8u;
    c.sb_stride = (uint32_t)p.N * 8u;
    ColLds col;
    col.request(smem_mx + T::LDS_BYTES, T::NW, p.bias, 0x80000000u, nullptr, 0x3F800000u, n0, cols);
    typename T::acc_t acc[T::FM][T::FN];
    T::run(c, smem_mx, acc);

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave / WN, wn = wave % WN;
    auto value = [](float v, const ColWords& w, int e) { return v + __uint_as_float(w.bias[e]); };
    const TileOut out = tile_out(p.C, m0, n0, p.N, rows, cols, p.c_type == DT_F32 ? 4 : 2);
    if (p.atomic != C_STORE) {
        auto at = [&](int cl, uint32_t a) { return __uint_as_float(a) + __uint_as_float(col.bias(cl)); };
        if (p.c_type == DT_F32)
            atomic_epilogue<T, DT_F32>(smem_mx, acc, out, rows, cols, p.atomic,
                                       [&](int cl, uint32_t a) { return __float_as_uint(at(cl, a)); });
        else
            atomic_epilogue<T, DT_BF16>(smem_mx, acc, out, rows, cols, p.atomic,
                                        [&](int cl, uint32_t a) { return (uint32_t)f32_to_bf16_sat(at(cl, a)); });
        return;
    }
    if (p.c_type == DT_F32)
        ct_store<T, OUT_4>(out, true, cols, acc, wm, wn, lane, col,
                           [&](float a, const ColWords& w, int e) { return __float_as_uint(value(a, w, e)); });
    else
        ct_store<T, OUT_BF16>(out, ((uintptr_t)p.C | (uintptr_t)out.pitch) % 4 == 0, cols, acc, wm, wn, lane, col, value);
}

// E8M0 scales -> [stage][row][8]: block 4 s + g of a stage's eight at byte 2 g + s (the order a lane of the MFMA reads
// its two in); blocks past sK, whose elements the GEMM reads as zeros, get the scale 127 = 2^0, so no NaN code meets
// them.  pairs 0: [R, sK] row-major, 4-byte aligned; 1: [sK / 2, R, 2].  Both operands in one launch, one thread per (row, two stages):
// its sixteen blocks are one run of a row-major row.
struct MxScaleJob {
    uint8_t* dst;
    const uint8_t* src;
    int64_t R;
    int pairs;
};
__global__ __launch_bounds__(256) void mx_pipe_scale_kernel(MxScaleJob ja, MxScaleJob jb, int64_t sK, int64_t stages,
                                                            uint32_t blocks_a)
{
    const bool is_a = blockIdx.x < blocks_a;
    const MxScaleJob j = is_a ? ja : jb;
    const int64_t sp = (stages + 1) / 2, total = sp * j.R;
    const int64_t i = (int64_t)(is_a ? blockIdx.x : blockIdx.x - blocks_a) * 256 + threadIdx.x;
    if (i >= total) return;
    // neighbouring threads take the runs of one row where rows are contiguous, neighbouring rows where pairs are
    const uint32_t x = (uint32_t)i, R = (uint32_t)j.R, runs = (uint32_t)sp;
    const uint32_t r = j.pairs ? x % R : x / runs, q = j.pairs ? x / R : x % runs;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t st = 2 * q + h, b = st * 8;
        if (st >= stages) break;
        uint32_t lo, hi;  // k-step 0's blocks, k-step 1's
        if (j.pairs) {
            const uint16_t* s16 = (const uint16_t*)j.src + (int64_t)(b / 2) * R + r;
            auto pair = [&](uint32_t d) -> uint32_t { return b + 2 * d < sK ? s16[(int64_t)d * R] : 0x7F7Fu; };
            lo = pair(0) | (pair(1) << 16);
            hi = pair(2) | (pair(3) << 16);
        } else {  // (K % 128 == 0: sK is a multiple of four, so rows and runs are 4-byte aligned)
            const uint32_t* s32 = (const uint32_t*)(j.src + (int64_t)r * sK + b);
            lo = s32[0];
            hi = b + 4 < sK ? s32[1] : 0x7F7F7F7Fu;
        }
        *(u32x2*)(j.dst + ((int64_t)st * R + r) * 8) =
            (u32x2){__builtin_amdgcn_perm(hi, lo, 0x05010400u), __builtin_amdgcn_perm(hi, lo, 0x07030602u)};
    }
}

template <int BM, int BN, int WM, int WN>
static hipError_t launch_mx_pipe(const MxGemmArgs& a, const uint8_t* sa, const uint8_t* sb, hipStream_t st)
{
    using T = GemmPipe<BM, BN, WM, WN, OP_MXFP4>;
    constexpr int LDS = (int)T::LDS_BYTES + 1024;  // (bias only)
    const int tiles = (int)(((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN));
    const hipError_t e = ensure_dynamic_lds<mx_pipe_kernel<BM, BN, WM, WN>>(LDS);
    if (e != hipSuccess) return e;
    launch_k((mx_pipe_kernel<BM, BN, WM, WN>), dim3(tiles), dim3(T::NT), LDS, st, a, sa, sb);
    return hipGetLastError();
}

hipError_t launch_mx_fp4_pipe(const MxGemmArgs& a, hipStream_t st)
{
    const int64_t sK = (a.K + 63) / 64 * 2, stages = pipe_mx_stages(a.K), sp = (stages + 1) / 2;
    uint8_t* sa = a.ws_scales;
    uint8_t* sb = a.ws_scales + (a.M * stages * 8 + 16 + 255) / 256 * 256;
    const uint32_t ba = (uint32_t)((a.M * sp + 255) / 256), bb = (uint32_t)((a.N * sp + 255) / 256);
    hipLaunchKernelGGL(mx_pipe_scale_kernel, dim3(ba + bb), dim3(256), 0, st, MxScaleJob{sa, a.sA, a.M, a.sa_layout == 1},
                       MxScaleJob{sb, a.sB, a.N, a.sb_layout == 0}, sK, stages, ba);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    switch (pick_pipe_tile(a.M, a.N, a.K / 2)) {
    case PIPE_256x256: return launch_mx_pipe<256, 256, 2, 4>(a, sa, sb, st);
    case PIPE_192x256: return launch_mx_pipe<192, 256, 2, 4>(a, sa, sb, st);
    case PIPE_256x192: return launch_mx_pipe<256, 192, 4, 2>(a, sa, sb, st);
    case PIPE_128x256: return launch_mx_pipe<128, 256, 2, 4>(a, sa, sb, st);
    case PIPE_128x192: return launch_mx_pipe<128, 192, 4, 2>(a, sa, sb, st);
    case PIPE_128x128: return launch_mx_pipe<128, 128, 2, 2>(a, sa, sb, st);
    default: return launch_mx_pipe<64, 128, 2, 2>(a, sa, sb, st);
    }
}

}  // namespace ascq
