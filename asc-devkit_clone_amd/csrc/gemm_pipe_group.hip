// gemm_pipe_group.hip -- the quantized group matmul (MoE) above decode size on the pipelined tiles of gemm_pipe.h: X
// [M, K] int8 with 16-byte-aligned rows, W [G, N, K] the same or [G, K, N] with 4-byte-aligned rows, K a multiple of 16.
// Tiles and their order are group_tile.h's; the epilogue is gemm_i8.hip's (quant_group_matmul_custom.asc:424-452):
// AscendDequant acc x scale[g, n] in fp32 (its int32 -> fp32 conversion rounds ties away from zero above 2^24), x the
// per-token scale in fp32, optional FasterGelu, one rounding to the output type.
#include "common.h"
#include "gemm_pipe.h"
#include "group_tile.h"
#include "launch.h"

namespace ascq {

template <int BM, int BN, int WM, int WN, bool BTR>
__global__ __launch_bounds__(WM * WN * 64, 2) void group_gemm_pipe_kernel(GroupGemmArgs p)
{
    using T = GemmPipe<BM, BN, WM, WN, OP_I8, 0, BTR>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    GroupTile tile;
    if (!find_group_tile<T::NT, BM, BN>(p, tile)) return;
    const int rows = (int)(tile.m_end - tile.m0 < BM ? tile.m_end - tile.m0 : BM);
    const int cols = (int)(p.N - tile.n0 < BN ? p.N - tile.n0 : BN);
    PipeArgs c{};
    c.a = make_rsrc4(p.X, (uint32_t)(p.M * p.K));
    c.b = make_rsrc4(p.W + (int64_t)tile.g * p.K * p.N, (uint32_t)(p.K * p.N));
    c.lda = (uint32_t)p.K;
    c.ldb = (uint32_t)(BTR ? p.N : p.K);
    c.a0 = (uint32_t)(tile.m0 * p.K);
    c.b0 = (uint32_t)(BTR ? tile.n0 : tile.n0 * p.K);
    c.kbytes = (int32_t)p.K;
    // the epilogue's scales go to LDS now, behind the ring: older than the main loop's copies, whose first wait covers
    // them.  Rows past the group and columns past N read 0.
    float* s_pt = (float*)(smem + T::LDS_BYTES);
    float* s_sc = s_pt + 256;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (wave == 0) dma16(make_rsrc4(p.pts + tile.m0, (uint32_t)rows * 4u), lds_addr(s_pt), (uint32_t)lane * 16u);
    else if (wave == 1)
        dma16(make_rsrc4(p.scale + (int64_t)tile.g * p.N + tile.n0, (uint32_t)cols * 4u), lds_addr(s_sc), (uint32_t)lane * 16u);
    typename T::acc_t acc[T::FM][T::FN];
    T::run(c, smem, acc);

    const int wm = wave / WN, wn = wave % WN;
    const TileOut out = tile_out(p.Y, tile.m0, tile.n0, p.N, rows, cols, 2);
    const bool vec = ((uintptr_t)p.Y | (uintptr_t)out.pitch) % 4 == 0;
    auto cols4 = [&](int cl) { return *(const v4f*)(s_sc + cl); };
    auto plain = [&](int32_t a, const v4f& sc, int e, int row) { return i32_to_f32_rna(a) * sc[e] * s_pt[row]; };
    auto gelu = [&](int32_t a, const v4f& sc, int e, int row) { return faster_gelu(i32_to_f32_rna(a) * sc[e] * s_pt[row]); };
    if (p.out_type == DT_F16) {
        if (p.act) ct_store<T, OUT_F16>(out, vec, cols, acc, wm, wn, lane, cols4, gelu);
        else ct_store<T, OUT_F16>(out, vec, cols, acc, wm, wn, lane, cols4, plain);
    } else {
        if (p.act) ct_store<T, OUT_BF16>(out, vec, cols, acc, wm, wn, lane, cols4, gelu);
        else ct_store<T, OUT_BF16>(out, vec, cols, acc, wm, wn, lane, cols4, plain);
    }
}

template <int BM, int BN, int WM, int WN, bool BTR>
static hipError_t launch_group_pipe_tile(const GroupGemmArgs& a, hipStream_t st)
{
    using T = GemmPipe<BM, BN, WM, WN, OP_I8, 0, BTR>;
    constexpr int LDS = (int)T::LDS_BYTES + 2048;
    const int64_t upper = ((a.M + BM - 1) / BM + a.G) * ((a.N + BN - 1) / BN);  // tiles, at most
    const hipError_t e = ensure_dynamic_lds<group_gemm_pipe_kernel<BM, BN, WM, WN, BTR>>(LDS);
    if (e != hipSuccess) return e;
    launch_k((group_gemm_pipe_kernel<BM, BN, WM, WN, BTR>), dim3((unsigned)((upper + 7) / 8 * 8)), dim3(T::NT), LDS, st, a);
    return hipGetLastError();
}

template <bool BTR>
static hipError_t launch_group_pipe_layout(const GroupGemmArgs& a, hipStream_t st)
{
    switch ((int)pick_pipe_tile(a.M, a.N, a.K, a.G)) {
    case PIPE_256x256: return launch_group_pipe_tile<256, 256, 2, 4, BTR>(a, st);
    case PIPE_192x256: return launch_group_pipe_tile<192, 256, 2, 4, BTR>(a, st);
    case PIPE_256x192: return launch_group_pipe_tile<256, 192, 4, 2, BTR>(a, st);
    case PIPE_128x256: return launch_group_pipe_tile<128, 256, 2, 4, BTR>(a, st);
    case PIPE_128x192: return launch_group_pipe_tile<128, 192, 4, 2, BTR>(a, st);
    case PIPE_128x128: return launch_group_pipe_tile<128, 128, 2, 2, BTR>(a, st);
    default: return launch_group_pipe_tile<64, 128, 2, 2, BTR>(a, st);
    }
}

hipError_t launch_group_pipe(const GroupGemmArgs& a, hipStream_t st)
{
    return a.w_trans ? launch_group_pipe_layout<false>(a, st) : launch_group_pipe_layout<true>(a, st);
}

}  // namespace ascq
