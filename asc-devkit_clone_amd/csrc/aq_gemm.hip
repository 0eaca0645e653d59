// aq_gemm.hip -- weight-only antiquant matmul (W8A16 / W4A16) above the decode shapes (M > 64) on gfx950.
//
// Reference: AscendAntiQuant per group (include/adv_api/quantization/ascend_antiquant.h:47-62;
// impl/adv_api/detail/quantization/antiquant/ascend_antiquant_impl.h:63-96, 366-411) composed with a half Matmul whose
// L0C is fp32 (impl/adv_api/detail/matmul/utils/matmul_utils.h:171-174): y = f16( x @ w_f16 ), fp32 accumulation,
// w_f16 = half( half(q + offset) * scale ) per group of K.
//
// The decode kernels (gemv_antiquant.hip) dequantise each weight fragment in registers for a block of at most 128 rows.
// Here the half-tile pipeline of gemm_pipe.h multiplies tiles of up to 256 rows on v_mfma_f32_16x16x32_f16, x copied
// straight to LDS and each packed weight dequantised once per tile, one fragment per wave under each phase's MFMAs.
// Packed layout (ascq_weight_pack): 16-column x 128-k tiles, lane l holding column l % 16 and, per 32-k step j,
// k = 32 j + 8 (l / 16) .. + 7.
#include "common.h"
#include "gemm_pipe.h"
#include "launch.h"

namespace ascq {

struct AqGemmArgs {
    uint16_t* y;            // [M, N] f16
    const uint16_t* x;      // [M, K] f16
    const uint8_t* wp;      // packed weight
    const uint16_t* scale;  // [K / g, N] f16
    const uint16_t* offset; // [K / g, N] f16 or null
    uint32_t M, N, K;
    uint32_t gshift;        // g = 64 << gshift; 31: one group over all of K
    uint32_t x_bytes, w_bytes, s_bytes;
    int atomic;
};

struct NoCols {};

// FMT: bit 0 int4, bit 1 offsets
template <int BM, int BN, int WM, int WN, int FMT>
__global__ __launch_bounds__(WM * WN * 64, 2) void aq_pipe_kernel(AqGemmArgs p)
{
    using T = GemmPipe<BM, BN, WM, WN, OP_AQ, FMT>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem_aq[];
    int tm, tn;
    pipe_tile((int)blockIdx.x, (int)((p.M + BM - 1) / BM), (int)((p.N + BN - 1) / BN), tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int rows = (int)(p.M - m0 < BM ? p.M - m0 : BM), cols = (int)(p.N - n0 < BN ? p.N - n0 : BN);
    PipeArgs c{};
    c.a = make_rsrc4(p.x, p.x_bytes);
    c.lda = p.K * 2;
    c.a0 = (uint32_t)m0 * p.K * 2;
    c.kbytes = (int32_t)(p.K * 2);
    c.wp = p.wp;
    c.scale = p.scale;
    c.offset = p.offset;
    c.w_bytes = p.w_bytes;
    c.s_bytes = p.s_bytes;
    c.n = p.N;
    c.n0 = (uint32_t)n0;
    c.gshift = p.gshift;
    typename T::acc_t acc[T::FM][T::FN];
    T::run(c, smem_aq, acc);

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave / WN, wn = wave % WN;
    const TileOut out = tile_out(p.y, m0, n0, p.N, rows, cols, 2);
    if (p.atomic != C_STORE)
        atomic_epilogue<T, DT_F16>(smem_aq, acc, out, rows, cols, p.atomic,
                                   [](int, uint32_t a) { return (uint32_t)f32_to_f16_sat(__uint_as_float(a)); });
    else
        ct_store<T, OUT_F16>(out, (uintptr_t)p.y % 4 == 0, cols, acc, wm, wn, lane, [](int) { return NoCols{}; },
                             [](float v, const NoCols&, int) { return v; });
}

template <int BM, int BN, int WM, int WN>
static hipError_t launch_aq_pipe(const AqGemmArgs& a, bool int4, hipStream_t st)
{
    const unsigned tiles = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
    auto go = [&](auto F) -> hipError_t {
        constexpr int FMT = decltype(F)::value;
        using T = GemmPipe<BM, BN, WM, WN, OP_AQ, FMT>;
        constexpr auto kern = aq_pipe_kernel<BM, BN, WM, WN, FMT>;
        const hipError_t e = ensure_dynamic_lds<kern>((int)T::LDS_BYTES);
        if (e != hipSuccess) return e;
        launch_k(kern, dim3(tiles), dim3(T::NT), (uint32_t)T::LDS_BYTES, st, a);
        return hipGetLastError();
    };
    if (int4) return a.offset ? go(std::integral_constant<int, 3>{}) : go(std::integral_constant<int, 1>{});
    return a.offset ? go(std::integral_constant<int, 2>{}) : go(std::integral_constant<int, 0>{});
}

// The tile of a problem and about what it takes in microseconds, from times of every tile at M = 96 .. 3072, (N, K) =
// (4096 | 11008, 4096), (4096, 11008), int4, g = 128 (int8 within 5 %).  A CU runs c = ceil(tiles / 256) tiles; `fill` is
// the share of the c rounds that has work.  Per 64-k stage and tile: 256 x 192 1.10 us with few CUs at work to 1.25 with
// all, 128 x 192 0.80 - 0.86, 128 x 128 0.65, or side by side on a CU 0.40 - 0.57, 64 x 128 0.55, or 0.40.  E.g.
// 3072 x 11008 x 4096: 253 us against 301 (128 x 128) and 328 (128 x 192); 1024 x 4096 x 11008: 121 (128 x 128) against
// 143 (64 x 128), 145, 196 (256 x 192); 192 x 4096 x 4096: 39 (64 x 128) against 45, 55, 76.  256 x 128, 192 x 256 and
// 128 x 256 tiles came in behind these everywhere, 256 x 256 ones spill.
enum AqTile { AQ_256x192, AQ_128x192, AQ_128x128, AQ_64x128, AQ_TILES };
struct AqPick {
    AqTile tile;
    float us;
};
static AqPick pick_aq_tile(int64_t M, int64_t N, int64_t K)
{
    static const struct {
        int bm, bn;
        float solo, full, tail;      // one tile per CU
        float more_solo, more_full;  // more than one
        float more_tail;
    } T[AQ_TILES] = {{256, 192, 1.10f, 1.25f, 6.0f, 1.10f, 1.25f, 6.0f},
                     {128, 192, 0.80f, 0.86f, 5.0f, 0.80f, 0.86f, 5.0f},
                     {128, 128, 0.65f, 0.66f, 5.0f, 0.40f, 0.57f, 0.0f},
                     {64, 128, 0.55f, 0.55f, 4.5f, 0.40f, 0.40f, 0.0f}};
    const float stages = (float)(K / 64);
    AqPick best{AQ_256x192, 0.0f};
    for (int t = 0; t < AQ_TILES; ++t) {
        const int64_t tiles = ((M + T[t].bm - 1) / T[t].bm) * ((N + T[t].bn - 1) / T[t].bn);
        const float c = (float)((tiles + 255) / 256), fill = (float)tiles / (256.0f * c);
        const float us = c > 1.0f ? c * ((T[t].more_solo + (T[t].more_full - T[t].more_solo) * fill) * stages + T[t].more_tail)
                                  : (T[t].solo + (T[t].full - T[t].solo) * fill) * stages + T[t].tail;
        if (t == 0 || us < best.us) best = {(AqTile)t, us};
    }
    return best;
}

float aq_gemm_us(int64_t M, int64_t N, int64_t K) { return pick_aq_tile(M, N, K).us; }

// K % 128 == 0, N % 16 == 0, group 64 << s or all of K (checked here), every buffer below 2^31 - 2^16 bytes
hipError_t launch_aq_gemm(uint16_t* y, const uint16_t* x, const void* wp, int w_type, const uint16_t* scale,
                          const uint16_t* offset, int64_t group, int64_t M, int64_t N, int64_t K, int atomic,
                          hipStream_t st)
{
    const int64_t g = group > 0 && group < K ? group : K;
    const bool int4 = w_type == DT_INT4;
    const uint64_t lim = 0x7FFF0000ull;
    const uint64_t w_bytes = (uint64_t)K * N / (int4 ? 2 : 1), s_bytes = (uint64_t)((K + g - 1) / g) * N * 2;
    const uint64_t x_bytes = (uint64_t)M * K * 2;
    if (K % 128 != 0 || N % 16 != 0 || (g != K && (g % 64 != 0 || ((g / 64) & (g / 64 - 1)) != 0)) || w_bytes >= lim ||
        s_bytes >= lim || x_bytes >= lim || M * N >= (int64_t)lim)
        return hipErrorInvalidValue;
    AqGemmArgs a;
    a.y = y;
    a.x = x;
    a.wp = (const uint8_t*)wp;
    a.scale = scale;
    a.offset = offset;
    a.M = (uint32_t)M;
    a.N = (uint32_t)N;
    a.K = (uint32_t)K;
    a.gshift = g == K ? 31u : (uint32_t)__builtin_ctzll((unsigned long long)(g / 64));
    a.x_bytes = (uint32_t)x_bytes;
    a.w_bytes = (uint32_t)w_bytes;
    a.s_bytes = (uint32_t)s_bytes;
    a.atomic = atomic;
    switch (pick_aq_tile(M, N, K).tile) {
    case AQ_256x192: return launch_aq_pipe<256, 192, 4, 2>(a, int4, st);
    case AQ_128x192: return launch_aq_pipe<128, 192, 4, 2>(a, int4, st);
    case AQ_128x128: return launch_aq_pipe<128, 128, 2, 2>(a, int4, st);
    default: return launch_aq_pipe<64, 128, 2, 2>(a, int4, st);
    }
}

}  // namespace ascq
