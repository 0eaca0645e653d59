// gemm_pipe.h -- the half-tile pipelined MFMA main loop of the medium and large int8 / fp8 / MX Matmuls (gfx950),
// and of the weight-only Matmul: A [M, K] K-contiguous, B [N, K] the same or (int8, fp8) [K, N].
//
// What bounds a large tile is the feed from L2 / HBM into LDS.  GemmCore's two-stage loop waits for a whole stage
// (64 KiB at 256 x 256) that was requested less than one stage of MFMAs earlier, and reads each k-step's fragments
// right in front of the MFMAs that take them, so every barrier starts with the matrix cores idle.  Here a stage (128 K
// bytes of every tile row) is four halves -- the upper and lower half of A's rows and of B's -- and the loop runs in
// phases of a quarter stage.  A phase multiplies one A half by one B half (a quadrant of the wave's accumulators)
// out of registers, reads the half that the phase after next needs first from LDS into registers, and requests one
// half from memory into the slot whose half went to registers in the phase before.  Requests so run six phases
// ahead of their reads (1.5 stages of MFMAs: 96 KiB in flight of a 128 KiB ring of two stages), no MFMA waits for an LDS
// read issued in front of it, and a barrier has MFMA operands ready in registers on its far side.
//
// Order of the halves: H(4k) = A0(k), H(4k+1) = B0(k), H(4k+2) = B1(k), H(4k+3) = A1(k).  Phase t = 4k + p:
//   p = 0: A0 B0, p = 1: A0 B1, p = 2: A1 B1, p = 3: A1 B0 -- each half is read once and consecutive phases share one;
//   it reads H(t + 2) and requests H(t + 9).  Each wave's quadrant rows are (half) x (wave row) x 32-row blocks.
// B0(k + 1) is read while B0(k) is still multiplied: it goes to the registers B1(k) has left, so the two register sets
// of B swap roles from stage to stage.
//
// MFMA: the 16x16 forms, v_mfma_i32_16x16x64_i8 and v_mfma_[scale_]f32_16x16x128_f8f6f4.  On operands that vary like
// data the matrix cores run at a power limit, and the 16x16 forms do more within it than the 32x32 ones (256
// workgroups of 8 waves multiplying out of registers, normal data, on one MI355X: int8 4.00 against 3.23 POPS, fp8 e4m3
// 4.40 against 3.85, fp4 7.44 against 6.79 PFLOP/s).  Lane l holds row l % 16; with g = l / 16, int8 and fp4 take the
// 16 bytes 16 g .. of a k-step's 64 (fp4: one MX block of 32), fp8 the 16 bytes 16 g .. and 64 + 16 g .. of its 128.
// The MFMAs take the B fragment first, so an accumulator holds the transposed 16 x 16 block: lane l holds columns
// 4 g .. 4 g + 3 of row l % 16.
//
// LDS rows of a K-contiguous operand are 128 bytes, 16-byte chunk c of row r at c ^ (r / 2 % 8): the 16 rows of a
// fragment read hit 16 distinct 16-byte bank groups, and a copy writes 1 KiB contiguous (the swizzle is applied on the
// global side).
// B given [K, N] (BTR): a half of B is its columns' 128 K rows, copied as they lie, and read with ds_read_b64_tr_b8: a
// 16-lane group g reads 8 K rows x 16 columns and lane j receives the 8 K of column j, so two reads (K rows 16 g ..
// + 7 and 16 g + 8 .. + 15) give the lane's 16 K bytes.  Chunk c of K row k lies at c ^ swz_tr(k), which spreads the 16
// pieces that two lane groups read together over 16 distinct 16-byte bank groups.
// MX-FP4: the E8M0 scales arrive stage-major, the eight of (stage, row) -- k-step s, block g of it -- at byte 2 g + s of
// its eight, and each stage's go to one of four scale slots, requested three stages ahead, one copy per wave and stage;
// a lane reads the two bytes of block g of its row and the MFMA's op_sel picks the k-step's.
// K: a lane's 16-byte chunks at or past the end of K are not read (zeros), nor are a [K, N] B's rows.  So K of K-contiguous
// operands is a multiple of 16 bytes; with an int8 B [K, N] K is any, A's bytes from K to the end of its chunk lying within
// its pitch (they meet zeros; an fp8 NaN would not vanish against them).
//
// Weight-only antiquant (OP_AQ): A is f16 (a stage is 64 k), B the packed int4 / int8 weight.  A wave loads one 16-column
// strip of a half per stage into registers (packed codes, the columns' scale and offset), six phases ahead, dequantises
// one fragment per phase under its MFMAs and writes it to the half's rows in LDS at the top of the next phase, so each
// weight is dequantised once per tile.  B0(k + 1) is written in phases 0 and 1 of stage k, B1(k + 1) in phases 2 and 3:
// after the reads of B0(k) and B1(k), so B's ring is one stage.  (Two stages' codes per load, eight phases ahead, measured
// the same to 5 % slower; copies of the kernel without the weight loads took 15 - 20 % less, without the dequantisation
// the same time.)
#pragma once

#include "aq_frag.h"
#include "gemm_core.h"

namespace ascq {

// A buffer resource as four dwords, and its copy of 16 bytes per lane into LDS at `lds` (a byte address, wave-uniform)
// + 16 * lane.  Written in assembly because through the builtin the compiler takes every later LDS transpose read for a
// possible reader of the copy's destination and drains all copies in flight (s_waitcnt vmcnt(0)) in front of it; the
// copies are ordered by the pipeline's own counted waits and barriers.  It has no register outputs.
typedef uint32_t rsrc4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ rsrc4_t make_rsrc4(const void* base, uint32_t bytes)
{
    const uint64_t a = (uint64_t)base;
    rsrc4_t r = {(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, bytes, 0x00020000u};
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)r[i]);
    return r;
}
__device__ __forceinline__ void dma16(const rsrc4_t& r, uint32_t lds, uint32_t off)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :
                 : "s"(lds), "v"(off), "s"(r)
                 : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_addr(const void* p)
{
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

struct PipeArgs {
    rsrc4_t a, b;       // A: [rows][lda] bytes; B: [columns][ldb] bytes, or (BTR) [K][ldb]; ranges end with the operand
    uint32_t lda, ldb;
    uint32_t a0, b0;    // byte offsets of the tile origin
    int32_t kbytes;     // K
    // MX: the stage-major scales ([stage][rows][8]) of both operands through one resource: byte offsets of the tile's
    // first row in stage 0, and the stage strides
    rsrc4_t aux;
    uint32_t sa_off, sa_stride, sb_off, sb_stride;
    // OP_AQ: the packed weight (kbytes / 256 tiles per 16-column strip), the group rows of scale and offset [K / g][n],
    // g = 64 << gshift, and the tile's first column
    const uint8_t* wp;
    const uint16_t *scale, *offset;
    uint32_t w_bytes, s_bytes, n, n0, gshift;
};

// B operand of the weight-only antiquant pipeline; FMT bit 0: int4 codes (else int8), bit 1: with offsets
constexpr int OP_AQ = 16;

template <int BM, int BN, int WM, int WN, int OP, int FMT = 0, bool BTR = false>
struct GemmPipe {
    static constexpr int ST = 2;  // stages of the ring
    static constexpr bool IS_F8 = OP == OP_F8;
    static constexpr bool IS_MX = OP == OP_MXFP4;
    static constexpr bool IS_AQ = OP == OP_AQ;
    static_assert(OP == OP_I8 || OP == OP_F8 || ((IS_MX || IS_AQ) && !BTR),
                  "int8, fp8, MX-FP4 with a K-contiguous B, or f16 with a packed weight");
    static constexpr int CBSZ = IS_MX ? F8F6F4_E2M1 : FMT & 7;  // f8f6f4 formats of A and B
    static constexpr int BLGP = IS_MX ? F8F6F4_E2M1 : (FMT >> 3) & 7;
    static constexpr int TBM = BM, TBN = BN, TWN = WN;
    static constexpr int ROWB = 128;
    static constexpr int KPS = IS_F8 ? 1 : 2;        // k-steps per stage
    static constexpr int AR = 4;                     // registers of an accumulator fragment
    static constexpr int NW = WM * WN, NT = NW * 64;
    // rows of half h (192 rows: 128 and 64), of a wave in it, and their 16-row fragments
    static constexpr int hm(int h) { return BM % 128 == 0 || BM == 64 ? BM / 2 : (h ? BM / 3 : BM / 3 * 2); }
    static constexpr int hn(int h) { return BN % 128 == 0 || BN == 64 ? BN / 2 : (h ? BN / 3 : BN / 3 * 2); }
    static constexpr int whm(int h) { return hm(h) / WM; }
    static constexpr int whn(int h) { return hn(h) / WN; }
    static constexpr int fmh(int h) { return whm(h) / 16; }
    static constexpr int fnh(int h) { return whn(h) / 16; }
    static constexpr int FM = fmh(0) + fmh(1), FN = fnh(0) + fnh(1);
    static constexpr int ca(int h) { return hm(h) / 8 / NW; }  // 1 KiB copies per wave of an A / B half
    static constexpr int cb(int h) { return hn(h) / 8 / NW; }
    static constexpr int A_REG = ST * BM * ROWB, B_REG = (IS_AQ ? 1 : ST) * BN * ROWB;
    static_assert(!IS_AQ || (cb(0) <= 2 && cb(1) <= 2), "a wave dequantises columns of one strip per half");
    static constexpr int SCA = IS_MX ? (BM * 8 + 1023) / 1024 : 0, SCB = IS_MX ? (BN * 8 + 1023) / 1024 : 0;  // scale copies
    static constexpr int SC_SLOT = (SCA + SCB) * 1024;
    static constexpr size_t LDS_BYTES = (size_t)A_REG + B_REG + 4 * SC_SLOT;
    typedef typename std::conditional<OP == OP_I8, v4i, v4f>::type acc_t;
    typedef typename std::conditional<IS_F8, v8i, v4i>::type frag_t;
    static_assert(whm(0) % 16 == 0 && whm(1) % 16 == 0 && whn(0) % 32 == 0 && whn(1) % 32 == 0, "wave quadrants");
    static_assert(hm(0) % (8 * NW) == 0 && hm(1) % (8 * NW) == 0 && hn(0) % (8 * NW) == 0 && hn(1) % (8 * NW) == 0,
                  "copies split evenly over the waves");
    static_assert(NW == 4 || NW == 8, "the swizzles of a lane's copies agree");
    static_assert(A_REG <= 65536 && B_REG <= 65536, "LDS read offsets are 16 bits");
    static_assert(LDS_BYTES <= 160 * 1024, "LDS");
    static_assert(SCA + SCB <= NW, "one scale copy per wave");
    static_assert(!BTR || ((hn(0) == 128 || hn(0) == 64) && (hn(1) == 128 || hn(1) == 64)), "[K, N] halves");

    // copies of half H(i)
    static constexpr int half_copies(int i) { return i % 4 == 0 ? ca(0) : i % 4 == 1 ? cb(0) : i % 4 == 2 ? cb(1) : ca(1); }
    // OP_AQ: loads of a weight half into registers
    static constexpr int WLOADS = FMT & 2 ? 3 : 2;
    // copies a wave may have outstanding at the barrier in front of phase p: H(t + 3) .. H(t + 4 ST).  OP_AQ: phase 1 loads
    // B0 three stages ahead, phase 2 requests A1 two ahead, phase 3 loads B1 and requests A0 three ahead; phase 1 reads
    // A1 (after its copies came B1, A0, B0, A1, B1, A0), phase 2 A0 (B0, A1, B1, A0, B0), phases 0 and 3 what ds_writes
    // put there
    static constexpr int outstanding(int p)
    {
        if (IS_AQ) return p == 1 ? 2 * ca(0) + ca(1) + 3 * WLOADS : p == 2 ? ca(0) + ca(1) + 3 * WLOADS : 63;
        int n = 0;
        for (int i = p + 3; i <= p + 4 * ST; ++i) n += half_copies(i);
        if (IS_MX)  // ... and the scale copies of the phases 2 among the 4 ST - 2 before
            for (int t = p + 2; t < p + 4 * ST; ++t) n += t % 4 == 2;
        return n;
    }
    static constexpr int RING = ST * (ca(0) + ca(1) + cb(0) + cb(1));  // copies of the whole ring
    static_assert(RING < 64, "vmcnt");

    // the tile row of fragment row i, and the first of the four columns of fragment column j
    __device__ __forceinline__ static int block_row(int wm, int i)
    {
        return i < fmh(0) ? wm * whm(0) + i * 16 : hm(0) + wm * whm(1) + (i - fmh(0)) * 16;
    }
    __device__ __forceinline__ static int block_col(int wn, int j)
    {
        return j < fnh(0) ? wn * whn(0) + j * 16 : hn(0) + wn * whn(1) + (j - fnh(0)) * 16;
    }
    __device__ __forceinline__ static int ct_row(int wm, int i, int lane) { return block_row(wm, i) + (lane & 15); }
    __device__ __forceinline__ static int ct_col(int wn, int j, int lane) { return block_col(wn, j) + 4 * (lane >> 4); }
    __device__ __forceinline__ static int el_row(int wm, int i, int, int lane) { return ct_row(wm, i, lane); }
    __device__ __forceinline__ static int el_col(int wn, int j, int r, int lane) { return ct_col(wn, j, lane) + r; }

    // BTR: chunks per K row of half h, and the chunk swizzle of K row k in it
    static constexpr int tch(int h) { return hn(h) / 16; }
    __device__ __forceinline__ static int swz_tr(int h, int k)
    {
        return tch(h) == 8 ? ((k >> 1) & 3) | (((k >> 4) & 1) << 2) : ((k >> 2) & 1) | (((k >> 4) & 1) << 1);
    }

    // s_waitcnt vmcnt(N) lgkmcnt(0)
    template <int N>
    __device__ __forceinline__ static void wait_half()
    {
        __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
    }

    __device__ __forceinline__ static void run(const PipeArgs& p, uint8_t* smem, acc_t (&acc)[FM][FN])
    {
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        const int t = (int)threadIdx.x, lane = t & 63;
        const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
        const int wm = wave / WN, wn = wave % WN;
        const int r16 = lane & 15, g = lane >> 4;
        uint8_t* sA = smem;
        uint8_t* sB = smem + A_REG;
        const uint32_t lA = lds_addr(sA), lB = lds_addr(sB);

        // copy u of this wave in a half covers 1 KiB of it at u * NW + wave; the chunk swizzles repeat from copy to copy,
        // so one lane offset per operand (BTR: per half of B) serves them all
        const int nk = (p.kbytes + ROWB - 1) / ROWB;
        const int kchunk = (int)((lane & 7) ^ ((wave * 4 + (lane >> 4)) & 7)) * 16;
        const uint32_t va = p.a0 + (uint32_t)(lane >> 3) * p.lda + (uint32_t)kchunk;
        uint32_t vb[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (BTR) {
                const int kr = lane / tch(h), k = wave * (64 / tch(h)) + kr;
                vb[h] = p.b0 + (uint32_t)kr * p.ldb + (uint32_t)((lane % tch(h)) ^ swz_tr(h, k)) * 16u;
            } else {
                vb[h] = p.b0 + (uint32_t)(lane >> 3) * p.ldb + (uint32_t)kchunk;
            }
        }
        // half HI (0: A0, 1: B0, 2: B1, 3: A1) of stage kt into `slot`; nothing is read past K.  (Rows past the operand's
        // last lie past its resource's range; rows past the tile's own are read, their products dropped.)
        auto request = [&](auto HI, int kt, int slot) {
            constexpr int hi = decltype(HI)::value;
            constexpr bool isa = hi == 0 || hi == 3;
            constexpr int h = hi >= 2 ? 1 : 0;
            const uint32_t dst = isa ? lA + slot * (BM * ROWB) + h * hm(0) * ROWB : lB + slot * (BN * ROWB) + h * hn(0) * ROWB;
            uint32_t v = isa ? va : vb[h], s = (uint32_t)kt * ROWB;
            if constexpr (BTR && !isa) s = kt < nk ? s * p.ldb : OOB;
            else if constexpr (IS_AQ) s = kt < nk ? s : OOB;  // (whole stages)
            else v += kt * ROWB + kchunk < p.kbytes ? 0u : OOB;
#pragma unroll
            for (int u = 0; u < (isa ? ca(h) : cb(h)); ++u) {
                const int c = u * NW + wave;
                uint32_t row;
                if constexpr (isa) row = (uint32_t)(h * hm(0) + c * 8) * p.lda;
                else if constexpr (BTR) row = (uint32_t)(c * (64 / tch(h))) * p.ldb + (uint32_t)(h * hn(0));
                else row = (uint32_t)(h * hn(0) + c * 8) * p.ldb;
                dma16(isa ? p.a : p.b, dst + c * 1024, v + (s + row));
            }
        };

        // MX: this wave's 1 KiB of a stage's scales (waves past the copies repeat one)
        const uint8_t* sS = smem + A_REG + B_REG;
        uint32_t sc_off = 0, sc_stride = 0, sc_dst = 0;
        if constexpr (IS_MX) {
            const int c = wave % (SCA + SCB);
            const bool isb = c >= SCA;
            sc_off = (isb ? p.sb_off + (uint32_t)(c - SCA) * 1024u : p.sa_off + (uint32_t)c * 1024u) + (uint32_t)lane * 16u;
            sc_stride = isb ? p.sb_stride : p.sa_stride;
            sc_dst = lds_addr(sS) + (uint32_t)c * 1024u;
        }
        auto request_scales = [&](int kt) {
            if constexpr (IS_MX)
                dma16(p.aux, sc_dst + (uint32_t)(kt & 3) * SC_SLOT, sc_off + (kt < nk ? (uint32_t)kt * sc_stride : OOB));
        };

        // OP_AQ: this wave's strip of half h and the lane's offsets into the packed weight and the group rows
        struct WeightRegs {
            uint32_t w[2][2];  // [fragment][code words]
            uint32_t sc, of;
        };
        constexpr bool I4 = FMT & 1, HAS_OFF = (FMT & 2) != 0;
        constexpr int CW = I4 ? 1 : 2;  // code words per fragment
        [[maybe_unused]] WeightRegs wr[2][2];  // [stage parity][half]
        uint32_t w_at[2] = {}, s_at[2] = {}, magic = 0;
        const rsrc_t r_w = make_rsrc(p.wp, p.w_bytes), r_s = make_rsrc(p.scale, p.s_bytes),
                     r_o = make_rsrc(HAS_OFF ? p.offset : p.scale, p.s_bytes);
        if constexpr (IS_AQ) {
            magic = half_magic_vgpr();
#pragma unroll
            for (int h = 0; h < 2; ++h) {  // two fragments of a stage (32 k each) per wave, or one
                const uint32_t col = p.n0 + (uint32_t)(h * hn(0)) + (cb(h) == 2 ? wave : wave >> 1) * 16u;
                const bool ok = col < p.n;
                w_at[h] = ok ? col / 16u * (uint32_t)(p.kbytes / 256) * (CW * 1024u) + lane * (CW * 16u) +
                                   (cb(h) == 2 ? 0 : wave & 1) * (CW * 4u)
                             : OOB;
                s_at[h] = ok ? (col + r16) * 2u : OOB;
            }
        }
        auto load_w = [&](auto HH, auto PAR, int kt) {
            constexpr int h = decltype(HH)::value, par = decltype(PAR)::value & 1;
            WeightRegs& r = wr[par][h];
            const uint32_t k = (uint32_t)(kt < nk ? kt : nk - 1);  // (stages past the last: read, never multiplied)
            const uint32_t off = w_at[h] + par * (CW * 8u);
            const int soff = (int)((k >> 1) * (CW * 1024u));
            if constexpr (cb(h) * CW == 4) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r_w, off, soff, 0);
                r.w[0][0] = v[0], r.w[0][1] = v[1], r.w[1][0] = v[2], r.w[1][1] = v[3];
            } else if constexpr (cb(h) * CW == 2) {
                const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r_w, off, soff, 0);
                r.w[0][0] = v[0];
                r.w[I4 ? 1 : 0][I4 ? 0 : 1] = v[1];
            } else {
                r.w[0][0] = __builtin_amdgcn_raw_buffer_load_b32(r_w, off, soff, 0);
            }
            const int grow = (int)((k >> p.gshift) * p.n * 2u);
            r.sc = __builtin_amdgcn_raw_buffer_load_b16(r_s, s_at[h], grow, 0);
            if constexpr (HAS_OFF) r.of = __builtin_amdgcn_raw_buffer_load_b16(r_o, s_at[h], grow, 0);
        };

        // lane offsets of the fragment reads: 16-byte chunk 4 c + g of the lane's row (within a half, wave row 0); BTR: the
        // lane's 8-byte piece of fragment column j
        constexpr int FA = fmh(0) > fmh(1) ? fmh(0) : fmh(1), FB = fnh(0) > fnh(1) ? fnh(0) : fnh(1);
        uint32_t rl[2], rt[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) rl[c] = (uint32_t)(r16 * ROWB + (((4 * c + g) ^ ((r16 >> 1) & 7)) * 16));
        if constexpr (BTR) {
            const int k = 16 * g + (r16 >> 1);
#pragma unroll
            for (int h = 0; h < 2; ++h)  // of fragment column 0; column j's chunk differs by an XOR (fnh is a power of two)
                rt[h] = (uint32_t)(k * hn(h) + ((wn * fnh(h)) ^ swz_tr(h, k)) * 16 + (r16 & 1) * 8);
        }
        // fragment u of the weights held for half h, dequantised; its place: column l % 16 of the strip, chunk 4 jj + l / 16
        // (the layout of the reads)
        [[maybe_unused]] h8 wfrag;
        auto dequant_w = [&](auto HH, auto PAR, int u) {
            constexpr int h = decltype(HH)::value, par = decltype(PAR)::value & 1;
            if (u >= cb(h)) return;
            const WeightRegs& r = wr[par][h];
            const _Float16 sv = __builtin_bit_cast(_Float16, (uint16_t)r.sc);
            const _Float16 ov = HAS_OFF ? __builtin_bit_cast(_Float16, (uint16_t)r.of) : (_Float16)0.0f;
            wfrag = dequant8<I4, HAS_OFF>(r.w[u][0], I4 ? 0u : r.w[u][1], (h2){ov, ov}, (h2){sv, sv}, magic);
        };
        auto store_w = [&](auto HH, int u) {
            constexpr int h = decltype(HH)::value;
            if (u >= cb(h)) return;
            const int strip = cb(h) == 2 ? wave : wave >> 1;
            const uint32_t o = cb(h) == 2 ? rl[u] : rl[0] ^ ((wave & 1) * 64u);
            *(h8*)(sB + (h * hn(0) + strip * 16) * ROWB + o) = wfrag;
        };
        const uint32_t wa[2] = {(uint32_t)(wm * whm(0) * ROWB), (uint32_t)((hm(0) + wm * whm(1)) * ROWB)};
        const uint32_t wb[2] = {(uint32_t)(wn * whn(0) * ROWB), (uint32_t)((hn(0) + wn * whn(1)) * ROWB)};
        frag_t fa[2][FA][KPS], fb[2][FB][KPS];
        auto read_frag = [&](const uint8_t* base, const uint32_t (&off)[2], int s) -> frag_t {
            if constexpr (IS_F8) {
                const v4i x = *(const v4i*)(base + off[0]);
                const v4i y = *(const v4i*)(base + off[1]);
                return (v8i){x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
            } else {
                return *(const v4i*)(base + off[s]);
            }
        };
        // the lane offsets of a read, added up in front of it: kept over the loop for every half they cost more
        // registers than the 256 x 256 tiles have
        auto at = [&](uint32_t (&off)[2], uint32_t w) {
            asm volatile("" : "+s"(w));
            off[0] = rl[0] + w;
            off[1] = rl[1] + w;
        };
        // MX: the scale bytes of fragment rows i and i + 1 (k-steps 0 and 1 each) in one register
        us2_t swa[2][(FA + 1) / 2], swb[2][(FB + 1) / 2];
        const uint32_t rs = (uint32_t)(r16 * 8 + 2 * g);
        auto read_scale = [&](int kt, int row) -> uint16_t {
            return *(const uint16_t*)(sS + (kt & 3) * SC_SLOT + row * 8 + rs);
        };
        auto read_a = [&](auto HH, int slot, int kt) {
            constexpr int h = decltype(HH)::value;
            uint32_t off[2];
            at(off, wa[h]);
            if constexpr (IS_MX) {
#pragma unroll
                for (int i = 0; i < fmh(h); ++i) swa[h][i / 2][i % 2] = read_scale(kt, h * hm(0) + wm * whm(h) + i * 16);
            }
#pragma unroll
            for (int i = 0; i < fmh(h); ++i)
#pragma unroll
                for (int s = 0; s < KPS; ++s) fa[h][i][s] = read_frag(sA + slot * (BM * ROWB) + i * 16 * ROWB, off, s);
        };
        typedef int v2i_t __attribute__((ext_vector_type(2)));
        auto read_tr = [&](const uint8_t* base, int h, uint32_t off, int s) -> v4i {  // K rows 64 s + 16 g .. + 15
            typedef __attribute__((address_space(3))) v2i_t* lp;
            const v2i_t x = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lp)(base + off + s * 64 * hn(h)));
            const v2i_t y = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lp)(base + off + (s * 64 + 8) * hn(h)));
            return (v4i){x[0], x[1], y[0], y[1]};
        };
        auto read_b = [&](auto HH, int set, int slot, int kt) {
            constexpr int h = decltype(HH)::value;
            uint32_t off[2];
            if constexpr (!BTR) at(off, A_REG + wb[h]);
            if constexpr (IS_MX) {
#pragma unroll
                for (int j = 0; j < fnh(h); ++j)
                    swb[set][j / 2][j % 2] = read_scale(kt, SCA * 128 + h * hn(0) + wn * whn(h) + j * 16);
            }
#pragma unroll
            for (int j = 0; j < fnh(h); ++j) {
                uint32_t tr = 0;
                if constexpr (BTR) {
                    uint32_t x = (uint32_t)j * 16u;
                    asm volatile("" : "+s"(x));  // (as in `at`)
                    tr = (rt[h] ^ x) + A_REG;
                }
#pragma unroll
                for (int s = 0; s < KPS; ++s) {
                    if constexpr (BTR) {
                        const uint8_t* base = sA + slot * (BN * ROWB) + h * hn(0) * ROWB;
                        if constexpr (IS_F8) {
                            const v4i x = read_tr(base, h, tr, 0), y = read_tr(base, h, tr, 1);
                            fb[set][j][s] = (v8i){x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
                        } else {
                            fb[set][j][s] = read_tr(base, h, tr, s);
                        }
                    } else {
                        fb[set][j][s] = read_frag(sA + slot * (BN * ROWB) + j * 16 * ROWB, off, s);
                    }
                }
            }
        };
        // MFMAs x0 .. x1 - 1 (k-step, then B fragment, then A fragment) of the quadrant (A half HA, B half HB held in
        // register set `set`)
        auto multiply = [&](auto HA, auto HB, int set, int x0, int x1) {
            constexpr int ha = decltype(HA)::value, hb = decltype(HB)::value, fm = fmh(ha), fn = fnh(hb);
#pragma unroll
            for (int x = 0; x < KPS * fn * fm; ++x) {
                if (x < x0 || x >= x1) continue;
                const int s = x / (fn * fm), j = x / fm % fn, i = x % fm;
                acc_t& c = acc[ha * fmh(0) + i][hb * fnh(0) + j];
                if constexpr (IS_AQ)
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, fb[set][j][s]),
                                                               __builtin_bit_cast(h8, fa[ha][i][s]), c, 0, 0, 0);
                else if constexpr (OP == OP_I8)
                    c = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[set][j][s], fa[ha][i][s], c, 0, 0, 0);
                else if constexpr (OP == OP_F8)
                    c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[set][j][s], fa[ha][i][s], c, BLGP, CBSZ, 0, 0, 0,
                                                                         0);
                else {
                    const v4i u = fb[set][j][s], v = fa[ha][i][s];
                    const v8i b8 = (v8i){u[0], u[1], u[2], u[3], 0, 0, 0, 0}, a8 = (v8i){v[0], v[1], v[2], v[3], 0, 0, 0, 0};
                    const int sb = __builtin_bit_cast(int, swb[set][j / 2]), sa = __builtin_bit_cast(int, swa[ha][i / 2]);
                    // (the byte of an operand's scale register: 2 (fragment % 2) + s; an immediate of the instruction)
                    auto f = [&](auto SB, auto SA) {
                        c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b8, a8, c, BLGP, CBSZ, decltype(SB)::value, sb,
                                                                             decltype(SA)::value, sa);
                    };
                    if (s == 0) {
                        if (j % 2 == 0 && i % 2 == 0) f(I0{}, I0{});
                        if (j % 2 == 0 && i % 2 == 1) f(I0{}, I2{});
                        if (j % 2 == 1 && i % 2 == 0) f(I2{}, I0{});
                        if (j % 2 == 1 && i % 2 == 1) f(I2{}, I2{});
                    } else {
                        if (j % 2 == 0 && i % 2 == 0) f(I1{}, I1{});
                        if (j % 2 == 0 && i % 2 == 1) f(I1{}, I3{});
                        if (j % 2 == 1 && i % 2 == 0) f(I3{}, I1{});
                        if (j % 2 == 1 && i % 2 == 1) f(I3{}, I3{});
                    }
                }
            }
        };

#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = (acc_t){};

        // prologue: the ring's halves in flight, H(0) and H(1) into registers, then H(4 ST) into the slot of H(0)
        // (scales where the loop's phases 2 would have requested them, so that `outstanding` holds from phase 0 on)
        if constexpr (IS_AQ) {  // in the loop's order, so that `outstanding` holds from phase 1 on
            load_w(I0{}, I0{}, 0);
            load_w(I1{}, I0{}, 0);
            load_w(I0{}, I1{}, 1);
            __builtin_amdgcn_sched_barrier(0);
            request(I0{}, 0, 0);
            request(I3{}, 0, 0);
            load_w(I1{}, I1{}, 1);
            __builtin_amdgcn_sched_barrier(0);
            request(I0{}, 1, 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                dequant_w(I0{}, I0{}, u);
                store_w(I0{}, u);
                dequant_w(I1{}, I0{}, u);
                store_w(I1{}, u);
            }
            __builtin_amdgcn_sched_barrier(0);
            load_w(I0{}, I0{}, 2);
            __builtin_amdgcn_sched_barrier(0);
            request(I3{}, 1, 1);
            load_w(I1{}, I0{}, 2);
            dequant_w(I0{}, I1{}, 0);
            __builtin_amdgcn_sched_barrier(0);
            wait_half<ca(0) + 2 * ca(1)>();
            stage_barrier();
            read_a(I0{}, 0, 0);
            read_b(I0{}, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            wait_half<63>();
            stage_barrier();
            request(I0{}, ST, 0);
            __builtin_amdgcn_sched_barrier(0);
        } else {
        request_scales(0);
#pragma unroll
        for (int k = 0; k < ST; ++k) {
            request(I0{}, k, k);
            request(I1{}, k, k);
            request(I2{}, k, k);
            if (k >= ST - 2) request_scales(k - ST + 3);
            request(I3{}, k, k);
        }
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<RING - ca(0) - cb(0)>();
        stage_barrier();
        read_a(I0{}, 0, 0);
        read_b(I0{}, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        wait_half<RING - ca(0) - cb(0)>();
        stage_barrier();
        request(I0{}, ST, 0);
        __builtin_amdgcn_sched_barrier(0);
        }

        // phase P of stage kt, which lies in slot SL of the ring (kt = SL modulo ST)
        auto phase = [&](auto PP, auto SS, int kt) {
            constexpr int P = decltype(PP)::value, SL = decltype(SS)::value, SN = (SL + 1) % ST;
            constexpr int set0 = SL & 1, set1 = 1 - set0;  // register sets of B0(kt), B1(kt)
            using HA = std::integral_constant<int, P >= 2>;
            using HB = std::integral_constant<int, P == 1 || P == 2>;
            constexpr int set = HB::value ? set1 : set0;
            constexpr int NX = KPS * fnh(HB::value) * fmh(HA::value);
            constexpr int LEAD = NX >= 8 ? NX / 4 : 1;  // MFMAs issued ahead of the reads
            __builtin_amdgcn_sched_barrier(0);
            wait_half<outstanding(P)>();
            stage_barrier();
            if constexpr (IS_AQ) {
                store_w(std::integral_constant<int, (P >= 2)>{}, P & 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            multiply(HA{}, HB{}, set, 0, LEAD);
            __builtin_amdgcn_sched_barrier(0);
            constexpr int SB = IS_AQ ? 0 : SL, SBN = IS_AQ ? 0 : SN;  // B's slots
            if constexpr (P == 0) read_b(I1{}, set1, SB, kt);
            if constexpr (P == 1) read_a(I1{}, SL, kt);
            if constexpr (P == 2) read_a(I0{}, SN, kt + 1);
            if constexpr (P == 3) read_b(I0{}, set1, SBN, kt + 1);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (IS_AQ) {
                if constexpr (P == 1) load_w(I0{}, std::integral_constant<int, SN>{}, kt + 3);
                if constexpr (P == 3) load_w(I1{}, std::integral_constant<int, SN>{}, kt + 3);
                __builtin_amdgcn_sched_barrier(0);
            } else {
                if constexpr (P == 0) request(I1{}, kt + ST, SL);
                if constexpr (P == 1) request(I2{}, kt + ST, SL);
            }
            if constexpr (P == 2) {
                request_scales(kt + 3);
                request(I3{}, kt + ST, SL);
            }
            if constexpr (P == 3) request(I0{}, kt + 1 + ST, SN);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (IS_AQ)  // (phase 3: of the stage after)
                dequant_w(std::integral_constant<int, (P == 1 || P == 2)>{}, std::integral_constant<int, P == 3 ? SL : SN>{},
                          P == 0 || P == 2);
            multiply(HA{}, HB{}, set, LEAD, NX);
        };
        auto stage = [&](auto SS, int kt) {
            phase(I0{}, SS, kt);
            phase(I1{}, SS, kt);
            phase(I2{}, SS, kt);
            phase(I3{}, SS, kt);
        };
        int kt = 0;
        for (; kt + ST <= nk; kt += ST) {
            stage(I0{}, kt);
            stage(I1{}, kt + 1);
        }
        if (kt < nk) stage(I0{}, kt);
        // drain: no copy may still target LDS when the caller reuses it or the wave ends
        wait_vmcnt<0>();
    }
};

// The tile of a problem: the one whose rounds over the 256 CUs cost least.  Measured per tile shape (int8, DEQF16 out,
// K = 4096, one MI355X): microseconds per 128-byte stage of K with few CUs at work (`solo`) and with all of them
// (`full`: the matrix cores and the memory system then share a power and a bandwidth limit), and what a tile costs
// beyond its stages when all write at once (`tail`: first stage's latency, epilogue).  A CU runs c = ceil(tiles / 256)
// tiles, one after the other or side by side (128 x 128 two at a time, 64 x 128 three: no gain per tile, so the same
// sum), a fraction of the CUs one fewer.  E.g. K = 4096, N = 11008 (start: this layout's tiles before these kernels):
// M = 2048 256 x 192 in 78 us against 91 (256 x 256), 84 (128 x 256), 88 (128 x 128); M = 512 128 x 192 in 25.0 against
// 25.6 (128 x 256), 27.8 (128 x 128), 30.2 (64 x 128); M = 256 128 x 128 in 16.6 against 20.3 (128 x 192), 20.6
// (64 x 128); M = 128 64 x 128 in 12.5 against 16.0 (128 x 128).  The tails of the three largest shapes are alike per
// element: at short K the stores of all rounds are what a call takes (M = 4096, N = 11008, K = 256: 256 x 256 in 31 us,
// 192 x 256 33).
enum PipeTile { PIPE_256x256, PIPE_192x256, PIPE_256x192, PIPE_128x256, PIPE_128x192, PIPE_128x128, PIPE_64x128, PIPE_TILES };
// groups: of a group matmul, whose M rows fall into groups of sizes the host does not know: half a row tile more each.
inline PipeTile pick_pipe_tile(int64_t M, int64_t N, int64_t kbytes, int64_t groups = 0)
{
    static const struct {
        int bm, bn;
        float solo, full, tail;
    } T[PIPE_TILES] = {{256, 256, 1.08f, 1.45f, 6.0f}, {192, 256, 0.86f, 1.16f, 4.5f}, {256, 192, 0.86f, 1.16f, 4.5f},
                       {128, 256, 0.59f, 0.90f, 4.0f}, {128, 192, 0.50f, 0.67f, 3.5f}, {128, 128, 0.375f, 0.47f, 1.9f},
                       {64, 128, 0.25f, 0.30f, 0.65f}};
    const float stages = (float)((kbytes + 127) / 128);
    PipeTile best = PIPE_256x256;
    float least = 0.0f;
    for (int t = 0; t < PIPE_TILES; ++t) {
        const int64_t tiles = ((M + T[t].bm - 1) / T[t].bm + groups / 2) * ((N + T[t].bn - 1) / T[t].bn);
        const float c = (float)((tiles + 255) / 256), fill = (float)tiles / (256.0f * c);
        const float cost = c * ((T[t].solo + (T[t].full - T[t].solo) * fill) * stages + T[t].tail * fill);
        if (t == 0 || cost < least) {
            best = (PipeTile)t;
            least = cost;
        }
    }
    return best;
}

// XCD-aware tile order of the pipelined kernels: consecutive workgroup ids go round-robin over the 8 XCDs, so XCD x
// gets the x-th of 8 contiguous runs (equal within one tile) of a raster that walks GM tile rows at a time: the tiles
// that one XCD runs together share A rows and B columns through its L2.
__device__ __forceinline__ void pipe_tile(int pid, int tiles_m, int tiles_n, int& tm, int& tn)
{
    const int total = tiles_m * tiles_n, q = total / 8, r = total % 8, x = pid % 8;
    pid = x * q + (x < r ? x : r) + pid / 8;
    constexpr int GM = 8;
    const int width = GM * tiles_n;
    const int first_m = (pid / width) * GM;
    const int gm = (tiles_m - first_m) < GM ? (tiles_m - first_m) : GM;
    const int in_group = pid % width;
    tm = first_m + in_group % gm;
    tn = in_group / gm;
}

// Store epilogue of transposed accumulators.  Lane l = 16 g + r holds columns 4 g .. 4 g + 3 of row r of each 16 x 16
// fragment.  v_permlane16_swap trades the odd lane rows of fragment j's registers for the even ones of fragment
// j + 1's, after which a lane owns eight consecutive columns -- 8 (g / 2) .. of fragment j + g % 2: one 16-byte
// (2-byte elements), 8-byte (1-byte) or 4-byte (int4 codes, ES 0) store where there were eight of one element.  4-byte
// elements leave as they are, one 16-byte store per fragment.
// cols4(tile column) gives the parameters of four columns; conv(accumulator, parameters, e[, tile row]) the element's
// bits, or, for the 2-byte types (OUT_F16, OUT_BF16), its fp32 value, which is converted here two at a time.
// vec: the output's base and row pitch are multiples of four bytes; otherwise, and in runs that cross the tile's last
// column, elements are stored one by one.
enum { OUT_I4 = 0, OUT_1 = 1, OUT_F16 = 2, OUT_BF16 = 3, OUT_4 = 4 };
template <class T, int OUT, class Cols, class Conv>
__device__ __forceinline__ void ct_store(const TileOut& out, bool vec, int cols, const typename T::acc_t (&acc)[T::FM][T::FN],
                                         int wm, int wn, int lane, Cols cols4, Conv conv)
{
    constexpr bool HALF = OUT == OUT_F16 || OUT == OUT_BF16;
    auto call = [&](auto a, const auto& par, int e, int row) {
        if constexpr (std::is_invocable_v<Conv, decltype(a), decltype(par), int, int>) return conv(a, par, e, row);
        else return conv(a, par, e);
    };
    const int g = lane >> 4;
#pragma unroll
    for (int j = 0; j < T::FN; j += 2) {
        const int c0 = T::ct_col(wn, j, lane), c1 = c0 + 16;
        const auto p0 = cols4(c0), p1 = cols4(c1);
#pragma unroll
        for (int i = 0; i < T::FM; ++i) {
            const int row = T::ct_row(wm, i, lane);
            const uint32_t roff = (uint32_t)row * out.pitch;
            const int c = T::block_col(wn, j + (g & 1)) + 8 * (g >> 1);  // this lane's eight columns after the swap
            if constexpr (OUT == OUT_4) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    uint32_t x[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[e] = call(acc[i][j + q][e], q ? p1 : p0, e, row);
                    const int cq = q ? c1 : c0;
                    if (cq + 4 <= cols) {
                        __builtin_amdgcn_raw_buffer_store_b128((u32x4){x[0], x[1], x[2], x[3]}, out.r,
                                                               roff + (uint32_t)cq * 4, 0, 0);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            __builtin_amdgcn_raw_buffer_store_b32(x[e], out.r,
                                                                  cq + e < cols ? roff + (uint32_t)(cq + e) * 4 : OOB, 0, 0);
                    }
                }
            } else {
                constexpr int PER = HALF ? 2 : (OUT == OUT_1 ? 4 : 8);  // elements per dword
                constexpr int SH = 32 / PER;                            // bits per element
                uint32_t lo[2], hi[2], d[8 / PER];                      // fragment j's four elements, j + 1's
                if constexpr (HALF) {
                    float v[8];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e] = call(acc[i][j][e], p0, e, row);
                        v[4 + e] = call(acc[i][j + 1][e], p1, e, row);
                    }
                    us2_t top = {0, 0};
                    lo[0] = cvt_pair<OUT == OUT_BF16>(v[0], v[1], top);
                    lo[1] = cvt_pair<OUT == OUT_BF16>(v[2], v[3], top);
                    hi[0] = cvt_pair<OUT == OUT_BF16>(v[4], v[5], top);
                    hi[1] = cvt_pair<OUT == OUT_BF16>(v[6], v[7], top);
                    if (__builtin_expect(cvt_special<OUT == OUT_BF16>(top), 0)) {
                        auto one = [](float x) { return (uint32_t)(OUT == OUT_BF16 ? f32_to_bf16_sat(x) : f32_to_f16_sat(x)); };
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            lo[e] = one(v[2 * e]) | (one(v[2 * e + 1]) << 16);
                            hi[e] = one(v[4 + 2 * e]) | (one(v[4 + 2 * e + 1]) << 16);
                        }
                    }
                    const auto s0 = __builtin_amdgcn_permlane16_swap(lo[0], hi[0], false, false);
                    const auto s1 = __builtin_amdgcn_permlane16_swap(lo[1], hi[1], false, false);
                    d[0] = s0[0];
                    d[1] = s1[0];
                    d[2] = s0[1];
                    d[3] = s1[1];
                } else {
                    constexpr uint32_t MASK = (1u << SH) - 1u;
                    lo[0] = hi[0] = 0u;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        lo[0] |= (call(acc[i][j][e], p0, e, row) & MASK) << (SH * e);
                        hi[0] |= (call(acc[i][j + 1][e], p1, e, row) & MASK) << (SH * e);
                    }
                    const auto sw = __builtin_amdgcn_permlane16_swap(lo[0], hi[0], false, false);
                    if constexpr (OUT == OUT_I4) {
                        d[0] = sw[0] | (sw[1] << 16);
                    } else {
                        d[0] = sw[0];
                        d[1] = sw[1];
                    }
                }
                if (vec && c + 8 <= cols) {
                    if constexpr (OUT == OUT_I4)
                        __builtin_amdgcn_raw_buffer_store_b32(d[0], out.r, roff + (uint32_t)(c / 2), 0, 0);
                    else if constexpr (OUT == OUT_1)
                        __builtin_amdgcn_raw_buffer_store_b64((u32x2){d[0], d[1]}, out.r, roff + (uint32_t)c, 0, 0);
                    else
                        __builtin_amdgcn_raw_buffer_store_b128((u32x4){d[0], d[1], d[2], d[3]}, out.r,
                                                               roff + (uint32_t)c * 2, 0, 0);
                } else if constexpr (OUT == OUT_I4) {  // two codes per byte (an even number of columns)
#pragma unroll
                    for (int e = 0; e < 8; e += 2)
                        __builtin_amdgcn_raw_buffer_store_b8((uint8_t)(d[0] >> (4 * e)), out.r,
                                                             c + e < cols ? roff + (uint32_t)((c + e) / 2) : OOB, 0, 0);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const uint32_t v = d[e / PER] >> (SH * (e % PER));
                        const uint32_t o = c + e < cols ? roff + (uint32_t)((c + e) * (HALF ? 2 : 1)) : OOB;
                        if constexpr (HALF) __builtin_amdgcn_raw_buffer_store_b16((uint16_t)v, out.r, o, 0, 0);
                        else __builtin_amdgcn_raw_buffer_store_b8((uint8_t)v, out.r, o, 0, 0);
                    }
                }
            }
        }
    }
}

// The per-channel words of an epilogue, four columns at a time: the int32 / f32 bias and the QUANT_PRE words of the
// tile's columns go to LDS before the main loop (copies older than the loop's, whose first wait covers them), so the
// epilogue starts without a trip to memory.  Absent vectors give `no_bias` (0, or -0.0f: adding it changes no fp32
// value) and the scalar word (the bits of 1.0f where nothing is to be multiplied), so the arithmetic has no branches.
struct ColWords {
    uint32_t bias[4];
    float m1[4];
    uint32_t lo[4], hi[4];
};
struct ColLds {
    static constexpr int BYTES = 3072;  // up to 256 columns
    const uint8_t* base;
    bool has_bias, has_words;
    uint32_t no_bias;
    uint64_t scalar;
    // waves 0, 1 and 2 issue one 1 KiB copy each (modulo the workgroup's waves)
    __device__ __forceinline__ void request(uint8_t* lds, int nw, const void* bias, uint32_t none, const uint64_t* words,
                                            uint64_t qscalar, int64_t n0, int cols)
    {
        base = lds;
        has_bias = bias != nullptr;
        has_words = words != nullptr;
        no_bias = none;
        scalar = qscalar;
        const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
        if (has_bias && wave == 0)
            dma16(make_rsrc4((const uint32_t*)bias + n0, (uint32_t)cols * 4u), lds_addr(lds), (uint32_t)lane * 16u);
        if (has_words) {
            const rsrc4_t r = make_rsrc4(words + n0, (uint32_t)cols * 8u);
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (wave == (1 + h) % nw) dma16(r, lds_addr(lds) + 1024 + h * 1024, (uint32_t)(h * 1024 + lane * 16));
        }
    }
    // one column's
    __device__ __forceinline__ uint32_t bias(int c) const { return has_bias ? *(const uint32_t*)(base + c * 4) : no_bias; }
    __device__ __forceinline__ uint64_t word(int c) const
    {
        return has_words ? *(const uint64_t*)(base + 1024 + c * 8) : scalar;
    }
    __device__ __forceinline__ ColWords operator()(int c) const
    {
        ColWords w;
        const u32x4 b = has_bias ? *(const u32x4*)(base + c * 4) : (u32x4){no_bias, no_bias, no_bias, no_bias};
        const u32x4 s = {(uint32_t)scalar, (uint32_t)(scalar >> 32), (uint32_t)scalar, (uint32_t)(scalar >> 32)};
        const u32x4 x = has_words ? *(const u32x4*)(base + 1024 + c * 8) : s;
        const u32x4 y = has_words ? *(const u32x4*)(base + 1024 + c * 8 + 16) : s;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            w.bias[e] = b[e];
            w.lo[e] = e < 2 ? x[2 * e] : y[2 * e - 4];
            w.hi[e] = e < 2 ? x[2 * e + 1] : y[2 * e - 3];
            w.m1[e] = quant_pre_m1(w.lo[e]);
        }
        return w;
    }
};

}  // namespace ascq
