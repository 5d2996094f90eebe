// arc_pf_gemm.hpp -- the prompt pass's tiled GEMM on packed weights (gfx950
// MFMA): Y[m][n] = sum_k X[m][k] W[n][k], X fp16, W Q4_K or padded Q6_K
// decoded to fp16 in registers, fp32 accumulation.
//
// Workgroup of WN waves; each takes all MF*32 rows of X in the tile and 32 weight
// rows of its own with v_mfma_f32_32x32x16_f16 (lane l: X row / weight row l%32,
// 8 of the 16 K elements by half-wave kh = l/32).  The K order is the one that
// every kernel of the prompt pass has summed in (half block p of 128 elements,
// step r of 8, half-wave kh):
//   elements p*128 + (r>>1)*32 + 16kh + 8(r&1) .. +7,
// so that results stay the same bit for bit; X is read from LDS in the same
// order.  Both formats hold a lane's 8 elements of a step in whole dwords of the
// 16-byte pieces of the packed block that it loads:
//   Q4_K: nibble (r>>1)&1 of bytes 16kh + 8(r&1) .. +7 of qs chunk 2p + (r>>2)
//   Q6_K: quarter q = r>>1 of half p: ql bytes 64p + 32(q&1) + 16kh + 8(r&1) ..
//         +7, nibble q>>1, and qh bytes 32p + 16kh + 8(r&1) .. +7, bits 2q, 2q + 1
// (Half-wave kh on chunk 2p + kh or on quarter kh + 2(r>>2) would halve a lane's
// Q4_K factors, but costs Q6_K a fourth load and shifts by kh, and measured no
// faster: q|k|v at 23 rows 12.9 us against 12.5 here, down 56.4 against 55.5,
// gate/up at 256 rows 74.0 against 74.9.)
//
// What bounds it: instruction issue, and at full size the chip's power (a
// library fp16 product of 8192^3 runs at 1.23 PFLOP/s on this card, one of 256 x
// 37888 x 3584 without any decoding at 0.94).  A 32x32x16 MFMA takes 32 cycles
// and two of their eight issue slots, so six other vector instructions are free
// with two waves per SIMD (a 16x16x32 one takes 16 cycles and leaves two).  The
// loop spends 2.59 per Q4_K weight (0.75 to mask the codes, v_fma_mix_f32, half a
// v_cvt_pk_f16_f32, the rest factors, scales and addresses) and 3.70 per Q6_K
// weight.  Each wave takes all rows of the pass, so a weight is decoded once and
// feeds up to 8 MFMAs: as many other vector instructions and one LDS read (4
// cycles of the LDS) per MFMA.  Whole calls, before (34 instructions to decode 8
// weights, X through registers, two barriers' skew per super-block, a 30 KB
// epilogue) and now: gate/up 18944 x 3584 at 256 rows 100 / 78 us (890 TFLOP/s), at
// 100 rows 62 / 43; down 3584 x 18944 69 / 55; q|k|v at 23 rows 18.6 / 12.5.
// The weights are loaded 12 steps ahead: with 8 (and waited for together with X)
// weights from HBM cost 10 us more than weights from the Infinity Cache (gate/up at
// 256 rows); now 81.4 us over ten sets of weights in turn, 80.7 over one.  Inside a
// prompt the launch still takes 8 us longer (88.9 traced), the weights being no
// reason for it.  Tiles measured for the gate/up kernel alone: 32 x 256 per wave, 8
// waves 76-78 us; 64 x 128 (each weight decoded twice) 87; 48 x 128 and 48 x 256 with
// 16x16x32 77-78, 80 x 128 in 4 waves 78.
//
// X goes from global memory straight into LDS (16 bytes per lane, no
// registers), half a super-block (128 columns) per stage, two stages.  A stage's
// row is 256 bytes; its 16-byte pieces are stored at piece ^ (row % 16), so 16
// consecutive rows of a fragment read lie in 16 different bank groups.
// One barrier per stage, two fragments before its end: by then every wave holds
// those in registers, so the barrier both frees the stage for the next fill and
// publishes the other one, whose first fragments are read behind the MFMAs left.
#pragma once

#include "arc_device.hpp"

namespace arc {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // native vector: stays in registers

struct PfGemm {
    const uint8_t* w0;   // PLAIN: the weight rows; SWIGLU: gate
    const uint8_t* w1;   // SWIGLU: up
    uint64_t row_bytes;
    uint32_t N;          // weight rows = output columns
    uint32_t nb;         // super-blocks per weight row
    uint32_t bps;        // super-blocks per split (grid.y = splits)
    uint32_t M;          // valid rows
    uint32_t mpad;       // rows of the partial buffer per split
    const _Float16* x;   // [M][ldx], 16-byte aligned rows
    uint32_t ldx;
    float* out;          // PLAIN: [split][mpad][ldo], columns [0, N)
    uint32_t ldo;
    uint32_t tiles;      // column tiles (workgroups along x) of this operand
    _Float16* s;         // SWIGLU: the output, [M][lds_out]
    uint32_t lds_out;
};

constexpr int kMmKT = 128;             // K columns per LDS stage
constexpr int kMmRowB = kMmKT * 2;     // bytes of a stage row

// The bytes of one weight row's super-block that one lane consumes: the codes
// of its two halves and the scales as loaded ...
template <int FMT>
struct MmCodes;
template <>
struct MmCodes<kFmtQ4> {
    u32x4 q[2][2];   // half p, chunk 2p + i: qs bytes 64p + 32i + 16kh .. +15
};
template <>
struct MmCodes<kFmtQ6P> {
    u32x4 ql[2][2];  // half h: ql bytes 64h + 32i + 16kh .. +15
    u32x4 qh[2];     // half h: qh bytes 32h + 16kh .. +15
};
template <int FMT>
struct MmHdr;
template <>
struct MmHdr<kFmtQ4> {
    u32x4 hdr;    // d, dmin, the 12 scale/min bytes
};
template <>
struct MmHdr<kFmtQ6P> {
    u32x4 sc;     // the 16 int8 scales
    uint32_t d;   // d in the low half
};
// ... and with the lane's scales picked out.
template <int FMT>
struct MmScale;
template <>
struct MmScale<kFmtQ4> {
    uint32_t sc[2], mn[2];  // half p, byte j: sub-block 4p + j (steps 2j, 2j + 1)
    float d24, dmin;        // d * 2^24
};
template <>
struct MmScale<kFmtQ6P> {
    uint32_t sc[2][2];  // half h, byte 2j of dword i: quarter 2i + j, its 16-element half kh (steps 2(2i + j), +1)
    float d;
};
template <int FMT>
constexpr int mm_block_bytes()
{
    return FMT == kFmtQ4 ? kQ4Bytes : kQ6PBytes;
}

__device__ __forceinline__ u32x4 mm_ld16(__amdgpu_buffer_rsrc_t w, uint32_t voff, uint32_t soff)
{
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(w, voff, soff, 0));
}

// Through a buffer descriptor over the wave's weight rows: `row` is the
// lane's row, `blk` (uniform) the super-block's offset in it.
template <int FMT, int P>
__device__ __forceinline__ void mm_load_codes(__amdgpu_buffer_rsrc_t w, uint32_t row, uint32_t blk, uint32_t kh,
                                              MmCodes<FMT>& r)
{
    const uint32_t at = row + 16u * kh;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if constexpr (FMT == kFmtQ4)
            r.q[P][i] = mm_ld16(w, at + (16u + 64u * P + 32u * i), blk);
        else
            r.ql[P][i] = mm_ld16(w, at + (64u * P + 32u * i), blk);
    }
    if constexpr (FMT != kFmtQ4) r.qh[P] = mm_ld16(w, at + (128u + 32u * P), blk);
}

template <int FMT, int P>
__device__ __forceinline__ void mm_take(MmCodes<FMT>& to, const MmCodes<FMT>& from)
{
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if constexpr (FMT == kFmtQ4)
            to.q[P][i] = from.q[P][i];
        else
            to.ql[P][i] = from.ql[P][i];
    }
    if constexpr (FMT != kFmtQ4) to.qh[P] = from.qh[P];
}

template <int FMT>
__device__ __forceinline__ void mm_load_hdr(__amdgpu_buffer_rsrc_t w, uint32_t row, uint32_t blk, MmHdr<FMT>& r)
{
    if constexpr (FMT == kFmtQ4) {
        r.hdr = mm_ld16(w, row, blk);
    } else {
        r.sc = mm_ld16(w, row + 192u, blk);
        r.d = __builtin_amdgcn_raw_buffer_load_b32(w, row + 208u, blk, 0);
    }
}

template <int FMT>
__device__ __forceinline__ void mm_unpack(const MmHdr<FMT>& r, uint32_t kh, MmScale<FMT>& c)
{
    if constexpr (FMT == kFmtQ4) {
        c.sc[0] = r.hdr.y & 0x3f3f3f3fu;
        c.sc[1] = (r.hdr.w & 0x0f0f0f0fu) | ((r.hdr.y >> 2) & 0x30303030u);
        c.mn[0] = r.hdr.z & 0x3f3f3f3fu;
        c.mn[1] = ((r.hdr.w >> 4) & 0x0f0f0f0fu) | ((r.hdr.z >> 2) & 0x30303030u);
        c.d24 = f16_bits_to_f32(r.hdr.x) * 16777216.0f;
        c.dmin = f16_bits_to_f32(r.hdr.x >> 16);
    } else {
        // scale byte 8h + 2q + kh, q = 2i + j: byte 2j + kh of scale dword 2h + i
        const uint32_t sh = 8u * kh;
        c.sc[0][0] = r.sc.x >> sh;
        c.sc[0][1] = r.sc.y >> sh;
        c.sc[1][0] = r.sc.z >> sh;
        c.sc[1][1] = r.sc.w >> sh;
        c.d = f16_bits_to_f32(r.d);
    }
}

constexpr int kMmFactorSteps = 2;  // steps whose weights share one factor pair

// Factors of the steps from R on (R a multiple of kMmFactorSteps) of half P:
// weight = code * 2^-24 * a + n with the code read as an fp16 subnormal
// (Q4_K high nibbles as 16 * code).
template <int FMT, int P, int R>
__device__ __forceinline__ void mm_factors(const MmScale<FMT>& c, float& a, float& n)
{
    if constexpr (FMT == kFmtQ4) {
        a = ((R & 2) ? c.d24 * 0.0625f : c.d24) * byte_f(c.sc[P], R >> 1);
        n = -(c.dmin * byte_f(c.mn[P], R >> 1));
    } else {
        const float f = c.d * float(int8_t(uint8_t(c.sc[P][R >> 2] >> (8 * (R & 2)))));
        a = f * 16777216.0f;
        n = f * -32.0f;
    }
}

// Four weights from two dwords holding codes in the low bits of their
// halves: elements 0, 2 in `ev`, 1, 3 in `od`.  Each is the element decode's
// fp32 value (d has 11 significant bits, a scale at most 7, a code at most 6,
// so a and the product are exact in fp32 and only the last add rounds) rounded
// to fp16: v_fma_mix_f32 and, per pair, v_cvt_pk_f16_f32 (the one-instruction
// v_fma_mix{lo,hi}_f16 rounds once, which differs by an fp16 ulp where the fp32
// value is an fp16 tie, and runs at half rate: 8.5 cycles per wave against 4.3).
__device__ __forceinline__ void mm_mix4(uint32_t ev, uint32_t od, float a, float n, half8& o, int at)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const half2_t e = __builtin_bit_cast(half2_t, ev), d = __builtin_bit_cast(half2_t, od);
    const f32x2 v0 = {__builtin_fmaf(static_cast<float>(e.x), a, n),
                      __builtin_fmaf(static_cast<float>(d.x), a, n)};
    const f32x2 v1 = {__builtin_fmaf(static_cast<float>(e.y), a, n),
                      __builtin_fmaf(static_cast<float>(d.y), a, n)};
    const half2_t h0 = __builtin_convertvector(v0, half2_t), h1 = __builtin_convertvector(v1, half2_t);
    o[at] = h0.x;
    o[at + 1] = h0.y;
    o[at + 2] = h1.x;
    o[at + 3] = h1.y;
}

// The lane's 8 weights of step R of half P.
template <int FMT, int P, int R>
__device__ __forceinline__ half8 mm_dequant(const MmCodes<FMT>& c, float a, float n)
{
    half8 o;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int dw = 2 * (R & 1) + k;
        uint32_t ev, od;
        if constexpr (FMT == kFmtQ4) {
            constexpr uint32_t m = (R & 2) ? 0x00f000f0u : 0x000f000fu;
            ev = opaque(c.q[P][R >> 2][dw] & m);
            od = opaque((c.q[P][R >> 2][dw] >> 8) & m);
        } else {
            // 6-bit codes per byte: ql nibble | 2 qh bits (at 2q) of quarter q at bits 4, 5
            constexpr int q = R >> 1;
            const uint32_t l = c.ql[P][q & 1][dw], h = c.qh[P][dw];
            const uint32_t u = ((q < 2 ? l : l >> 4) & 0x0f0f0f0fu) |
                               ((q < 2 ? h << (4 - 2 * q) : h >> (2 * q - 4)) & 0x30303030u);
            ev = opaque(u & 0x00ff00ffu);
            od = opaque((u >> 8) & 0x00ff00ffu);
        }
        mm_mix4(ev, od, a, n, o, 4 * k);
    }
    return o;
}

// 16-byte piece (8 elements) of a 128-column stage row that half-wave kh
// multiplies in step r: mm_piece0(kh) ^ mm_piece_step(r) (their bits are apart).
__device__ __forceinline__ constexpr uint32_t mm_piece0(uint32_t kh)
{
    return kh * 2u;
}
__device__ __forceinline__ constexpr uint32_t mm_piece_step(int r)
{
    return uint32_t(r >> 1) * 4u + uint32_t(r & 1);
}

// v / (1 + e^-v) with the library's exponential and an IEEE division: within 1.7e-7
// of the exact value.  v_exp_f32(v * -log2 e) and v_rcp_f32 take some 20
// instructions less per value (gate/up at 256 rows 74.9 against 77.6 us, at 100
// rows 40.9 against 42.8), but the product's rounding enters the exponent, so
// the relative error grows with |v| (1.0e-6 at |v| = 20) and fp16 results flip.
__device__ __forceinline__ float mm_silu(float v)
{
    return v / (1.0f + expf(-v));
}

// Workgroup barrier ordering LDS only: global loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

typedef __attribute__((address_space(3))) void lds_void;

// The largest divisor of n that is at most `most`.
constexpr int mm_divisor(int n, int most)
{
    int d = most < n ? most : n;
    while (n % d) --d;
    return d;
}

template <int FMT, int MF, int WN>
struct Mm {
    static constexpr int kRows = 32 * MF;                // X rows of the tile
    static constexpr int kStageB = kRows * kMmRowB;      // bytes of a stage
    static constexpr int kFill = kRows / 4 / WN;          // 1 KB fills (4 rows) per wave and stage
    static constexpr int kD = 4;                         // X fragments held, read kD uses ahead
    static constexpr int kUses = 8 * MF;                 // X fragments of a stage
    static constexpr int kSync = kUses - kD / 2;         // fragment in front of which the stage changes
    static constexpr int kBB = mm_block_bytes<FMT>();
    static_assert(kRows % (4 * WN) == 0 && kUses % kD == 0, "whole fills per wave, whole rounds of the X ring");

    f32x16 acc[MF];
    half8 a[kD];
    half8 b[2];
    MmCodes<FMT> codes;         // in use
    MmCodes<FMT> next;          // in flight: 12 steps (about 3 us) from its load to its first use
    MmHdr<FMT> hdr;
    MmScale<FMT> scale;
    float fa, fn;
    uint32_t kh, wave;
    uint32_t frag;              // byte address of step 0's piece of the lane's first row
    uint32_t voff[kFill];       // byte offsets of the lane's fills (column 0)
    __amdgpu_buffer_rsrc_t xr;
    __amdgpu_buffer_rsrc_t wr;  // the wave's weight rows
    uint32_t wrow;              // byte offset of the lane's row

    __device__ __forceinline__ void init_x(const PfGemm& p)
    {
        const uint32_t lane = threadIdx.x & 63u, l31 = lane & 31u;
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        kh = lane >> 5;
        // (opaque: seen through, the row offsets became ors instead of immediates)
        frag = opaque(l31 * kMmRowB + ((mm_piece0(kh) ^ (l31 & 15u)) << 4));
        xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(p.x), (short)0, int(p.M * p.ldx * 2u), 0x00020000);
        // fill i of this wave: stage rows 4*(wave*kFill + i) + lane/16; the lane's
        // 16 bytes land at piece lane%16 of that row, which holds source piece
        // (lane%16) ^ (row%16).  Rows past M repeat the last one (their results
        // are not stored).
#pragma unroll
        for (int i = 0; i < kFill; ++i) {
            const uint32_t r = 4u * (wave * kFill + i) + (lane >> 4);
            voff[i] = min(r, p.M - 1u) * p.ldx * 2u + (((lane & 15u) ^ (r & 15u)) << 4);
        }
#pragma unroll
        for (int i = 0; i < MF; ++i)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[i][j] = 0.0f;
    }

    // Part PART of 4 of this wave's share of columns [128 kx, 128 kx + 128) of X
    // into a stage.
    template <int PART>
    __device__ __forceinline__ void fill(uint8_t* stage, uint32_t kx)
    {
        uint8_t* dst = stage + wave * (kFill * 1024u);
        const uint32_t col = kx * uint32_t(kMmRowB);
#pragma unroll
        for (int i = 0; i < kFill; ++i) {
            const uint32_t v = voff[i];
            if (i * 4 / kFill == PART) __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(dst + i * 1024), 16, v, col, 0, 0);
        }
    }

    // X fragment i of step r.
    __device__ __forceinline__ half8 frag_at(const uint8_t* stage, int r, int i) const
    {
        return *reinterpret_cast<const half8*>(stage + (frag ^ (mm_piece_step(r) << 4)) + i * (32 * kMmRowB));
    }

    // Half P of super-block kb's codes, and with half 0 its scales: kLoads<P>
    // load instructions.
    template <int P>
    static constexpr int kLoads = FMT == kFmtQ4 ? 2 + (P == 0) : 3 + 2 * (P == 0);
    template <int P>
    __device__ __forceinline__ void load_w(uint32_t kb, MmCodes<FMT>& c)
    {
        if constexpr (P == 0) mm_load_hdr<FMT>(wr, wrow, kb * uint32_t(kBB), hdr);
        mm_load_codes<FMT, P>(wr, wrow, kb * uint32_t(kBB), kh, c);
    }

    // Weight fragment of step (P, R).
    template <int P, int R>
    __device__ __forceinline__ half8 make_b()
    {
        if constexpr (P == 0 && R == 0) mm_unpack<FMT>(hdr, kh, scale);
        if constexpr (R % kMmFactorSteps == 0) mm_factors<FMT, P, R>(scale, fa, fn);
        return mm_dequant<FMT, P, R>(codes, fa, fn);
    }

    // Step R of half P of super-block kb from stage `st`; kn is the next
    // super-block.  In front of fragment kSync the stage changes: from there on
    // `st` takes half P of kn, a quarter of the fill per step (issued together
    // right behind the barrier, every wave of the workgroup queued on the load
    // path for about 1000 cycles).  Half P of kn's codes is loaded in step 3,
    // behind the last fill, so that the wait for the fills leaves it in flight
    // (loads complete in issue order): its fragments are made from the last step
    // of the other half on.
    template <int P, int R>
    __device__ __forceinline__ void step(uint8_t* st, uint8_t* ot, uint32_t kb, uint32_t kn)
    {
        constexpr int kNextP = R == 7 ? 1 - P : P, kNextR = (R + 1) & 7;
        if constexpr (R < 3) fill<R + 1>(ot, (P == 0 ? kb : kn) * 2u + (1 - P));
        if constexpr (R == 3) load_w<P>(kn, next);
        if constexpr (R == 7) mm_take<FMT, kNextP>(codes, next);
        b[1 - (R & 1)] = make_b<kNextP, kNextR>();
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            const int u = R * MF + i;
            if (u == kSync) {
                // this wave's fills of `ot`; step 3's weight loads stay in flight
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads<P>) : "memory");
                lds_barrier();
                fill<0>(st, kn * 2u + P);
#pragma unroll
                for (int v = kUses - kD; v < kSync; ++v) a[v % kD] = frag_at(ot, (v + kD - kUses) / MF, (v + kD - kUses) % MF);
            }
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[R & 1], a[u % kD], acc[i], 0, 0, 0);
            if (u + kD < kUses)
                a[u % kD] = frag_at(st, (u + kD) / MF, (u + kD) % MF);
            else if (u >= kSync)
                a[u % kD] = frag_at(ot, (u + kD - kUses) / MF, (u + kD - kUses) % MF);
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    template <int P>
    __device__ __forceinline__ void half_block(uint8_t* st, uint8_t* ot, uint32_t kb, uint32_t kn)
    {
        step<P, 0>(st, ot, kb, kn);
        step<P, 1>(st, ot, kb, kn);
        step<P, 2>(st, ot, kb, kn);
        step<P, 3>(st, ot, kb, kn);
        step<P, 4>(st, ot, kb, kn);
        step<P, 5>(st, ot, kb, kn);
        step<P, 6>(st, ot, kb, kn);
        step<P, 7>(st, ot, kb, kn);
    }

    // Super-blocks [kb0, kb1).
    __device__ __forceinline__ void run(uint8_t* s0, uint8_t* s1, uint32_t kb0, uint32_t kb1)
    {
        load_w<0>(kb0, codes);
        load_w<1>(kb0, next);
        fill<0>(s0, kb0 * 2u);
        fill<1>(s0, kb0 * 2u);
        fill<2>(s0, kb0 * 2u);
        fill<3>(s0, kb0 * 2u);
        fill<0>(s1, kb0 * 2u + 1u);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
#pragma unroll
        for (int u = 0; u < kD; ++u) a[u] = frag_at(s0, u / MF, u % MF);
        b[0] = make_b<0, 0>();
        for (uint32_t kb = kb0; kb < kb1; ++kb) {
            // the last super-block loads and stages itself again
            const uint32_t kn = kb + 1 < kb1 ? kb + 1 : kb;
            half_block<0>(s0, s1, kb, kn);
            half_block<1>(s1, s0, kb, kn);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last fills, before the stages are reused or freed
        lds_barrier();
    }
};

// D (weights as the A operand): register 4q + j of fragment i holds X row i*32 +
// lane%32 and weight row 8q + 4kh + j of the wave's, so a lane's groups of four
// values are consecutive output columns.
template <int FMT, int MF, int WN, bool SWIGLU>
__device__ __forceinline__ void mm_body(const PfGemm& p, uint32_t tile, uint8_t* s0, uint8_t* s1)
{
    using T = Mm<FMT, MF, WN>;
    static_assert(!SWIGLU || WN % 2 == 0, "gate and up waves");
    T t;
    t.init_x(p);
    const uint32_t l31 = threadIdx.x & 31u;
    constexpr int kCols = SWIGLU ? 16 * WN : 32 * WN;  // output columns of the tile
    const bool up = SWIGLU && t.wave >= WN / 2;
    const uint32_t c0 = (SWIGLU ? t.wave % (WN / 2) : t.wave) * 32u;  // the wave's first column in the tile
    const uint32_t kb0 = SWIGLU ? 0u : blockIdx.y * p.bps, kb1 = SWIGLU ? p.nb : min(p.nb, kb0 + p.bps);
    const uint32_t row0 = tile * kCols;  // < N
    // the wave's own weight rows (past N: the last row again), so that 32-bit
    // offsets reach every K that the host lets through
    const uint32_t first = min(row0 + c0, p.N - 1u), rows = min(p.N - first, 32u);
    t.wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(up ? p.w1 : p.w0) + uint64_t(first) * p.row_bytes, (short)0,
                                             int(rows * uint32_t(p.row_bytes)), 0x00020000);
    t.wrow = min(l31, rows - 1u) * uint32_t(p.row_bytes);
    t.run(s0, s1, kb0, kb1);

    auto quad = [&](int i, int q) {
        return f32x4{t.acc[i][4 * q], t.acc[i][4 * q + 1], t.acc[i][4 * q + 2], t.acc[i][4 * q + 3]};
    };
    if constexpr (SWIGLU) {
        // Gate values go to stage 0, up values to stage 1 ([row][column] fp32, 32
        // rows of X at a time), and all threads then take 8 columns of a row each:
        // silu(gate) * up, one 16-byte store.  Written out per accumulator by the
        // up waves instead (the gate waves idle), this code ran to 30 KB and the
        // launch's fixed cost to 23 us.
        constexpr int kLd = 32 * (kCols + 4) * 4 <= T::kStageB ? kCols + 4 : kCols;
        constexpr int kFit = T::kStageB / (32 * kLd * 4);
        static_assert(kFit >= 1, "a fragment fits a stage");
        constexpr int kI = mm_divisor(MF, kFit);  // fragments per round
        constexpr int kPieces = kCols / 8;
        const bool vec = ((reinterpret_cast<uintptr_t>(p.s) | (p.lds_out * 2u)) & 15u) == 0;
        float* mine = reinterpret_cast<float*>(up ? s1 : s0);
        const float* sg = reinterpret_cast<const float*>(s0);
        const float* su = reinterpret_cast<const float*>(s1);
#pragma unroll
        for (int ib = 0; ib < MF; ib += kI) {
#pragma unroll
            for (int i = 0; i < kI; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<f32x4*>(mine + (i * 32 + l31) * kLd + c0 + 8 * q + 4 * t.kh) = quad(ib + i, q);
            __syncthreads();
            for (uint32_t e = threadIdx.x; e < uint32_t(kI * 32 * kPieces); e += 64 * WN) {
                const uint32_t r = e / kPieces, c = (e % kPieces) * 8u;
                const uint32_t m = ib * 32u + r, col = tile * kCols + c;
                if (m >= p.M || col >= p.N) continue;
                half8 o;
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const f32x4 gv = *reinterpret_cast<const f32x4*>(sg + r * kLd + c + 4 * q);
                    const f32x4 uv = *reinterpret_cast<const f32x4*>(su + r * kLd + c + 4 * q);
#pragma unroll
                    for (int j = 0; j < 4; ++j) o[4 * q + j] = _Float16(mm_silu(gv[j]) * uv[j]);
                }
                _Float16* dst = p.s + uint64_t(m) * p.lds_out + col;
                if (vec && col + 8u <= p.N) {
                    *reinterpret_cast<half8*>(dst) = o;
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (col + j < p.N) dst[j] = o[j];
                }
            }
            __syncthreads();
        }
    } else {
        const bool vec = (p.ldo & 3u) == 0;  // the partial buffer is 16-byte aligned
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            const uint32_t m = i * 32u + l31;
            if (m >= p.M) continue;
            float* o = p.out + (uint64_t(blockIdx.y) * p.mpad + m) * p.ldo;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t col = row0 + c0 + 8u * q + 4u * t.kh;
                if (vec && col + 4u <= p.N) {
                    *reinterpret_cast<f32x4*>(o + col) = quad(i, q);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (col + j < p.N) o[col + j] = t.acc[i][4 * q + j];
                }
            }
        }
    }
}

template <int FMT, int MF, int WN, bool SWIGLU>
__global__ __launch_bounds__(64 * WN, 1) void k_mm(PfGemm p)
{
    using T = Mm<FMT, MF, WN>;
    __shared__ __align__(1024) uint8_t s0[T::kStageB];
    __shared__ __align__(1024) uint8_t s1[T::kStageB];
    mm_body<FMT, MF, WN, SWIGLU>(p, blockIdx.x, s0, s1);
}

// The q, k (Q4_K) and v (format VF) projections of one layer in one launch:
// q's column tiles, then k's, then v's; all write split partials into one
// [split][mpad][hidden + 2*kv_dim] buffer.
template <int VF, int MF, int WN>
__global__ __launch_bounds__(64 * WN, 1) void k_mm_qkv(PfGemm q, PfGemm k, PfGemm v)
{
    using T = Mm<kFmtQ4, MF, WN>;
    __shared__ __align__(1024) uint8_t s0[T::kStageB];
    __shared__ __align__(1024) uint8_t s1[T::kStageB];
    const uint32_t t = blockIdx.x;
    if (t < q.tiles)
        mm_body<kFmtQ4, MF, WN, false>(q, t, s0, s1);
    else if (t < q.tiles + k.tiles)
        mm_body<kFmtQ4, MF, WN, false>(k, t - q.tiles, s0, s1);
    else
        mm_body<VF, MF, WN, false>(v, t - q.tiles - k.tiles, s0, s1);
}

}  // namespace arc
