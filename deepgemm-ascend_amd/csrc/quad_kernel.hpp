// Four-wave GEMM tile kernel for gfx950: one wave per SIMD, each wave a quadrant of every half of the tile.
//
// The tile's A and B rows are cut into two halves each.  A stage is 128 bytes of K per row (128 e4m3 or
// e2m1, 64 bf16 elements) and runs in four phases, one per pair of halves, in the order
//   (A0, Bf) (A0, B1-f) (A1, B1-f) (A1, Bf),   f = stage parity,
// so that consecutive phases share one operand half and every phase needs only one new half in registers:
// phase 0 reads B1-f, phase 1 A1, phase 2 the next stage's A0 and phase 3 its first B half (B1-f, whose
// registers the phase before has finished with).  A wave owns every other 16-row (bf16: 32-row) block of an A
// half and half the columns of a B half, and reads each of its fragments from LDS exactly once per stage.
//
// LDS holds two stages.  Each half of a slot is refilled (buffer_load ... lds, stage c + 2) as soon as every
// wave has read it: A0 and Bf during phases 0-1, A1 and B1-f during phases 2-3, so a load has 1 to 1.5 stages
// to land and about 1.25 stages of bytes are in flight, against one stage for a ring that is refilled stage
// by stage.  There are two barriers per stage (before phases 0 and 2), each behind a counted vmcnt that
// leaves the loads of the last two half-stages in flight.
//
// What bounds it: matrix issue and, under sustained load, the board's power.  A 16x16x128 MFMA holds a
// SIMD's matrix pipe for 32 cycles, in which a wave can issue about six other instructions, so LDS reads and
// loads are dealt out one at a time between MFMAs (slots), the K offset of a stage rides in the loads' vector
// offset and the row steps in constant scalar offsets (two instructions per load).  Measured on MI355X (e4m3,
// 8192^3, the shortest of twenty passes in a row): MFMA busy 76 % of the cycles against 70 % for the eight-wave kernel
// it replaced, 2.85 against 2.57 PFLOP/s.
//
// e4m3 / e2m1: v_mfma_scale_f32_16x16x128_f8f6f4.  With random e4m3 operands in registers it sustains 4.26
// PFLOP/s against 3.95 for the 32x32x64 form (less power per FLOP); errors against fp64 are the same.
//   operand of lane l = r + 16 g (r = row 0..15, g = 0..3): e4m3 bytes [0,16) hold K [16 g, +16), bytes
//   [16,32) K [64 + 16 g, +16); e2m1 16 bytes hold K [32 g, +32); scale = UE8M0 byte of K block g of row r;
//   accumulator element i = column l % 16 of the second operand, row 4 g + i of the first.
// bf16: v_mfma_f32_32x32x16_bf16 (1.78 PFLOP/s in registers, 1.44 for 16x16x32), laid out as in gemm_kernel.hpp.
// B is the first MFMA operand, so a lane ends with runs of four consecutive columns of one row of D.
#pragma once

#include "gemm_kernel.hpp"

namespace dg {

typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(3))) i32x4 lds_i32x4;

// s_waitcnt vmcnt(VM) lgkmcnt(0)
template <int VM>
__device__ __forceinline__ void wait_vmcnt_lds() {
    constexpr int v = VM > 63 ? 63 : VM;
    __builtin_amdgcn_s_waitcnt((v & 0xf) | ((v >> 4) << 14) | (0x7 << 4));
}

// D += first . second on v_mfma_scale_f32_16x16x128_f8f6f4, the accumulator in AGPRs (IN_V: in VGPRs).
// Inline asm: given the builtin, the register allocator moves accumulators between the two register files
// inside the main loop.  An MFMA needs two wait states after a VALU write of one of its operands, and a read
// of its result must wait for the pipeline: the callers keep both distances.
template <bool FP4_FIRST, bool IN_V>
__device__ __forceinline__ void mfma_16x16x128(f32x4& d, const i32x4 (&x)[2], const i32x4 (&y)[2], int xs, int ys) {
    const i32x8 yv = __builtin_shufflevector(y[0], y[1], 0, 1, 2, 3, 4, 5, 6, 7);
    const i32x8 x8 = __builtin_shufflevector(x[0], x[1], 0, 1, 2, 3, 4, 5, 6, 7);
    const i32x4 x4 = x[0];
    if constexpr (FP4_FIRST && IN_V)
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0] cbsz:4"
                     : "+v"(d) : "v"(x4), "v"(yv), "v"(xs), "v"(ys));
    else if constexpr (FP4_FIRST)
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0] cbsz:4"
                     : "+a"(d) : "v"(x4), "v"(yv), "v"(xs), "v"(ys));
    else if constexpr (IN_V)
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0]"
                     : "+v"(d) : "v"(x8), "v"(yv), "v"(xs), "v"(ys));
    else
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0]"
                     : "+a"(d) : "v"(x8), "v"(yv), "v"(xs), "v"(ys));
}

// The same for v_mfma_f32_32x32x16_bf16 (16 bytes of each operand per lane).
template <bool IN_V>
__device__ __forceinline__ void mfma_32x32x16_bf16(f32x16& d, const i32x4& x, const i32x4& y) {
    if constexpr (IN_V) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(x), "v"(y));
    else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(d) : "v"(x), "v"(y));
}

// Transposing LDS read of 8 bytes a lane at `addr` + OFF (ds_read_b64_tr_b8 / _b16).  Inline asm: before the
// builtin the compiler waits for every buffer_load ... lds in flight (it cannot tell their destinations from
// the read's), which drained the whole ring at each read (e4m3 4096^3 with both operands MN-major 195 us
// against 55 us K-major).  The result arrives behind a counter the compiler does not see: arrived() before any
// use.
template <bool B16, int OFF>
__device__ __forceinline__ void read_tr(i32x2& out, int addr) {
    static_assert(OFF >= 0 && OFF < 65536, "LDS offset field");
    if constexpr (B16) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=&v"(out) : "v"(addr), "n"(OFF));
    else asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=&v"(out) : "v"(addr), "n"(OFF));
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// (after wait_lds: makes every later use of the values depend on the wait)
__device__ __forceinline__ void arrived(i32x2 (&v)[4]) {
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
}

// Four consecutive outputs of a row as two bf16 pairs (rounded to nearest even, or stochastically).
template <int EPI>
__device__ __forceinline__ i32x2 pack_quartet(f32x4 v, int n) {
    if constexpr (EPI == kEpiBf16SR) {
        const float x[4] = {v[0], v[1], v[2], v[3]};
        uint16_t o[4];
        sr_bf16_quartet(x, (uint32_t)n >> 2, o);
        return i32x2{(int)((uint32_t)o[0] | ((uint32_t)o[1] << 16)), (int)((uint32_t)o[2] | ((uint32_t)o[3] << 16))};
    } else {
        return i32x2{(int)pack_bf16x2(v[0], v[1]), (int)pack_bf16x2(v[2], v[3])};
    }
}

// Old D values (accumulate) of four consecutive columns, as loaded.
template <int EPI, typename T>
__device__ __forceinline__ f32x4 old_values(T w) {
    if constexpr (EPI == kEpiF32) {
        return w;
    } else {
        return f32x4{bf16_to_f32((uint16_t)(w[0] & 0xffff)), bf16_to_f32((uint16_t)((uint32_t)w[0] >> 16)),
                     bf16_to_f32((uint16_t)(w[1] & 0xffff)), bf16_to_f32((uint16_t)((uint32_t)w[1] >> 16))};
    }
}

// Four consecutive columns from n of row m, scaled by alpha already: bias, accumulate and the store, element by
// element where the row ends or its alignment asks for it (columns past the row hash as zeros under
// stochastic rounding).
template <int EPI>
__device__ __forceinline__ void store_quartet(const KParams& p, f32x4 v, uint8_t* d_base, int m, int n, int N, bool pad_row) {
    constexpr bool kF32 = EPI == kEpiF32;
    uint8_t* const d = d_base + ((int64_t)m * p.ldd + n) * (kF32 ? 4 : 2);
    const bool vec = p.vec_store && n + 4 <= N;
    f32x4 old = {0.f, 0.f, 0.f, 0.f};
    if (p.accumulate && vec) {
        typedef typename Cond<kF32, f32x4, i32x2>::type old_t;
        old = old_values<EPI>(*reinterpret_cast<const old_t*>(d));
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        if (n + x >= N) {
            v[x] = 0.f;
            continue;
        }
        if (p.has_bias) v[x] += kF32 ? reinterpret_cast<const float*>(p.bias)[n + x]
                                     : bf16_to_f32(reinterpret_cast<const uint16_t*>(p.bias)[n + x]);
        if (p.accumulate) v[x] += vec ? old[x] : kF32 ? reinterpret_cast<const float*>(d)[x]
                                                      : bf16_to_f32(reinterpret_cast<const uint16_t*>(d)[x]);
    }
    if (pad_row) v = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (kF32) {
        if (vec) {
            *reinterpret_cast<f32x4*>(d) = v;
        } else {
#pragma unroll
            for (int x = 0; x < 4; ++x)
                if (n + x < N) reinterpret_cast<float*>(d)[x] = v[x];
        }
    } else {
        i32x2 w = pack_quartet<EPI>(v, n);
        if (EPI == kEpiBf16SR && pad_row) w = i32x2{0, 0};
        if (vec) {
            *reinterpret_cast<i32x2*>(d) = w;
        } else {
#pragma unroll
            for (int x = 0; x < 4; ++x)
                if (n + x < N) reinterpret_cast<uint16_t*>(d)[x] = (uint16_t)((uint32_t)w[x >> 1] >> (16 * (x & 1)));
        }
    }
}

// FP8 output of a pair of 16-column blocks from column n: lane group q = lane / 16 holds columns
// n + 4 q + {0..3} and n + 16 + 4 q + {0..3} of row m.  (n % 128 == 0 by the host's check and a wave's columns
// start at a multiple of 32: a 32-column group lies inside the row or past it.)
__device__ __forceinline__ void store_fp8_pair(const KParams& p, f32x4 v0, f32x4 v1, uint8_t* d_base, int m, bool row_ok,
                                               int n, int N, int batch, int q) {
    uint32_t amax = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint16_t b = f32_to_bf16_rne(i < 4 ? v0[i & 3] : v1[i & 3]);
        if (i < 4) v0[i & 3] = bf16_to_f32(b); else v1[i & 3] = bf16_to_f32(b);
        amax = max(amax, (uint32_t)(b & 0x7fffu));
    }
    amax = max(amax, (uint32_t)__shfl_xor((int)amax, 16));
    amax = max(amax, (uint32_t)__shfl_xor((int)amax, 32));
    const uint32_t sexp = ue8m0_of_bf16_amax(amax);
    const float inv = __builtin_bit_cast(float, (254u - sexp) << 23);   // 2^(127 - s)
    if (!row_ok || n >= N) return;
    uint8_t* const d = d_base + (int64_t)m * p.ldd + n + 4 * q;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const f32x4 v = h ? v1 : v0;
        int w = __builtin_amdgcn_cvt_pk_fp8_f32(v[0] * inv, v[1] * inv, 0, false);
        w = __builtin_amdgcn_cvt_pk_fp8_f32(v[2] * inv, v[3] * inv, w, true);
        *reinterpret_cast<int*>(d + 16 * h) = w;
    }
    if (q == 0) {
        const int64_t col = (int64_t)batch * N + n;
        p.sfd[((col >> 6) * p.sfd_ld + m) * 2 + ((col >> 5) & 1)] = (uint8_t)sexp;
    }
}

// One operand's half-tile geometry in LDS and its loads.  MN: the operand is MN-major ([K][MN] storage).
// MR = rows of an MFMA block, BLKS = 32 / 16-row blocks the tile has.
template <int B, bool BF16, bool FP4, bool MN>
struct QuadSide {
    static constexpr int MR = BF16 ? 32 : 16;
    static constexpr int UNITS = B / (2 * MR);               // pairs of blocks (one per wave row / column)
    static_assert(UNITS * 2 * MR == B, "tile side");
    static constexpr int NB0 = (UNITS + 1) / 2, NB1 = UNITS / 2;   // blocks of a wave in half 0 / 1
    static constexpr int H0 = NB0 * 2 * MR, H1 = NB1 * 2 * MR;     // rows of half 0 / 1
    static_assert(H0 <= 192 && NB1 >= 1 && (!MN || H0 <= 128), "halves of at most 192 rows (MN-major: 128)");
    static constexpr int RB = FP4 ? 64 : 128;                // bytes of one K-major LDS row
    static constexpr int KROWS = BF16 ? 64 : 128;            // MN-major: K rows of a stage ...
    static constexpr int PITCH = BF16 ? 256 : 128;           // ... of 128 elements each
    // bytes of one half in LDS: K-major rows (e2m1 always 128 of them, so that every wave loads the same
    // number of pieces), MN-major the whole K range of 128 elements
    static constexpr int bytes(int h) { return MN ? KROWS * PITCH : FP4 ? 128 * RB : (h ? H1 : H0) * RB; }
    static constexpr int SLOT = bytes(0) + bytes(1);
    static constexpr int loads(int h) { return bytes(h) / 4096; }   // 1 KB wave loads per wave and half
    static constexpr int nb(int h) { return h ? NB1 : NB0; }
    static constexpr int rows(int h) { return h ? H1 : H0; }
    static constexpr int RPW = 1024 / (MN ? PITCH : RB);     // LDS rows of one wave load
    static constexpr int PPR = (MN ? PITCH : RB) / 16;       // 16-byte pieces of an LDS row
    static constexpr int PIECES = MN ? 4 : FP4 ? 1 : 2;      // LDS reads of a fragment (MN: 8 bytes each)
    // Piece swizzles that spread the rows of one LDS read over the banks (64 banks of 4 bytes; a read's
    // 16-lane phases are those of gemm_kernel.hpp).  K-major: as there for 128-byte rows; 64-byte rows read
    // by 16 rows x 4 pieces.  MN-major: the 8 (bf16: 4) K rows a 16-lane group of a transposing read touches,
    // and the groups served together, land on distinct bank groups.
    static __device__ __forceinline__ int swizzle(int row) {
        if constexpr (MN) return BF16 ? ((row & 3) << 2) : (((row >> 1) & 3) | (((row >> 4) & 1) << 2));
        else if constexpr (FP4) return (0 - (row >> 2)) & 3;
        else return slot_swizzle<8>(row);
    }
};

// A tile's sides and LDS: scales of two slots ([half][A even / odd 64 K, B even / odd 64 K]; 256 bytes each, 512
// where a wave owns more than four blocks of an A half), A, B.
template <int BM, int BN, int KIND, bool AMN, bool BMN>
struct QuadTile {
    static_assert(KIND == kFP8FP8 || KIND == kFP8FP4 || KIND == kBF16, "operand kinds");
    static_assert(KIND != kFP8FP4 || (!AMN && !BMN), "e2m1 operands are K-major");
    using SA = QuadSide<BM, KIND == kBF16, false, AMN>;
    using SB = QuadSide<BN, KIND == kBF16, KIND == kFP8FP4, BMN>;
    static constexpr bool kWide = SA::NB0 > 4;
    static_assert(SB::NB0 <= 4, "scale dwords of a B half: four blocks per wave");
    static constexpr int SF_A = kWide ? 512 : 256, SF_B = 256, SF_HALF = 2 * (SF_A + SF_B), SF_SLOT = KIND == kBF16 ? 0 : 2 * SF_HALF;
    static constexpr int A_OFF = 2 * SF_SLOT, B_OFF = A_OFF + 2 * SA::SLOT, LDS_BYTES = B_OFF + 2 * SB::SLOT;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
};

// One tile.  LIVE: blocks of A half 1 that hold valid rows; the others are not read and contribute no MFMA, and
// their sums are zero.  (A tile that takes another LIVE runs a body of its own: loops that join before one epilogue
// made the register allocator spill the accumulators.)
template <int BM, int BN, int KIND, int EPI, int CT, int CS, int CM, int CN, int CK, bool AMN, bool BMN, int LIVE>
__device__ __forceinline__ void quad_tile_body(const KParams& p, const TileLoc& tl, uint8_t* const smem) {
    constexpr bool kBf16 = KIND == kBF16;
    constexpr bool kFp4B = KIND == kFP8FP4;
    using T = QuadTile<BM, BN, KIND, AMN, BMN>;
    using SA = typename T::SA;
    using SB = typename T::SB;
    constexpr bool kWide = T::kWide;
    constexpr int SF_A = T::SF_A, SF_B = T::SF_B, SF_HALF = T::SF_HALF, SF_SLOT = T::SF_SLOT, A_OFF = T::A_OFF, B_OFF = T::B_OFF;
    constexpr int U = kBf16 ? 2 : 1;                 // 32-byte fragments of a lane per block and stage
    constexpr int KSTEPS = kBf16 ? 4 : 1;            // MFMAs per pair of blocks and stage
    constexpr int KS = kBf16 ? 64 : 128;             // K elements per stage
    constexpr int MR = SA::MR;
    constexpr int NA0 = SA::NB0, NB0 = SB::NB0;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int gemm_type = CT >= 0 ? CT : p.gemm_type;
    const int M = CM > 0 ? CM : p.m, N = CN > 0 ? CN : p.n;
    const int m0 = tl.m0, n0 = tl.n0, k_len = tl.k_len;
    const int rows_a = min(BM, tl.valid_end - m0), rows_b = min(BN, N - n0);
    // K stages of this workgroup: [c0, c0 + num_stages) of the whole K loop
    const int split_k = CS > 0 ? CS : p.split_k;
    const int all_stages = ceil_div(k_len, KS), nk64 = ceil_div(k_len, 64);
    const int c0 = split_k > 1 ? tl.split * p.split_stages : 0;
    const int num_stages = split_k > 1 ? min(p.split_stages, all_stages - c0) : all_stages;
    constexpr int E = kBf16 ? 2 : 1;                 // bytes of an element (MN-major operands)

    // ------------------------------------------------------------------ loads
    // Wave load `it` of a half: LDS rows [RPW (4 it + wave), + RPW), 16 bytes a lane.  The lane's offset
    // holds its row, its swizzled piece and the stage; the scalar offset the half and `it`.
    const int64_t lda = p.lda, ldb = p.ldb;
    const int kbytes_a = gemm_type == kKGrouped || CK > 0 ? k_len * E : p.kbytes_a;
    const int kbytes_b = gemm_type == kKGrouped || CK > 0 ? (kFp4B ? k_len / 2 : k_len * E) : p.kbytes_b;
    // (MN-major: the K rows of the contraction bound the range; K-major: the tile's rows)
    const __amdgpu_buffer_rsrc_t rs_a = AMN ? make_rsrc(tl.a_base + m0 * E, (int64_t)k_len * lda - m0 * E)
                                            : make_rsrc(tl.a_base + (int64_t)m0 * lda, (int64_t)rows_a * lda);
    const __amdgpu_buffer_rsrc_t rs_b = BMN ? make_rsrc(tl.b_base + n0 * E, (int64_t)k_len * ldb - n0 * E)
                                            : make_rsrc(tl.b_base + (int64_t)n0 * ldb, (int64_t)rows_b * ldb);
    const int lrow_a = wave * SA::RPW + lane / SA::PPR, lrow_b = wave * SB::RPW + lane / SB::PPR;
    const int piece_a = ((lane % SA::PPR) ^ SA::swizzle(lrow_a)) * 16, piece_b = ((lane % SB::PPR) ^ SB::swizzle(lrow_b)) * 16;
    const uint32_t lane_a = (uint32_t)(lrow_a * lda + piece_a), lane_b = (uint32_t)(lrow_b * ldb + piece_b);
    constexpr int kDeadOffset = 0x40000000;          // scalar offset that moves every lane out of range
    int soff_a[2][6], soff_b[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int it = 0; it < 6; ++it) {
            const int ra = 4 * SA::RPW * it;
            soff_a[h][it] = __builtin_amdgcn_readfirstlane((int)(AMN ? ra * lda + h * SA::H0 * E : (h * SA::H0 + ra) * lda));
        }
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int rb = 4 * SB::RPW * it;
            soff_b[h][it] = (int)(BMN ? rb * ldb + h * SB::H0 * E : (h * SB::H0 + rb) * ldb);
            // (e2m1 halves of fewer than 128 rows: the pieces past them are not loaded)
            if (kFp4B && rb + wave * SB::RPW >= SB::rows(h)) soff_b[h][it] = kDeadOffset;
            soff_b[h][it] = __builtin_amdgcn_readfirstlane(soff_b[h][it]);
        }
    }
    // Packed-SF loads, a dword = the bytes of a row pair and 64 K: per half stage the four waves fetch A's and
    // B's dwords of the even and the odd 64 K (kWide: each A wave row's by a wave, then B's by two waves and,
    // the same dwords again, by the other two).  LDS dword order [wave row / column][row pair][16-row block], so
    // that one 16-byte read hands a lane the dwords of its row in four blocks.
    constexpr int NSF = kBf16 ? 0 : kWide ? 2 : 1;    // SF loads per wave and half stage
    __amdgpu_buffer_rsrc_t rs_sc, rs_sc2;
    uint32_t lane_sc[2] = {kOOBOffset, kOOBOffset}, lane_sc2[2] = {kOOBOffset, kOOBOffset};
    int sc_stage = 0, sc_stage2 = 0;
    if constexpr (!kBf16) {
        const __amdgpu_buffer_rsrc_t rs_sfa = make_rsrc(tl.sfa + m0, ((int64_t)nk64 * p.sfa_ld - m0) * 2);
        const __amdgpu_buffer_rsrc_t rs_sfb = make_rsrc(tl.sfb + n0, ((int64_t)nk64 * p.sfb_ld - n0) * 2);
        const int lda2 = __builtin_amdgcn_readfirstlane((int)(p.sfa_ld * 2)), ldb2 = __builtin_amdgcn_readfirstlane((int)(p.sfb_ld * 2));
        const int pair = ((lane >> 2) & 7) * 2, blk = lane & 3, w = lane >> 5;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            // (A rows alternate between the wave rows block by block, a wave's B rows are contiguous)
            const int row_b = h * SB::H0 + w * (SB::rows(h) / 2) + blk * 16 + pair;
            const uint32_t off_b = blk < SB::nb(h) && row_b < rows_b ? (uint32_t)((wave & 1) * ldb2 + row_b * 2) : kOOBOffset;
            if constexpr (kWide) {
                const int wide_blk = lane & 7, row_a = h * SA::H0 + wide_blk * 32 + (wave & 1) * 16 + (lane >> 3) * 2;
                if (wide_blk < SA::nb(h) && row_a < rows_a) lane_sc[h] = (uint32_t)((wave >> 1) * lda2 + row_a * 2);
                lane_sc2[h] = off_b;
            } else {
                const int row_a = h * SA::H0 + blk * 32 + w * 16 + pair;
                const uint32_t off_a = blk < SA::nb(h) && row_a < rows_a ? (uint32_t)((wave & 1) * lda2 + row_a * 2) : kOOBOffset;
                lane_sc[h] = wave < 2 ? off_a : off_b;
            }
        }
        rs_sc = kWide || wave < 2 ? rs_sfa : rs_sfb;
        sc_stage = kWide || wave < 2 ? 2 * lda2 : 2 * ldb2;
        if constexpr (kWide) {
            rs_sc2 = rs_sfb;
            sc_stage2 = 2 * ldb2;
        }
    }
    // Offsets of the stage whose loads go out next; past the last stage, past the K of a row and (MN-major)
    // past the operand's columns they lie outside every range, and the lane writes zeros.
    uint32_t va[2], vb_[2], vs[2], vs2[2];
    auto set_stage = [&](int stage) {
        const bool on = stage < num_stages;
        const int c = c0 + stage;
        if constexpr (AMN) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
                va[h] = on && h * SA::H0 * E + piece_a < rows_a * E && piece_a < SA::rows(h) * E
                            ? lane_a + (uint32_t)(c * KS) * (uint32_t)lda : kOOBOffset;
        } else {
            va[0] = va[1] = on && c * SA::RB + piece_a < kbytes_a ? lane_a + c * SA::RB : kOOBOffset;
        }
        if constexpr (BMN) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
                vb_[h] = on && h * SB::H0 * E + piece_b < rows_b * E && piece_b < SB::rows(h) * E
                             ? lane_b + (uint32_t)(c * KS) * (uint32_t)ldb : kOOBOffset;
        } else {
            vb_[0] = vb_[1] = on && c * SB::RB + piece_b < kbytes_b ? lane_b + c * SB::RB : kOOBOffset;
        }
        if constexpr (!kBf16) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {   // (a dead lane stays past the range)
                vs[h] = on ? lane_sc[h] + c * sc_stage : kOOBOffset;
                if constexpr (kWide) vs2[h] = on ? lane_sc2[h] + c * sc_stage2 : kOOBOffset;
            }
        }
    };
    // loads of a group: A half HA, B half HB (and their scales)
    auto group_loads = [](int ha, int hb) constexpr { return SA::loads(ha) + SB::loads(hb) + NSF; };
    auto issue = [&](auto idx_tag, auto s_tag, auto ha_tag, auto hb_tag) {
        constexpr int IDX = decltype(idx_tag)::value, s = decltype(s_tag)::value;
        constexpr int ha = decltype(ha_tag)::value, hb = decltype(hb_tag)::value;
        constexpr int NLA = SA::loads(ha), NLB = SB::loads(hb);
        if constexpr (IDX < NLA) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rs_a, (lds_void*)(smem + A_OFF + s * SA::SLOT + ha * SA::bytes(0) + IDX * 4096 + wave * 1024), 16, va[ha],
                soff_a[ha][IDX], 0, 0);
        } else if constexpr (IDX < NLA + NLB) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rs_b, (lds_void*)(smem + B_OFF + s * SB::SLOT + hb * SB::bytes(0) + (IDX - NLA) * 4096 + wave * 1024), 16,
                vb_[hb], soff_b[hb][IDX - NLA], 0, 0);
        } else if constexpr (kWide && IDX == NLA + NLB) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_sc, (lds_void*)(smem + s * SF_SLOT + ha * SF_HALF + wave * 256), 4,
                                                     vs[ha], 0, 0, 0);
        } else if constexpr (kWide) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rs_sc2, (lds_void*)(smem + s * SF_SLOT + hb * SF_HALF + 2 * SF_A + (wave & 1) * 256), 4, vs2[hb], 0, 0, 0);
        } else if constexpr (!kBf16) {
            const int h = wave < 2 ? ha : hb;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_sc, (lds_void*)(smem + s * SF_SLOT + h * SF_HALF + wave * 256), 4,
                                                     ha == hb ? vs[ha] : wave < 2 ? vs[ha] : vs[hb], 0, 0, 0);
        }
    };
    auto issue_group = [&](int c, auto s_tag, auto ha_tag, auto hb_tag) {
        set_stage(c);
        static_for<group_loads(decltype(ha_tag)::value, decltype(hb_tag)::value)>([&](auto i) { issue(i, s_tag, ha_tag, hb_tag); });
    };

    // ------------------------------------------------------------------ fragments
    const int r = lane % MR, q = lane / MR;
    lds_u8* const lds = (lds_u8*)smem;
    // Per-lane LDS address of piece x of K step u of a wave's first block; half, slot and (K-major) block
    // are constant offsets from it.
    constexpr int XA = AMN ? 1 : SA::PIECES, XB = BMN ? 1 : SB::PIECES;
    int addr_a[U * XA * (AMN ? NA0 : 1)], addr_b[U * XB * (BMN ? NB0 : 1)];
    const int s16 = lane & 15, g16 = lane >> 4;
    auto mn_addr = [&](auto side, int row, int u) -> int {   // (row: first row of the block within the half)
        // transposing reads (gemm_kernel.hpp, load_frag_mn): in each 16-lane group lane s addresses 8 bytes of
        // K row kb + s / 2 (bf16: kb + s / 4), and lane i receives consecutive K of MN row i
        using S = decltype(side);
        if constexpr (!kBf16) {
            const int k = 16 * g16 + (s16 >> 1), pp = row >> 4;
            return k * S::PITCH + ((pp ^ S::swizzle(k)) << 4) + (s16 & 1) * 8;
        } else {
            const int k = u * 32 + 8 * q + (s16 >> 2), col = row + 16 * (g16 & 1) + 4 * (s16 & 3);
            return k * S::PITCH + (((col >> 3) ^ S::swizzle(k)) << 4) + ((col >> 2) & 1) * 8;
        }
    };
    // Rows of a wave's block j: A blocks alternate between the two wave rows (a tile of few valid rows then has
    // its live blocks spread over all waves), a wave's B columns are contiguous, rows(h) / 2 of them.  Blocks lie
    // a multiple of 16 (bf16: 32) rows apart, so that a lane's swizzle is the same for all of them.
    auto km_addr = [&](auto side, int first, int u, int x) -> int {
        using S = decltype(side);
        const int row = first + r;
        int piece;
        if constexpr (kBf16) piece = u * 4 + 2 * x + q;
        else if constexpr (S::RB == 64) piece = q;
        else piece = 4 * x + q;
        return row * S::RB + ((piece ^ S::swizzle(row)) << 4);
    };
    // (the wave columns of an uneven B side start half 1 at another column than half 0)
    constexpr bool kEvenB = SB::H0 == SB::H1;
    int addr_b1[kEvenB ? 1 : U * XB * (BMN ? NB0 : 1)];
    auto fill = [&](auto side, auto mn_tag, int first, int step, int off, auto& out, auto x_tag, auto nb_tag) {
        using S = decltype(side);
        constexpr bool mn = decltype(mn_tag)::value != 0;
        constexpr int X = decltype(x_tag)::value, NBX = decltype(nb_tag)::value;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if constexpr (mn) {
#pragma unroll
                for (int j = 0; j < NBX; ++j) out[u * NBX + j] = off + mn_addr(S{}, first + j * step, u);
            } else {
#pragma unroll
                for (int x = 0; x < X; ++x) out[u * X + x] = off + km_addr(S{}, first, u, x);
            }
        }
    };
    fill(SA{}, Int<AMN>{}, wm * MR, 2 * MR, A_OFF, addr_a, Int<XA>{}, Int<(AMN ? NA0 : 1)>{});
    fill(SB{}, Int<BMN>{}, wn * (SB::H0 / 2), MR, B_OFF, addr_b, Int<XB>{}, Int<(BMN ? NB0 : 1)>{});
    if constexpr (!kEvenB) fill(SB{}, Int<BMN>{}, wn * (SB::H1 / 2), MR, B_OFF, addr_b1, Int<XB>{}, Int<(BMN ? NB0 : 1)>{});
    // scales: 16 bytes = the dwords (row pair) of the wave's blocks; the lane's byte after a shift
    const int addr_sa = (g16 >> 1) * SF_A + wm * (SF_A / 2) + (s16 >> 1) * (kWide ? 32 : 16);
    const int addr_sb = 2 * SF_A + (g16 >> 1) * SF_B + wn * (SF_B / 2) + (s16 >> 1) * 16;
    const int sc_shift = ((s16 & 1) * 2 + (g16 & 1)) * 8;

    i32x4 fa[2][NA0][U][2], fb[2][NB0][U][2];        // [half][block][fragment][16 bytes]
    i32x2 ta[NA0][U][4], tb[NB0][U][4];              // MN-major: the 8-byte pieces of the half being read
    int sa[2][NA0], sb[2][NB0];                      // scales in the low byte
    i32x4 sc_raw[2];                                 // (dwords of four blocks each)
    // 16-byte (MN-major: 8-byte) read X of block j, K step u
    auto read_frag = [&](auto a_tag, auto s_tag, auto h_tag, auto j_tag, auto u_tag, auto x_tag) {
        constexpr bool A = decltype(a_tag)::value != 0, mn = A ? AMN : BMN;
        constexpr int s = decltype(s_tag)::value, h = decltype(h_tag)::value, j = decltype(j_tag)::value;
        constexpr int u = decltype(u_tag)::value, x = decltype(x_tag)::value;
        using S = typename Cond<A, SA, SB>::type;
        constexpr int NBX = A ? NA0 : NB0, X = A ? XA : XB;
        constexpr bool second = !A && h == 1 && !kEvenB;
        constexpr int idx = mn ? u * NBX + j : u * X + x;
        int base;
        if constexpr (A) base = addr_a[idx];
        else base = second ? addr_b1[second ? idx : 0] : addr_b[idx];
        constexpr int at = s * S::SLOT + h * S::bytes(0);
        if constexpr (mn) {
            // e4m3: K kb .. kb + 7 with kb = 16 g + {0, 8, 64, 72}; bf16: K kb .. kb + 3 with kb = 8 q + {0, 4, 16, 20}:
            // the K-major fragment's bytes in order
            constexpr int kb = kBf16 ? (x & 1) * 4 + (x >> 1) * 16 : (x & 1) * 8 + (x >> 1) * 64;
            if constexpr (A) read_tr<kBf16, at + kb * S::PITCH>(ta[j][u][x], base);
            else read_tr<kBf16, at + kb * S::PITCH>(tb[j][u][x], base);
        } else {
            i32x4 (&f)[2] = A ? fa[h][A ? j : 0][u] : fb[h][A ? 0 : j][u];
            f[x] = *(lds_i32x4*)(lds + base + at + j * (A ? 2 : 1) * MR * S::RB);
        }
    };
    // MN-major: the pieces of the half just read have arrived; the fragments take them over
    auto finish_read = [&](auto a_tag, auto h_tag, auto n_tag) {
        constexpr bool A = decltype(a_tag)::value != 0;
        constexpr int h = decltype(h_tag)::value;
        if constexpr (A ? AMN : BMN) {
            wait_lds();
            static_for<decltype(n_tag)::value>([&](auto j_c) {
                static_for<U>([&](auto u_c) {
                    constexpr int j = decltype(j_c)::value, u = decltype(u_c)::value;
                    i32x2 (&t)[4] = A ? ta[A ? j : 0][u] : tb[A ? 0 : j][u];
                    i32x4 (&f)[2] = A ? fa[h][A ? j : 0][u] : fb[h][A ? 0 : j][u];
                    arrived(t);
                    f[0] = __builtin_shufflevector(t[0], t[1], 0, 1, 2, 3);
                    f[1] = __builtin_shufflevector(t[2], t[3], 0, 1, 2, 3);
                });
            });
        }
    };
    auto read_scales = [&](auto a_tag, auto s_tag, auto h_tag, auto x_tag) {
        constexpr bool A = decltype(a_tag)::value != 0;
        constexpr int x = decltype(x_tag)::value;
        sc_raw[x] = *(lds_i32x4*)(lds + (A ? addr_sa : addr_sb) + decltype(s_tag)::value * SF_SLOT + decltype(h_tag)::value * SF_HALF + 16 * x);
    };
    constexpr bool kPinShift = !kWide || CK > 0;
    auto shift_scales = [&](auto a_tag, auto h_tag, auto n_tag, auto prologue_tag) {
        constexpr bool A = decltype(a_tag)::value != 0;
        constexpr int h = decltype(h_tag)::value;
        static_for<decltype(n_tag)::value>([&](auto j_c) {
            constexpr int j = decltype(j_c)::value;
            int v = (int)((uint32_t)sc_raw[j / 4][j % 4] >> sc_shift);
            // (the shift stays ahead of the s_nop that follows: where K is a compile-time constant of few stages the
            // loop is straight-line code, and the compiler moved it to one wait state ahead of the MFMA that reads it;
            // the ahead-of-time loops of the 384-row tiles hold it in place without, and have no register left for it)
            if constexpr (kPinShift || decltype(prologue_tag)::value != 0) asm volatile("" : "+v"(v));
            if constexpr (A) sa[h][j] = v; else sb[h][j] = v;
        });
    };

    typedef typename Cond<kBf16, f32x16, f32x4>::type acc_t;
    // (Tiles of 256 accumulators a lane or more would fill the 256 AGPRs to the last one, and the allocator then
    // moves a block in and out of them in the loop: what passes 248 (384-row tiles: 252), the last blocks, lives in
    // VGPRs.)
    auto nb_a = [](int h) constexpr { return h ? LIVE : SA::NB0; };   // live blocks of A half h
    constexpr int kAccRegs = kBf16 ? 16 : 4, kOver = (SA::NB0 + LIVE) * (SB::NB0 + SB::NB1) * kAccRegs - (kWide ? 252 : 248);
    constexpr int kInV = kOver > 0 ? (kOver + kAccRegs - 1) / kAccRegs : 0;
    auto in_v = [](int ha, int hb, int i, int j) constexpr {
        return ha == 1 && hb == 1 && (LIVE - 1 - i) * SB::NB1 + SB::NB1 - 1 - j < kInV;
    };
    acc_t acc[2][2][NA0][NB0];                        // [A half][B half]
    static_for<4>([&](auto h_c) {
        constexpr int ha = decltype(h_c)::value >> 1, hb = decltype(h_c)::value & 1;
        static_for<nb_a(ha)>([&](auto i) {
            static_for<SB::nb(hb)>([&](auto j) {
                acc_t& d = acc[ha][hb][decltype(i)::value][decltype(j)::value];
                d = acc_t{};
                // (zeros in place before the loop's first MFMA, two wait states and more ahead of it)
                if constexpr (in_v(ha, hb, decltype(i)::value, decltype(j)::value)) asm volatile("" : "+v"(d));
                else asm volatile("" : "+a"(d));
            });
        });
    });
    asm volatile("s_nop 3");
    auto mfma = [&](auto ha_t, auto hb_t, auto i_t, auto j_t, auto u_t) {
        constexpr int ha = decltype(ha_t)::value, hb = decltype(hb_t)::value, i = decltype(i_t)::value;
        constexpr int j = decltype(j_t)::value, u = decltype(u_t)::value;
        acc_t& d = acc[ha][hb][i][j];
        if constexpr (kBf16) {
            mfma_32x32x16_bf16<in_v(ha, hb, i, j)>(d, fb[hb][j][u >> 1][u & 1], fa[ha][i][u >> 1][u & 1]);
        } else {
            mfma_16x16x128<kFp4B, in_v(ha, hb, i, j)>(d, fb[hb][j][u], fa[ha][i][u], sb[hb][j], sa[ha][i]);
        }
    };

    // ------------------------------------------------------------------ main loop
    // Phase P of stage c in slot s (f = s).  Slot i of the phase: MFMA i, then at most one or two LDS reads
    // and loads; scheduling barriers keep the compiler from regrouping them.
    auto phase = [&](auto p_tag, auto s_tag, int c) {
        constexpr int P = decltype(p_tag)::value, s = decltype(s_tag)::value, f = s;
        constexpr int ha = P >= 2, hb = P == 0 || P == 3 ? f : 1 - f;
        constexpr int NA = nb_a(ha), NB = SB::nb(hb), NM = NA * NB * KSTEPS;
        constexpr int NS = NM < 4 ? 6 : NM;           // slots: the first NM hold an MFMA
        // the half read in this phase: B1-f, A1, the next stage's A0, its first B half (1 - f)
        constexpr bool kReadA = P == 1 || P == 2;
        constexpr int rslot = P >= 2 ? s ^ 1 : s, rh = P == 1 ? 1 : P == 2 ? 0 : 1 - f;
        constexpr int RN = kReadA ? nb_a(rh) : SB::nb(rh), RX = kReadA ? SA::PIECES : SB::PIECES;
        constexpr int NSR = kBf16 || RN == 0 ? 0 : kReadA && RN > 4 ? 2 : 1;   // reads of scales
        constexpr int NR = RN * RX * U + NSR;
        // the half stage refilled: {A0, Bf} in phases 0 and 1, {A1, B1-f} in phases 2 and 3
        constexpr int lha = P >= 2, lhb = P >= 2 ? 1 - f : f;
        constexpr int NL = SA::loads(lha) + SB::loads(lhb) + NSF;
        constexpr int L0 = (P & 1) ? (NL + 1) / 2 : 0, L1 = (P & 1) ? NL : (NL + 1) / 2;
        constexpr int first = (P & 1) == 0 ? 1 : 0;   // (slot 0 of phases 0 and 2 holds the barrier)
        // (after the phase's last MFMA and two wait states ahead of the next phase's: two slots earlier the wait for the
        // scales cost 128x128 tiles, of four slots a phase, 3-5 %)
        constexpr int kShift = kPinShift ? NS - 1 : NS - 3;
        // loads that may stay in flight at the barrier: the two half-stages issued last
        constexpr int kFlight = P == 0 ? SA::loads(0) + SB::loads(1 - f) + SA::loads(1) + SB::loads(f) + 2 * NSF
                                       : SA::loads(1) + SB::loads(f) + SA::loads(0) + SB::loads(f) + 2 * NSF;
        static_for<NS>([&](auto i_c) {
            constexpr int i = decltype(i_c)::value;
            if constexpr (i < NM) {
                constexpr int u = i / (NA * NB), blk = i % (NA * NB);
                // (the operand half read last is the outer loop: its first blocks arrived first)
                if constexpr (P < 2) mfma(Int<ha>{}, Int<hb>{}, Int<blk % NA>{}, Int<blk / NA>{}, Int<u>{});
                else mfma(Int<ha>{}, Int<hb>{}, Int<blk / NB>{}, Int<blk % NB>{}, Int<u>{});
            }
            if constexpr ((P & 1) == 0 && i == 0) {
                // what the next two phases read has landed and what they refill has been read by every wave
                // (this MFMA covers part of the wait)
                __builtin_amdgcn_sched_barrier(0);
                wait_vmcnt_lds<kFlight>();
                stage_barrier();
            }
            static_for<NR>([&](auto b_c) {
                constexpr int b = decltype(b_c)::value;
                // (MN-major: the last quarter of the phase is left for the reads to arrive in)
                constexpr int window = (kReadA ? AMN : BMN) ? (NS - first) * 3 / 4 : NS - first;
                constexpr int at = NR <= window ? first + b : first + b * window / NR;
                if constexpr (at == i) {
                    if constexpr (b < NSR) {
                        read_scales(Int<kReadA>{}, Int<rslot>{}, Int<rh>{}, Int<b>{});
                    } else {
                        constexpr int x = b - NSR, blkx = x / RX;
                        read_frag(Int<kReadA>{}, Int<rslot>{}, Int<rh>{}, Int<blkx % RN>{}, Int<blkx / RN>{}, Int<x % RX>{});
                    }
                }
            });
            static_for<L1 - L0>([&](auto l_c) {
                constexpr int l = decltype(l_c)::value;
                constexpr int at = first + l * (NS - first) / (L1 - L0);
                if constexpr (at == i) issue(Int<L0 + l>{}, s_tag, Int<lha>{}, Int<lhb>{});
            });
            if constexpr (NSR > 0 && i == kShift) {
                shift_scales(Int<kReadA>{}, Int<rh>{}, Int<RN>{}, Int<0>{});
                if constexpr (kPinShift) asm volatile("s_nop 1");
            }
            if constexpr (P == 3 && i == NS - 1) set_stage(c + 3);
            __builtin_amdgcn_sched_barrier(0);
        });
        finish_read(Int<kReadA>{}, Int<rh>{}, Int<RN>{});
    };
    auto stage = [&](int c, auto s_tag) {
        phase(Int<0>{}, s_tag, c);
        phase(Int<1>{}, s_tag, c);
        phase(Int<2>{}, s_tag, c);
        phase(Int<3>{}, s_tag, c);
    };
    issue_group(0, Int<0>{}, Int<0>{}, Int<0>{});
    issue_group(0, Int<0>{}, Int<1>{}, Int<1>{});
    issue_group(1, Int<1>{}, Int<0>{}, Int<1>{});
    issue_group(1, Int<1>{}, Int<1>{}, Int<0>{});
    wait_vmcnt_lds<SA::loads(1) + SB::loads(1) + SA::loads(0) + SB::loads(1) + SA::loads(1) + SB::loads(0) + 3 * NSF>();
    stage_barrier();
    static_for<2>([&](auto a_c) {
        constexpr bool A = decltype(a_c)::value == 0;
        if constexpr (!kBf16) {
            read_scales(Int<A>{}, Int<0>{}, Int<0>{}, Int<0>{});
            if constexpr (A && kWide) read_scales(Int<A>{}, Int<0>{}, Int<0>{}, Int<1>{});
            shift_scales(Int<A>{}, Int<0>{}, Int<(A ? NA0 : NB0)>{}, Int<1>{});
        }
        static_for<U>([&](auto u) {
            static_for<(A ? NA0 : NB0)>([&](auto j) {
                static_for<(A ? SA::PIECES : SB::PIECES)>([&](auto x) { read_frag(Int<A>{}, Int<0>{}, Int<0>{}, j, u, x); });
            });
        });
        finish_read(Int<A>{}, Int<0>{}, Int<(A ? NA0 : NB0)>{});
    });
    set_stage(2);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 3");
    int c = 0;
    for (; c + 1 < num_stages; c += 2) {
        stage(c, Int<0>{});
        stage(c + 1, Int<1>{});
    }
    if (c < num_stages) stage(c, Int<0>{});
    __builtin_amdgcn_s_waitcnt(0);
    // (the last MFMAs' results: 19 wait states at most)
    asm volatile("s_nop 15\n\ts_nop 7");
    // A block's accumulator, read where it is used: the empty asm keeps the compiler from copying the whole
    // tile out of the AGPRs ahead of the epilogue's branches.
    auto take = [&](auto ha_c, auto hb_c, auto i_c, auto j_c) -> acc_t {
        acc_t& t = acc[decltype(ha_c)::value][decltype(hb_c)::value][decltype(i_c)::value][decltype(j_c)::value];
        if constexpr (decltype(i_c)::value >= nb_a(decltype(ha_c)::value))
            t = acc_t{};
        else if constexpr (in_v(decltype(ha_c)::value, decltype(hb_c)::value, decltype(i_c)::value, decltype(j_c)::value))
            asm volatile("" : "+v"(t));
        else
            asm volatile("" : "+a"(t));
        return t;
    };

    // ------------------------------------------------------------------ epilogue
    auto row_of = [&](auto ha_c, auto i_c, int w, int rr) -> int {
        constexpr int ha = decltype(ha_c)::value;
        return m0 + ha * SA::H0 + decltype(i_c)::value * 2 * MR + w * MR + rr;
    };
    auto row_state = [&](int m, bool& row_ok, bool& pad_row) {
        row_ok = m < tl.tile_end && !(gemm_type == kMasked && m >= tl.valid_end);
        pad_row = false;
        if (gemm_type == kMGroupedPsum) pad_row = m >= tl.valid_end;
        else if (gemm_type == kMGroupedIdx) pad_row = tl.anchored ? m >= tl.valid_end : row_ok && p.layout[m] != tl.group;
    };
    // first column of the wave's blocks in half hb, within the tile
    auto col_of = [&](auto hb_c) -> int {
        constexpr int hb = decltype(hb_c)::value;
        return hb * SB::H0 + wn * (SB::rows(hb) / 2);
    };
    if (split_k > 1) {
        // This workgroup's partial tile, fp32 [BM][BN] (rows past M left out); quad_reduce_kernel sums the
        // ranges in order and runs the epilogue.
        float* const ws = p.ws + ((int64_t)tl.tile_id * split_k + tl.split) * (BM * BN);
        static_for<2>([&](auto ha_c) {
            static_for<SA::nb(decltype(ha_c)::value)>([&](auto i_c) {
                const int m = row_of(ha_c, i_c, wm, r);
                float* const row = ws + (m - m0) * BN;
                static_for<2>([&](auto hb_c) {
                    static_for<SB::nb(decltype(hb_c)::value)>([&](auto j_c) {
                        const acc_t a = take(ha_c, hb_c, i_c, j_c);
                        float* const d = row + col_of(hb_c) + decltype(j_c)::value * MR + 4 * q;
                        if (m < M) {
                            if constexpr (kBf16) {
#pragma unroll
                                for (int g = 0; g < 4; ++g)
                                    *reinterpret_cast<f32x4*>(d + 8 * g) = f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
                            } else {
                                *reinterpret_cast<f32x4*>(d) = a;
                            }
                        }
                    });
                });
            });
        });
        return;
    }
    constexpr bool kF32 = EPI == kEpiF32;
    constexpr int DE = kF32 ? 4 : 2;                  // bytes of a D element (other than FP8 output)
    if constexpr (EPI == kEpiFp8) {
        static_assert(!kBf16 && SB::NB0 % 2 == 0 && SB::NB1 % 2 == 0, "FP8 output: whole 32-column groups per wave");
        static_for<2>([&](auto ha_c) {
            constexpr int ha = decltype(ha_c)::value;
            static_for<SA::nb(ha)>([&](auto i_c) {
                const int m = row_of(ha_c, i_c, wm, r);
                bool row_ok, pad_row;
                row_state(m, row_ok, pad_row);
                static_for<2>([&](auto hb_c) {
                    constexpr int hb = decltype(hb_c)::value;
                    static_for<SB::nb(hb) / 2>([&](auto j_c) {
                        constexpr int j = 2 * decltype(j_c)::value;
                        store_fp8_pair(p, take(ha_c, hb_c, i_c, Int<j>{}) * p.alpha, take(ha_c, hb_c, i_c, Int<j + 1>{}) * p.alpha, tl.d_base, m, row_ok,
                                       n0 + col_of(hb_c) + 16 * j, N, tl.batch, q);
                    });
                });
            });
        });
        return;
    } else {
    // Vector path: D rows of aligned quartets.  Whole blocks of columns are stored from registers; the one that
    // the row's end cuts goes through LDS as a strip of the tile's rows and is stored element by element.  Rows of
    // unaligned quartets all go through LDS, a block row at a time.
    if (p.vec_store) {
        const int row_cols = N - n0;                  // columns of D from the tile's first
        const int cut = row_cols < BN && row_cols % MR != 0 ? row_cols / MR * MR : BN;   // the cut block's first
        const int stored = min(row_cols, cut);        // columns stored from registers
        auto whole = [&](int first) -> bool { return first < stored; };                   // (a block's first column)
        float* const lds_bias = reinterpret_cast<float*>(smem);                           // [BN], zeros past the row
        float* const strip = lds_bias + 256;                                              // [BM][MR]
        static_assert(BN <= 256 && 1024 + BM * MR * 4 <= T::LDS_BYTES, "staging areas");
        if (p.has_bias || cut < BN) __syncthreads();   // (every wave has read its last fragments)
        if (p.has_bias) {
            if (tid < BN) {
                lds_bias[tid] = tid >= row_cols ? 0.f
                              : kF32 ? reinterpret_cast<const float*>(p.bias)[n0 + tid]
                                     : bf16_to_f32(reinterpret_cast<const uint16_t*>(p.bias)[n0 + tid]);
            }
            __syncthreads();
        }
        // m_indices: which of the lane's rows are padding, read in one burst (read where each row block is stored,
        // every read waited for the stores before it)
        uint32_t idx_pad = 0;
        if (gemm_type == kMGroupedIdx && !tl.anchored) {
            static_for<SA::NB0 + SA::NB1>([&](auto b_c) {
                constexpr int b = decltype(b_c)::value, ha = b >= SA::NB0;
                const int m = row_of(Int<ha>{}, Int<(ha ? b - SA::NB0 : b)>{}, wm, r);
                idx_pad |= (p.layout[min(m, tl.tile_end - 1)] != tl.group ? 1u : 0u) << b;
            });
        }
        constexpr int NQ = (SB::NB0 + SB::NB1) * (kBf16 ? 4 : 1);   // quartets of a row a lane holds
        auto first_of = [&](int t) -> int {   // first column of a quartet's block within the tile
            const int b = kBf16 ? t / 4 : t;
            return b >= SB::NB0 ? col_of(Int<1>{}) + (b - SB::NB0) * MR : col_of(Int<0>{}) + b * MR;
        };
        auto col_at = [&](int t) -> int { return first_of(t) + 4 * q + (kBf16 ? 8 * (t % 4) : 0); };   // its own
        // Old D values (accumulate) of the lane's row in a row block.  Each block's are loaded ahead of the stores of
        // the one before: a load is waited for together with every store that went out before it.  Rows and blocks
        // that are not stored from registers read a place that is, so that no load is conditional.
        constexpr bool kMayAccumulate = EPI == kEpiF32 || EPI == kEpiBf16;
        typedef typename Cond<kF32, f32x4, i32x2>::type old_t;
        old_t old[NQ];
        const bool add_old = kMayAccumulate && p.accumulate && row_cols >= MR;
        auto load_old = [&](auto block_c) {
            constexpr int b = decltype(block_c)::value, ha = b >= SA::NB0;
            const int m = min(row_of(Int<ha>{}, Int<(ha ? b - SA::NB0 : b)>{}, wm, r), tl.tile_end - 1);
            const uint8_t* const row = tl.d_base + ((int64_t)m * p.ldd + n0) * DE;
#pragma unroll
            for (int t = 0; t < NQ; ++t) old[t] = *reinterpret_cast<const old_t*>(row + (whole(first_of(t)) ? col_at(t) : 0) * DE);
        };
        // PLAIN: no bias, no old values and no cut block.  The straight-line code of a tile's rows runs once per tile, so
        // that its size is time.
        auto store_rows = [&](auto plain_tag) {
            constexpr bool PLAIN = decltype(plain_tag)::value != 0;
            if (!PLAIN && add_old) load_old(Int<0>{});
            static_for<2>([&](auto ha_c) {
                constexpr int ha = decltype(ha_c)::value;
                static_for<SA::nb(ha)>([&](auto i_c) {
                    constexpr int row_block = (ha ? SA::NB0 : 0) + decltype(i_c)::value;
                    const int m = row_of(ha_c, i_c, wm, r);
                    const bool row_ok = m < tl.tile_end && !(gemm_type == kMasked && m >= tl.valid_end);
                    const bool pad_row = (gemm_type == kMGroupedPsum || (gemm_type == kMGroupedIdx && tl.anchored)) ? m >= tl.valid_end
                                                                                                                   : (idx_pad >> row_block & 1) != 0;
                    uint8_t* const drow = tl.d_base + ((int64_t)m * p.ldd + n0) * DE;
                    f32x4 v[NQ];
                    int col[NQ];   // a quartet's first column within the tile
                    static_for<SB::NB0 + SB::NB1>([&](auto b_c) {
                        constexpr int b = decltype(b_c)::value, hb = b >= SB::NB0, j = hb ? b - SB::NB0 : b;
                        const acc_t a = take(ha_c, Int<hb>{}, i_c, Int<j>{});
                        const int c0 = col_of(Int<hb>{}) + j * MR + 4 * q;
                        if constexpr (kBf16) {
#pragma unroll
                            for (int g = 0; g < 4; ++g) {
                                v[4 * b + g] = f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]} * p.alpha;
                                col[4 * b + g] = c0 + 8 * g;
                            }
                        } else {
                            v[b] = a * p.alpha;
                            col[b] = c0;
                        }
                        if (!PLAIN && first_of(kBf16 ? 4 * b : b) == cut) {
                            float* const row = strip + (m - m0) * MR + 4 * q;
#pragma unroll
                            for (int g = 0; g < (kBf16 ? 4 : 1); ++g) *reinterpret_cast<f32x4*>(row + 8 * g) = v[kBf16 ? 4 * b + g : b];
                        }
                    });
                    if constexpr (!PLAIN && kMayAccumulate) {
                        if (p.has_bias) {
#pragma unroll
                            for (int t = 0; t < NQ; ++t) v[t] = v[t] + *reinterpret_cast<const f32x4*>(lds_bias + col[t]);
                        }
                        if (add_old) {
#pragma unroll
                            for (int t = 0; t < NQ; ++t) v[t] = v[t] + old_values<EPI>(old[t]);
                            if constexpr (row_block + 1 < SA::NB0 + SA::NB1) load_old(Int<row_block + 1>{});
                        }
                    }
                    if (pad_row) {
#pragma unroll
                        for (int t = 0; t < NQ; ++t) v[t] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
                    if constexpr (kF32) {
                        if (row_ok) {
#pragma unroll
                            for (int t = 0; t < NQ; ++t)
                                if (whole(first_of(t))) *reinterpret_cast<f32x4*>(drow + col[t] * 4) = v[t];
                        }
                    } else {
                        i32x2 pk[NQ];
#pragma unroll
                        for (int t = 0; t < NQ; ++t) {
                            pk[t] = pack_quartet<EPI>(v[t], n0 + col[t]);
                            if (EPI == kEpiBf16SR && pad_row) pk[t] = i32x2{0, 0};
                        }
                        if constexpr (kBf16) {
                            // per 32-column block: after swapping the wave's halves a lane holds 16 columns in a row
                            i32x4 w[NQ / 4][2];
#pragma unroll
                            for (int b = 0; b < NQ / 4; ++b) {
#pragma unroll
                                for (int h = 0; h < 2; ++h) {
                                    const auto s02 = __builtin_amdgcn_permlane32_swap(pk[4 * b + 2][h], pk[4 * b][h], false, false);
                                    const auto s13 = __builtin_amdgcn_permlane32_swap(pk[4 * b + 3][h], pk[4 * b + 1][h], false, false);
                                    w[b][0][h] = (int)s02[0]; w[b][0][2 + h] = (int)s02[1];
                                    w[b][1][h] = (int)s13[0]; w[b][1][2 + h] = (int)s13[1];
                                }
                            }
                            if (row_ok) {
#pragma unroll
                                for (int b = 0; b < NQ / 4; ++b) {
                                    if (!whole(first_of(4 * b))) continue;
                                    uint8_t* const d = drow + (first_of(4 * b) + (q ? 0 : 16)) * 2;
                                    *reinterpret_cast<i32x4*>(d) = w[b][0];
                                    *reinterpret_cast<i32x4*>(d + 16) = w[b][1];
                                }
                            }
                        } else {
                            // per pair of 16-column blocks of a half: after swapping the odd and even lane groups a lane
                            // holds eight columns in a row of block q % 2, from 8 (q / 2) on
                            i32x4 w[NQ / 2];
                            static_for<2>([&](auto hb_c) {
                                constexpr int hb = decltype(hb_c)::value;
                                static_for<SB::nb(hb) / 2>([&](auto j_c) {
                                    constexpr int j = decltype(j_c)::value, t = (hb ? SB::NB0 : 0) + 2 * j;
                                    const auto s0 = __builtin_amdgcn_permlane16_swap(pk[t][0], pk[t + 1][0], false, false);
                                    const auto s1 = __builtin_amdgcn_permlane16_swap(pk[t][1], pk[t + 1][1], false, false);
                                    w[(hb ? SB::NB0 / 2 : 0) + j] = i32x4{(int)s0[0], (int)s1[0], (int)s0[1], (int)s1[1]};
                                });
                            });
                            if (row_ok) {
                                static_for<2>([&](auto hb_c) {
                                    constexpr int hb = decltype(hb_c)::value;
                                    const int cb = col_of(hb_c);
                                    static_for<SB::nb(hb) / 2>([&](auto j_c) {
                                        constexpr int j = decltype(j_c)::value;
                                        const int first = cb + 32 * j + 16 * (q & 1);
                                        if (whole(first)) {
                                            i32x4* const d = reinterpret_cast<i32x4*>(drow + (first + 8 * (q >> 1)) * 2);
                                            if (p.stream_d) __builtin_nontemporal_store(w[(hb ? SB::NB0 / 2 : 0) + j], d);
                                            else *d = w[(hb ? SB::NB0 / 2 : 0) + j];
                                        }
                                    });
                                    if constexpr (SB::nb(hb) % 2 != 0) {
                                        constexpr int j = SB::nb(hb) - 1;
                                        if (whole(cb + 16 * j))
                                            *reinterpret_cast<i32x2*>(drow + (cb + 16 * j + 4 * q) * 2) = pk[(hb ? SB::NB0 : 0) + j];
                                    }
                                });
                            }
                        }
                    }
                });
            });
        };
        if (p.has_bias || p.accumulate || cut < BN) store_rows(Int<0>{});
        else store_rows(Int<1>{});
        if (cut < BN) {
            __syncthreads();
            for (int e = tid; e < BM * (MR / 4); e += 256) {
                const int m = m0 + e / (MR / 4), n = n0 + cut + e % (MR / 4) * 4;
                bool row_ok, pad_row;
                row_state(m, row_ok, pad_row);
                if (!row_ok || n >= N) continue;
                store_quartet<EPI>(p, *reinterpret_cast<const f32x4*>(strip + e * 4), tl.d_base, m, n, N, pad_row);
            }
        }
        return;
    }
    static_for<2>([&](auto ha_c) {
        constexpr int ha = decltype(ha_c)::value;
        static_for<SA::nb(ha)>([&](auto i_c) {
            // the block row of both wave rows, fp32: [2 MR][BN]
            static_assert(2 * MR * BN * 4 <= T::LDS_BYTES, "staging area");
            float* const st = reinterpret_cast<float*>(smem);
            __syncthreads();
            static_for<2>([&](auto hb_c) {
                constexpr int hb = decltype(hb_c)::value;
                static_for<SB::nb(hb)>([&](auto j_c) {
                    constexpr int j = decltype(j_c)::value;
                    float* const d = st + (wm * MR + r) * BN + col_of(hb_c) + j * MR + 4 * q;
                    if constexpr (kBf16) {
                        const acc_t a = take(ha_c, hb_c, i_c, j_c);
#pragma unroll
                        for (int g = 0; g < 4; ++g)
                            *reinterpret_cast<f32x4*>(d + 8 * g) = f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
                    } else {
                        *reinterpret_cast<f32x4*>(d) = take(ha_c, hb_c, i_c, j_c);
                    }
                });
            });
            __syncthreads();
            for (int e = tid; e < 2 * MR * (BN / 4); e += 256) {
                const int rr = e / (BN / 4), n = n0 + e % (BN / 4) * 4;
                const int m = row_of(ha_c, i_c, rr / MR, rr % MR);
                bool row_ok, pad_row;
                row_state(m, row_ok, pad_row);
                if (!row_ok || n >= N) continue;
                store_quartet<EPI>(p, *reinterpret_cast<const f32x4*>(st + rr * BN + (n - n0)) * p.alpha, tl.d_base, m, n, N, pad_row);
            }
        });
    });
    }
}

// CT / CS / CM / CN / CK: GEMM type, K split and sizes fixed at compile time (-1 / 0: from the arguments).
template <int BM, int BN, int KIND, int EPI, int CT = -1, int CS = 0, int CM = 0, int CN = 0, int CK = 0,
          bool AMN = false, bool BMN = false>
__device__ __forceinline__ void quad_body(const KParams& p, const int vb) {
    using T = QuadTile<BM, BN, KIND, AMN, BMN>;
    using SA = typename T::SA;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[T::LDS_BYTES];
    TileLoc tl;
    if (!locate_tile<BM, BN, 256, KIND, CT, CS, CM, CN, CK, AMN, BMN>(p, vb, -1, threadIdx.x, tl)) return;
    auto run = [&](auto live) {
        quad_tile_body<BM, BN, KIND, EPI, CT, CS, CM, CN, CK, AMN, BMN, decltype(live)::value>(p, tl, smem);
    };
    if constexpr (T::kWide) {
        // anchored tiles end with their group: of 8192 rows routed to 32 groups, 180 to 333 each, a third of
        // the tiles' blocks is dead (N=4096 K=7168: 309 us with every block, 303 without the dead ones)
        const int live = ceil_div(tl.valid_end - tl.m0 - SA::H0, 2 * SA::MR);
        if (!tl.anchored || live > 4) run(Int<SA::NB1>{});
        else if (live > 2) run(Int<4>{});
        else run(Int<2>{});
    } else {
        run(Int<SA::NB1>{});
    }
}

// Workgroups per CU: as many as the LDS holds.  Two 128 x 128 tiles of K-major operands (68 KB each) share a CU and cover
// each other's prologue, epilogue and LDS latency; an MN-major side takes the LDS of 128 elements in each half.
template <int BM, int BN, int KIND, bool AMN, bool BMN>
constexpr int quad_occupancy() { return 2 * QuadTile<BM, BN, KIND, AMN, BMN>::LDS_BYTES <= 160 * 1024 ? 2 : 1; }

template <int BM, int BN, int KIND, int EPI, bool AMN = false, bool BMN = false>
__global__ __launch_bounds__(256, (quad_occupancy<BM, BN, KIND, AMN, BMN>())) void quad_kernel(const KParams p) {
    quad_body<BM, BN, KIND, EPI, -1, 0, 0, 0, 0, AMN, BMN>(p, blockIdx.x + p.vbase);
}

// Second launch of a split-K quad plan: a thread per four consecutive columns of D sums the partials of the
// K ranges in order and stores the outputs.  Bound by the partials' bytes: one coalesced 16-byte read per
// range, all in flight before the first add.
template <int EPI>
__global__ __launch_bounds__(256) void quad_reduce_kernel(const KParams p) {
    const int bm = p.reduce_bm, bn = p.reduce_bn;
    const int64_t e = ((int64_t)(blockIdx.x + p.vbase) * 256 + threadIdx.x) * 4;   // element of the tiles
    const int64_t tile = e / (bm * bn);
    if (tile >= p.num_tiles) return;
    const int in = (int)(e - tile * (bm * bn)), rr = in / bn, cc = in % bn;
    const int per = p.num_m_blocks * p.num_n_blocks, batch = (int)(tile / per);
    int mb, nb;
    swizzle_tile((int)(tile - (int64_t)batch * per), p.num_m_blocks, p.num_n_blocks, p.group_m, mb, nb);
    const int m = mb * bm + rr, n = nb * bn + cc;
    const bool live = m < p.m && n < p.n;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (live) {
        const float* const src = p.ws + tile * p.split_k * (bm * bn) + in;
        f32x4 part[8];
        for (int s0 = 0; s0 < p.split_k; s0 += 8) {
#pragma unroll
            for (int s = 0; s < 8; ++s)
                part[s] = s0 + s < p.split_k ? *reinterpret_cast<const f32x4*>(src + (int64_t)(s0 + s) * (bm * bn))
                                             : f32x4{-0.f, -0.f, -0.f, -0.f};   // (the identity of IEEE addition)
#pragma unroll
            for (int s = 0; s < 8; ++s) v = s0 + s == 0 ? part[0] : v + part[s];
        }
    }
    v = v * p.alpha;
    uint8_t* const d_base = p.d + (int64_t)batch * p.bsd * p.out_esize;
    if constexpr (EPI == kEpiFp8) {
        // eight neighbouring threads hold 32 columns of a row
        uint32_t amax = 0;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const uint16_t b = f32_to_bf16_rne(v[x]);
            v[x] = bf16_to_f32(b);
            amax = max(amax, (uint32_t)(b & 0x7fffu));
        }
#pragma unroll
        for (int off = 1; off < 8; off <<= 1) amax = max(amax, (uint32_t)__shfl_xor((int)amax, off));
        const uint32_t sexp = ue8m0_of_bf16_amax(amax);
        const float inv = __builtin_bit_cast(float, (254u - sexp) << 23);
        if (!live) return;
        int w = __builtin_amdgcn_cvt_pk_fp8_f32(v[0] * inv, v[1] * inv, 0, false);
        w = __builtin_amdgcn_cvt_pk_fp8_f32(v[2] * inv, v[3] * inv, w, true);
        *reinterpret_cast<int*>(d_base + (int64_t)m * p.ldd + n) = w;
        if (n % 32 == 0) {
            const int64_t col = (int64_t)batch * p.n + n;
            p.sfd[((col >> 6) * p.sfd_ld + m) * 2 + ((col >> 5) & 1)] = (uint8_t)sexp;
        }
    } else {
        if (live) store_quartet<EPI>(p, v, d_base, m, n, p.n, false);
    }
}

}  // namespace dg
