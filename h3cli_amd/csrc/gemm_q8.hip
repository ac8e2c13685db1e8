// W8A16 projections with the int8 conversion inside a hand-scheduled K loop:
// y[M,N] = x[M,K] . w[N,K]^T (+bias) (+GELU-tanh or SwiGLU), w = bf16(code * scale), one
// scale per output column, FP32 accumulation.
//
// For a few hundred to a few thousand rows converting the whole weight first (five bytes
// of memory traffic per value instead of one) costs as much as a third of the products,
// and gemm_mid's compiler-scheduled loop leaves the matrix cores idle half of the time.
// Here a 256 x 256 output tile is computed by four waves of 128 x 128, one per SIMD, on
// v_mfma_f32_32x32x16_bf16 (4 x 4 accumulator blocks in AGPRs; between these MFMAs, unlike
// between 16 x 16 x 32 ones, VALU instructions cost little). The K loop is one inline-asm
// block; per K tile of 64 (stage ST), four substeps of sixteen MFMAs (16 K each):
//  * the eight fragments of the next substep are read in the first eight MFMA slots into
//    the other register set;
//  * substeps 0-2 convert the next tile's weights: 64 codes per lane, already in
//    registers, about four VALU instructions per MFMA, written to LDS as BF16;
//  * a barrier: every wave has read all fragments of this tile and written its part of
//    the next one;
//  * substep 3 issues the loads of x two tiles and of the codes three tiles ahead, and reads
//    the codes of the tile after next from LDS (each lane the chunks its own wave loaded).
// LDS (160 KB): x stages at 0 and 32 KB, BF16 weight stages at 64 and 96 KB, code stages at
// 128 and 144 KB; 128-byte rows with XOR-swizzled 16-byte chunks, codes in load order.
// Fixed registers: fragment set S v[64 + 32 S ..] (W block I at + 4 I, x block J at + 16 + 4 J),
// codes v128-143, their values v144-159, packed v160-167.
//
// Bound by the power that the MFMAs draw and, behind them, LDS and the conversion (9% faster
// without its VALU instructions). Scales per group of K, loaded with each K tile, cost 20%
// here and stay with gemm_mid. Measured against gemm_mid or, for the 1200 rows, a conversion
// pass and gemm_bf16_pipe, in microseconds: 729 rows, 5376 -> 28672: 214 to 228 (259), 5376 ->
// 21504: 149 (168), 7168 -> 5376: 71 (85), 14336 -> 5376: 114 (129); 1200 rows, 13824 ->
// 5120: 166 (202). A wave of workgroups starts and stores in 16 us (gemm_mid: 7 to 12), which
// leaves no gain for a short K: 700 rows, 1024 -> 14336: 38 (40).
#include "common.h"
#include "internal.h"
#include "gemm.h"

namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int TM = 256, TN = 256, TK = 64;
constexpr int ROW_BYTES = TK * 2, TILE = 256 * ROW_BYTES, CODES = 256 * TK, LDS = 4 * TILE + 2 * CODES;
constexpr int GROUP_M = 4;

__device__ inline unsigned swz(unsigned row, unsigned ch) { return ch ^ ((row >> 1) & 7); }

#define Q_MFMA(S, I, J)                                                                                             \
    "v_mfma_f32_32x32x16_bf16 %[c" #I #J "], v[64+32*" #S "+4*" #I ":64+32*" #S "+4*" #I "+3], "                      \
    "v[64+32*" #S "+16+4*" #J ":64+32*" #S "+16+4*" #J "+3], %[c" #I #J "]\n"
// Fragment F of substep KS (bases w<KS>, x<KS>), stage ST, into set T.
#define Q_RW(T, F, KS, ST)                                                                                          \
    "ds_read_b128 v[64+32*" #T "+4*" #F ":64+32*" #T "+4*" #F "+3], %[w" #KS "] offset:32768*" #ST "+4096*" #F "\n"
#define Q_RX(T, F, KS, ST)                                                                                          \
    "ds_read_b128 v[64+32*" #T "+16+4*" #F ":64+32*" #T "+16+4*" #F "+3], %[x" #KS "] offset:32768*" #ST "+4096*" #F "\n"
// A substep of set S that reads the fragments of substep KS of stage ST into set T; D0..D15
// behind its MFMAs.
#define Q_SUB(S, T, KS, ST, D0, D1, D2, D3, D4, D5, D6, D7, D8, D9, D10, D11, D12, D13, D14, D15)                     \
    Q_MFMA(S, 0, 0) Q_RW(T, 0, KS, ST) D0 Q_MFMA(S, 0, 1) Q_RX(T, 0, KS, ST) D1                                      \
    Q_MFMA(S, 0, 2) Q_RX(T, 1, KS, ST) D2 Q_MFMA(S, 0, 3) Q_RX(T, 2, KS, ST) D3                                      \
    Q_MFMA(S, 1, 0) Q_RX(T, 3, KS, ST) D4 Q_MFMA(S, 1, 1) Q_RW(T, 1, KS, ST) D5                                      \
    Q_MFMA(S, 1, 2) Q_RW(T, 2, KS, ST) D6 Q_MFMA(S, 1, 3) Q_RW(T, 3, KS, ST) D7                                      \
    Q_MFMA(S, 2, 0) D8 Q_MFMA(S, 2, 1) D9 Q_MFMA(S, 2, 2) D10 Q_MFMA(S, 2, 3) D11                                    \
    Q_MFMA(S, 3, 0) D12 Q_MFMA(S, 3, 1) D13 Q_MFMA(S, 3, 2) D14 Q_MFMA(S, 3, 3) D15
#define Q_SUB_EXP(...) Q_SUB(__VA_ARGS__)

// Conversion of chunk C (16 codes): value E from byte E % 4 of code word E / 4, times the
// chunk's scale, rounded in pairs, and the two 16-byte stores into stage ST.
#define Q_CV(C, E, W, B) "v_cvt_f32_i32_sdwa v[144+" #E "], sext(v[128+4*" #C "+" #W "]) dst_sel:DWORD dst_unused:UNUSED_PAD " \
    "src0_sel:BYTE_" #B "\n"
#define Q_CV4(C, W) Q_CV(C, 4*W, W, 0) Q_CV(C, 4*W+1, W, 1) Q_CV(C, 4*W+2, W, 2) Q_CV(C, 4*W+3, W, 3)
#define Q_MU(C, E) "v_mul_f32 v[144+" #E "], v[144+" #E "], %[s" #C "]\n"
#define Q_MU4(C, Q) Q_MU(C, 4*Q) Q_MU(C, 4*Q+1) Q_MU(C, 4*Q+2) Q_MU(C, 4*Q+3)
#define Q_PK(E) "v_cvt_pk_bf16_f32 v[160+" #E "], v[144+2*" #E "], v[144+2*" #E "+1]\n"
#define Q_PKL Q_PK(0) Q_PK(1) Q_PK(2) Q_PK(3)
#define Q_PKH Q_PK(4) Q_PK(5) Q_PK(6) Q_PK(7)
#define Q_WR0(C, ST) "ds_write_b128 %[d0], v[160:163] offset:32768*" #ST "+8192*" #C "\n"
#define Q_WR1(C, ST) "ds_write_b128 %[d1], v[164:167] offset:32768*" #ST "+8192*" #C "\n"
#define Q_RAW(C, ST) "ds_read_b128 v[128+4*" #C ":128+4*" #C "+3], %[rr] offset:16384*" #ST "+4096*" #C "\n"
// Loads: x block T into stage ST, code chunk C into code stage ST.
#define Q_LX(ST, T) "s_add_u32 m0, %[mb], 32768*" #ST "+4096*" #T "\n buffer_load_dwordx4 %[o" #T "], %[sx], %[kx] offen lds\n"
#define Q_LW(ST, C) "s_add_u32 m0, %[mb], 131072+16384*" #ST "+4096*" #C "\n buffer_load_dwordx4 %[q" #C "], %[sw], %[kw] offen lds\n"

// K tile in stage ST (the other one OT): the next tile is converted into OT.
#define Q_TILE(ST, OT)                                                                                              \
    Q_SUB_EXP(0, 1, 1, ST, Q_CV4(0, 0), Q_CV4(0, 1), Q_CV4(0, 2), Q_CV4(0, 3), Q_MU4(0, 0), Q_MU4(0, 1),        \
              Q_MU4(0, 2), Q_MU4(0, 3), Q_PKL, Q_PKH, Q_WR0(0, OT), Q_WR1(0, OT), Q_CV4(1, 0), Q_CV4(1, 1),    \
              Q_CV4(1, 2), Q_CV4(1, 3))                                                                              \
    "s_waitcnt lgkmcnt(0)\n"                                                                                        \
    Q_SUB_EXP(1, 0, 2, ST, Q_MU4(1, 0), Q_MU4(1, 1), Q_MU4(1, 2), Q_MU4(1, 3), Q_PKL, Q_PKH,            \
              Q_WR0(1, OT), Q_WR1(1, OT), Q_CV4(2, 0), Q_CV4(2, 1), Q_CV4(2, 2), Q_CV4(2, 3), Q_MU4(2, 0),          \
              Q_MU4(2, 1), Q_MU4(2, 2), Q_MU4(2, 3))                                                       \
    "s_waitcnt lgkmcnt(0)\n"                                                                                        \
    Q_SUB_EXP(0, 1, 3, ST, Q_PKL, Q_PKH, Q_WR0(2, OT), Q_WR1(2, OT), Q_CV4(3, 0), Q_CV4(3, 1), Q_CV4(3, 2),            \
              Q_CV4(3, 3), Q_MU4(3, 0), Q_MU4(3, 1), Q_MU4(3, 2), Q_MU4(3, 3), Q_PKL, Q_PKH,            \
              Q_WR0(3, OT), Q_WR1(3, OT))                                                                            \
    "s_waitcnt vmcnt(0) lgkmcnt(0)\n"                                                                               \
    "s_barrier\n"                                                                                                   \
    "s_min_u32 %[kx], %[kxn], %[kxm]\n s_add_u32 %[kxn], %[kxn], 128\n"                                             \
    "s_min_u32 %[kw], %[kwn], %[kwm]\n s_add_u32 %[kwn], %[kwn], 64\n"                                              \
    Q_SUB_EXP(1, 0, 0, OT, Q_LX(ST, 0), Q_LX(ST, 1), Q_LX(ST, 2), Q_LX(ST, 3), Q_LX(ST, 4), Q_LX(ST, 5), Q_LX(ST, 6),   \
              Q_LX(ST, 7), Q_RAW(0, ST) Q_LW(OT, 0), Q_RAW(1, ST) Q_LW(OT, 1), Q_RAW(2, ST) Q_LW(OT, 2),               \
              Q_RAW(3, ST) Q_LW(OT, 3), "", "", "", "")                             \
    "s_waitcnt lgkmcnt(0)\n"
// A whole chunk without MFMAs (prologue).
#define Q_CHUNK(C, ST) Q_CV4(C, 0) Q_CV4(C, 1) Q_CV4(C, 2) Q_CV4(C, 3) Q_MU4(C, 0) Q_MU4(C, 1) Q_MU4(C, 2)            \
    Q_MU4(C, 3) Q_PKL Q_PKH Q_WR0(C, ST) Q_WR1(C, ST)
#define Q_LX8(ST) Q_LX(ST, 0) Q_LX(ST, 1) Q_LX(ST, 2) Q_LX(ST, 3) Q_LX(ST, 4) Q_LX(ST, 5) Q_LX(ST, 6) Q_LX(ST, 7)
#define Q_LW4(ST) Q_LW(ST, 0) Q_LW(ST, 1) Q_LW(ST, 2) Q_LW(ST, 3)
#define Q_RAW4(ST) Q_RAW(0, ST) Q_RAW(1, ST) Q_RAW(2, ST) Q_RAW(3, ST)
#define Q_ACC4(I) [c##I##0] "+a"(c[I][0]), [c##I##1] "+a"(c[I][1]), [c##I##2] "+a"(c[I][2]), [c##I##3] "+a"(c[I][3])
#define Q_CL10(x) "v" #x "0", "v" #x "1", "v" #x "2", "v" #x "3", "v" #x "4", "v" #x "5", "v" #x "6", "v" #x "7",      \
    "v" #x "8", "v" #x "9"

__device__ inline void q8_tile(const GemmArgs &a, unsigned pid, unsigned &m0, unsigned &n0) {
    unsigned tm, tn;
    band_tile((a.m + TM - 1) / TM, (a.n + TN - 1) / TN, GROUP_M, pid, tm, tn);
    m0 = __builtin_amdgcn_readfirstlane(tm * TM);
    n0 = __builtin_amdgcn_readfirstlane(tn * TN);
}

// Weight row of tile row r: SwiGLU alternates 32 gate rows and the 32 up rows of the same
// columns, so that a lane's blocks 2 i and 2 i + 1 hold both.
__device__ inline unsigned weight_row(const GemmArgs &a, unsigned r) {
    return a.gelu == H3_GEMM_SWIGLU ? r / 32 % 2 * (a.n / 2) + r / 64 * 32 + r % 32 : r;
}

// 32 columns of one output row, as BF16 register groups g of lane half hf (columns
// 8 g + 4 hf + 0..3), in 16-byte stores: v_permlane32_swap gives the low half both halves
// of group g, the high half those of group g + 1.
__device__ inline void store32(uint16_t *dst, unsigned hf, const u16x4 *o) {
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
        unsigned w[2][2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            w[h][0] = o[g + h][0] | ((unsigned)o[g + h][1] << 16);
            w[h][1] = o[g + h][2] | ((unsigned)o[g + h][3] << 16);
        }
        const auto s0 = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
        *reinterpret_cast<u32x4 *>(dst + 8 * (g + hf)) = u32x4{s0[0], s1[0], s0[1], s1[1]};
    }
}

// Accumulator blocks 2 ip and 2 ip + 1 (64 columns from col) of one output row.
__device__ inline void q8_store(const GemmArgs &a, unsigned row, unsigned col, unsigned hf, const f32x4 (*c)[4]) {
    u16x4 o[4];
    if (a.gelu == H3_GEMM_SWIGLU) {
        if (col / 2 >= a.n / 2) return;
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                o[g][e] = f32_to_bf16(swiglu_fast(bf16_to_f32(f32_to_bf16(c[0][g][e])), bf16_to_f32(f32_to_bf16(c[1][g][e]))));
        store32(a.y + (size_t)row * (a.n / 2) + col / 2, hf, o);
        return;
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const unsigned first = col + 32 * h;
        if (first >= a.n) return;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            u16x4 bias{};
            if (a.bias) bias = *reinterpret_cast<const u16x4 *>(a.bias + first + 8 * g + 4 * hf);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float v = c[h][g][e];
                if (a.bias) v += bf16_to_f32(bias[e]);
                o[g][e] = f32_to_bf16(v);
                if (a.gelu) o[g][e] = f32_to_bf16(gelu_tanh(bf16_to_f32(o[g][e])));
            }
        }
        store32(a.y + (size_t)row * a.n + first, hf, o);
    }
}

__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(1, 1)))
void gemm_q8_pipe(GemmArgs a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const unsigned tid = threadIdx.x, lane = tid % 64, n32 = lane % 32, hf = lane / 32;
    const unsigned wave = __builtin_amdgcn_readfirstlane(tid / 64), wm = wave / 2, wn = wave % 2;
    unsigned ksteps = a.k / TK;
    const TileShare t = tile_share(a.tile, ksteps);
    const unsigned k0 = t.first * TK;
    unsigned m0, n0;
    q8_tile(a, t.pid, m0, n0);
    const unsigned first = a.gelu == H3_GEMM_SWIGLU ? n0 / 2 : n0;
    const unsigned wrows = a.gelu == H3_GEMM_SWIGLU ? a.n - first : min(a.n - n0, (unsigned)TN);
    const uint64_t xbase = (uint64_t)(a.x + (size_t)m0 * a.k + k0);
    const uint64_t wbase = (uint64_t)((const int8_t *)a.w + (size_t)first * a.k + k0);
    const unsigned xrows = min(a.m - m0, (unsigned)TM);
    // Rows past M or N are past the resources' size and load zeros.
    auto resource = [](uint64_t base, unsigned bytes) {
        return i32x4{(int)__builtin_amdgcn_readfirstlane((unsigned)base),
                     (int)__builtin_amdgcn_readfirstlane((unsigned)(base >> 32)),
                     (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000};
    };
    const i32x4 sx = resource(xbase, (xrows * a.k - k0) * 2), sw = resource(wbase, wrows * a.k - k0);
    // x block wave + 4 t: rows 8 wave + lane / 8 + 32 t, swizzled chunk lane % 8.
    const unsigned lrow = 8 * wave + lane / 8;
    unsigned o[8];
#pragma unroll
    for (int t = 0; t < 8; t++) o[t] = (lrow + 32 * t) * a.k * 2 + swz(lrow, lane % 8) * 16;
    // Code chunk tid + 256 c: row wrow + 64 c, 16-byte part wpart; eight consecutive lanes take
    // rows of one parity, so that their LDS stores hit eight different chunks.
    const unsigned wrow = wave * 16 + 2 * (lane % 8) + lane % 16 / 8, wpart = lane / 16;
    unsigned q[4];
    float scale[4];      // rows past N read the last row's; their codes are zero
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const unsigned r = weight_row(a, wrow + 64 * c);
        q[c] = r * a.k + wpart * 16;
        scale[c] = a.scales[min(first + r, a.n - 1)];
    }
    const unsigned d0 = 2 * TILE + wrow * ROW_BYTES + swz(wrow, 2 * wpart) * 16;
    const unsigned d1 = 2 * TILE + wrow * ROW_BYTES + swz(wrow, 2 * wpart + 1) * 16;
    const unsigned rr = 4 * TILE + tid * 16, mb = __builtin_amdgcn_readfirstlane(wave * 1024);
    unsigned pw[4], px[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const unsigned part = n32 * ROW_BYTES + swz(n32, 2 * s + hf) * 16;
        pw[s] = 2 * TILE + wn * 128 * ROW_BYTES + part;
        px[s] = wm * 128 * ROW_BYTES + part;
    }
    const unsigned last = __builtin_amdgcn_readfirstlane(ksteps - 1);
    const unsigned kxm = last * 128, kwm = last * 64;
    unsigned kx = 0, kw = 0, kxn = 0, kwn = 0, steps = __builtin_amdgcn_readfirstlane(ksteps);
    f32x16 c[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) c[i][j] = f32x16{};
#define Q_NEXT_X "s_min_u32 %[kx], %[kxn], %[kxm]\n s_add_u32 %[kxn], %[kxn], 128\n"
#define Q_NEXT_W "s_min_u32 %[kw], %[kwn], %[kwm]\n s_add_u32 %[kwn], %[kwn], 64\n"
    // Prologue: x of tiles 0 and 1, codes of tiles 0 to 2, tile 0 converted, the
    // codes of tile 1 in registers, substep 0 of tile 0 in set 0. The loop body is two
    // tiles, left after the first where their count is odd; what is loaded or converted past
    // the end is a copy of the last tile that nobody reads.
    asm volatile(
        Q_NEXT_W Q_LW4(0)
        Q_NEXT_X Q_LX8(0)
        Q_NEXT_W Q_LW4(1)
        Q_NEXT_X Q_LX8(1)
        "s_waitcnt vmcnt(0)\n"
        Q_RAW4(0)
        "s_waitcnt lgkmcnt(0)\n"
        Q_CHUNK(0, 0) Q_CHUNK(1, 0) Q_CHUNK(2, 0) Q_CHUNK(3, 0)
        Q_NEXT_W Q_LW4(0)
        "s_waitcnt lgkmcnt(0)\n"
        Q_RAW4(1)
        "s_waitcnt vmcnt(0) lgkmcnt(0)\n"
        "s_barrier\n"
        Q_RW(0, 0, 0, 0) Q_RW(0, 1, 0, 0) Q_RW(0, 2, 0, 0) Q_RW(0, 3, 0, 0)
        Q_RX(0, 0, 0, 0) Q_RX(0, 1, 0, 0) Q_RX(0, 2, 0, 0) Q_RX(0, 3, 0, 0)
        "s_waitcnt lgkmcnt(0)\n"
        "q8_loop_%=:\n"
        Q_TILE(0, 1)
        "s_sub_u32 %[steps], %[steps], 1\n"
        "s_cmp_eq_u32 %[steps], 0\n"
        "s_cbranch_scc1 q8_end_%=\n"
        Q_TILE(1, 0)
        "s_sub_u32 %[steps], %[steps], 1\n"
        "s_cmp_lg_u32 %[steps], 0\n"
        "s_cbranch_scc1 q8_loop_%=\n"
        "q8_end_%=:\n"
        "s_waitcnt vmcnt(0) lgkmcnt(0)\n"
        // The last MFMAs' results are complete before the epilogue reads the accumulators
        // (hipcc does not see the MFMAs inside this block).
        "s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n"
        : Q_ACC4(0), Q_ACC4(1), Q_ACC4(2), Q_ACC4(3), [kx] "+s"(kx), [kw] "+s"(kw), [kxn] "+s"(kxn),
          [kwn] "+s"(kwn), [steps] "+s"(steps)
        : [sx] "s"(sx), [sw] "s"(sw), [o0] "v"(o[0]), [o1] "v"(o[1]), [o2] "v"(o[2]), [o3] "v"(o[3]),
          [o4] "v"(o[4]), [o5] "v"(o[5]), [o6] "v"(o[6]), [o7] "v"(o[7]), [q0] "v"(q[0]), [q1] "v"(q[1]), [q2] "v"(q[2]),
          [q3] "v"(q[3]), [s0] "v"(scale[0]), [s1] "v"(scale[1]), [s2] "v"(scale[2]), [s3] "v"(scale[3]), [d0] "v"(d0), [d1] "v"(d1),
          [rr] "v"(rr), [mb] "s"(mb), [kxm] "s"(kxm), [kwm] "s"(kwm), [w0] "v"(pw[0]),
          [w1] "v"(pw[1]), [w2] "v"(pw[2]), [w3] "v"(pw[3]), [x0] "v"(px[0]), [x1] "v"(px[1]), [x2] "v"(px[2]),
          [x3] "v"(px[3])
        : "v64", "v65", "v66", "v67", "v68", "v69", Q_CL10(7), Q_CL10(8), Q_CL10(9), Q_CL10(10), Q_CL10(11), Q_CL10(12),
          Q_CL10(13), Q_CL10(14), Q_CL10(15), "v160", "v161", "v162", "v163", "v164", "v165", "v166", "v167", "m0", "scc",
          "memory");

    // Block (i, j): lane holds output row m0 + 128 wm + 32 j + n32.
    if (t.partial) {
        f32x4 *dst = reinterpret_cast<f32x4 *>(a.tile.part) +
                     ((size_t)t.tile * a.tile.split + t.share) * (TM * TN / 4) + tid;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (m0 + wm * 128 + j * 32 >= a.m) break;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                hold(c[i][j]);
#pragma unroll
                for (int r = 0; r < 4; r++)
                    dst[((j * 4 + i) * 4 + r) * 256] =
                        f32x4{c[i][j][4 * r], c[i][j][4 * r + 1], c[i][j][4 * r + 2], c[i][j][4 * r + 3]};
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const unsigned row = m0 + wm * 128 + j * 32 + n32;
#pragma unroll
        for (int ip = 0; ip < 2; ip++) {
            f32x4 block[2][4];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                f32x16 &x = c[2 * ip + h][j];
                hold(x);
#pragma unroll
                for (int r = 0; r < 4; r++)
                    block[h][r] = f32x4{x[4 * r], x[4 * r + 1], x[4 * r + 2], x[4 * r + 3]};
            }
            if (row < a.m) q8_store(a, row, n0 + wn * 128 + ip * 64, hf, block);
        }
    }
}

// The split tiles' shares added in order, and the epilogue. One workgroup per (tile, row
// block j, column block pair).
__global__ __launch_bounds__(256) void gemm_q8_reduce(GemmArgs a) {
    const unsigned tile = blockIdx.x / 8, j = blockIdx.x % 8 / 2, ip = blockIdx.x % 2;
    const unsigned tid = threadIdx.x, wave = tid / 64, lane = tid % 64, n32 = lane % 32, hf = lane / 32;
    unsigned m0, n0;
    q8_tile(a, split_tile(a.tile, tile), m0, n0);
    const unsigned row = m0 + wave / 2 * 128 + j * 32 + n32;
    if (row >= a.m) return;
    const f32x4 *src = reinterpret_cast<const f32x4 *>(a.tile.part) + (size_t)tile * a.tile.split * (TM * TN / 4) +
                       (j * 4 + 2 * ip) * 4 * 256 + tid;
    f32x4 block[2][4];
#pragma unroll
    for (int r = 0; r < 8; r++) block[r / 4][r % 4] = src[r * 256];
#pragma unroll 2
    for (unsigned s = 1; s < a.tile.split; s++) {
        src += TM * TN / 4;
#pragma unroll
        for (int r = 0; r < 8; r++) block[r / 4][r % 4] += src[r * 256];
    }
    q8_store(a, row, n0 + wave % 2 * 128 + ip * 64, hf, block);
}

}  // namespace

bool h3_gemm_q8_fits(const GemmArgs &a) {
    // 32-bit offsets inside a tile's rows (SwiGLU: from gate to up rows).
    const size_t reach = a.gelu == H3_GEMM_SWIGLU ? (size_t)a.n : 256;
    return a.k % TK == 0 && a.n % 64 == 0 && a.group == a.k && !a.alpha &&
           reach * a.k < (1ull << 31) && (size_t)256 * a.k * 2 < (1ull << 31);
}

int h3_gemm_q8(h3_gpu *g, GemmArgs a, unsigned split) {
    static bool configured = false;
    if (!configured) {
        if (!h3_hip_check(g, hipFuncSetAttribute((const void *)gemm_q8_pipe, hipFuncAttributeMaxDynamicSharedMemorySize, LDS),
                          "GEMM shared memory"))
            return 0;
        configured = true;
    }
    const unsigned tiles = (a.m + TM - 1) / TM * ((a.n + TN - 1) / TN);
    a.tile = split_last_wave(g, tiles, split, a.k / TK, TM * TN);
    const unsigned rest = tiles - a.tile.full;
    h3_note_kernel(g, "gemm_q8_pipe", 0, a.tile.split);
    hipEvent_t timing = h3_kernel_timing_begin(g);
    hipLaunchKernelGGL(gemm_q8_pipe, dim3(a.tile.full + rest * a.tile.split), dim3(256), LDS, g->compute, a);
    if (rest && h3_launch_status(g, "W8A16 GEMM"))
        hipLaunchKernelGGL(gemm_q8_reduce, dim3(rest * 8), dim3(256), 0, g->compute, a);
    h3_kernel_timing_end(g, timing);
    return h3_launch_status(g, "W8A16 GEMM");
}
