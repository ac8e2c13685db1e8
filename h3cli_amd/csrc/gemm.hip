// Projection GEMMs of the DiT block for gfx950: y[M,N] = x[M,K] . W[N,K]^T (+bias)
// (+GELU-tanh), BF16 activations and output, FP32 accumulation.
//
// Weights are either BF16 (reference h3_gpu_linear_bf16, src/cuda/gpu_cuda.cu:927-1011)
// or W8A16 q8: int8 codes [N,K] with fp32 scales per (row, K-group); the group is
// 64 in the reference q8 recipe (src/weights/q8.c:26-56) or K for one scale per
// output channel. The q8 arithmetic is the reference's Metal kernel
// (src/metal/shaders.metal:799-855): every weight is reconstructed as
// w = bf16(code * scale) and multiplied in FP32 accumulation, bf16 output (+bias).
//
// Kernels, chosen per call (choose(), at the end):
//  * gemm_bf16_pipe, here: a hand-scheduled K loop at one wave per SIMD (see its
//    comment), for many rows. For W8A16 weights a conversion pass first writes
//    w = bf16(code * scale) for the whole weight into a BF16 buffer of the context
//    (in registers, 16 codes per thread), which costs about 1% of the GEMM at
//    M = 32400 and leaves the MFMA loop free of VALU work;
//  * gemm_mid.hip: fewer rows, any N, int8 weights converted in the kernel;
//  * gemm_q8.hip: per-column int8 weights converted in a hand-scheduled loop;
//  * gemm_skinny.hip: at most 16 rows;
//  * gemm_small, here: any shape.
// The tiled kernels compute C^T = W . X^T, so a lane owns one output row and
// consecutive columns, move operands global -> LDS directly (XOR-swizzled 16-byte
// chunks), and remap tile ids so that the workgroups an XCD runs together share
// weight columns in its L2.
#include "common.h"
#include "internal.h"
#include "gemm.h"
#include <cmath>


namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int TM = 256, TN = 256, TK = 64;
constexpr int ROW_BYTES = TK * 2;               // 128 B per BF16 tile row
constexpr int TILE_BYTES = 256 * ROW_BYTES;     // 32 KB per operand tile

// 16-byte chunk swizzle of a 128-byte LDS row. A ds_read_b128 serves sixteen
// lanes (sixteen consecutive rows) per cycle across 256 bytes of banks: rows
// 2i and 2i+1 sit in different halves, and (row >> 1) & 7 spreads the eight
// pairs over eight chunks.
__device__ inline unsigned swz(unsigned row, unsigned ch) { return ch ^ ((row >> 1) & 7); }

// ------------------------------------------------------------ hand-scheduled BF16 GEMM
// gemm_bf16_pipe: a 256 x 256 output tile per workgroup, computed by
// four waves of 128 x 128 (one per SIMD, 2 x 2) on v_mfma_f32_16x16x32_bf16,
// each wave with 8 x 8 accumulator blocks of 16 x 16 in AGPRs, so one
// fragment read from LDS feeds eight MFMAs. (The same loop on 32 x 32 x 16
// MFMAs, 4 x 4 blocks of 16 AGPRs, measured 6% slower on the config-4 shapes.)
// The whole K loop is one inline-asm block, because its value is the order of
// the instructions; with one wave per SIMD nothing else hides a stall:
//  * a K tile (64) is two substeps of 64 MFMAs (32 K each); the 16 fragments
//    of the next substep are read during the first half of the current one,
//    one ds_read_b128 after every second MFMA, into the other register set;
//  * the 16 global -> LDS loads of a K tile (buffer_load ... lds, 1 KB each)
//    are issued two tiles ahead, two per eight MFMAs of the second substep,
//    into the stage this tile has finished reading;
//  * one barrier per tile, between the substeps: every wave has then read
//    all fragments of this tile and its loads of the next tile (issued a
//    tile earlier) have landed; the next tile's first reads follow it.
// LDS (128 KB): X stage 0 at 0, X stage 1 at 32 KB, W stage 0 at 64 KB,
// W stage 1 at 96 KB; rows of 64 BF16 (128 B) with the 16-byte chunk swizzle
// of swz(). Requirements: K % 128 == 0 (tiles come in stage pairs),
// N % 256 == 0, M * K * 2 < 2^31 and N * K * 2 < 2^31 (32-bit offsets).
constexpr int PIPE_LDS = 4 * TILE_BYTES;     // 128 KB
// Tile rows per grouped band of the pipe kernel: an XCD's 32 resident
// workgroups then cover 4 row tiles x 8 column tiles (measured on the config-4
// shapes: 4 and 8 within 1% of each other, 4 ahead; 16 rows 13% slower).
constexpr int PIPE_GROUP_M = 4;

// Load T (0..7) of a K tile's X (PIPE_LD_X) or W (PIPE_LD_W) into stage ST:
// LDS block wave + 4 T (1 KB), rows 8 wave + lane / 8 + 32 T from the lane
// offset o<T>. The offsets are precomputed so that the loop holds no VALU
// instruction besides the MFMAs (with one wave per SIMD each one delays the
// next MFMA); kc is the tile's K byte offset.
#define PIPE_LD_X(ST, T) "s_add_u32 m0, %[mb], 32768*" #ST "+4096*" #T "\n"                                  \
    "buffer_load_dwordx4 %[o" #T "], %[sx], %[kc] offen lds\n"
#define PIPE_LD_W(ST, T) "s_add_u32 m0, %[mb], 65536+32768*" #ST "+4096*" #T "\n"                            \
    "buffer_load_dwordx4 %[w" #T "], %[sw], %[kc] offen lds\n"
#define PIPE_LOADS_X(ST) PIPE_LD_X(ST, 0) PIPE_LD_X(ST, 1) PIPE_LD_X(ST, 2) PIPE_LD_X(ST, 3)                      \
    PIPE_LD_X(ST, 4) PIPE_LD_X(ST, 5) PIPE_LD_X(ST, 6) PIPE_LD_X(ST, 7)
#define PIPE_LOADS_W(ST) PIPE_LD_W(ST, 0) PIPE_LD_W(ST, 1) PIPE_LD_W(ST, 2) PIPE_LD_W(ST, 3)                      \
    PIPE_LD_W(ST, 4) PIPE_LD_W(ST, 5) PIPE_LD_W(ST, 6) PIPE_LD_W(ST, 7)

#define PIPE_X8(ST) PIPE_LD_X(ST, 0), PIPE_LD_X(ST, 1), PIPE_LD_X(ST, 2), PIPE_LD_X(ST, 3), PIPE_LD_X(ST, 4),      \
    PIPE_LD_X(ST, 5), PIPE_LD_X(ST, 6), PIPE_LD_X(ST, 7)
#define PIPE_W8(ST) PIPE_LD_W(ST, 0), PIPE_LD_W(ST, 1), PIPE_LD_W(ST, 2), PIPE_LD_W(ST, 3), PIPE_LD_W(ST, 4),      \
    PIPE_LD_W(ST, 5), PIPE_LD_W(ST, 6), PIPE_LD_W(ST, 7)

// MFMA (i, j) of set S: W block i (16 rows) x X block j.
#define P16_MFMA(S, I, J) "v_mfma_f32_16x16x32_bf16 %[c" #I #J "], %[" #S "w" #I "], %[" #S "x" #J "], %[c" #I #J "]\n"
#define P16_ROW(S, I, E0, E1, E2, E3, E4, E5, E6, E7)                                                        \
    P16_MFMA(S, I, 0) E0 P16_MFMA(S, I, 1) E1 P16_MFMA(S, I, 2) E2 P16_MFMA(S, I, 3) E3                        \
    P16_MFMA(S, I, 4) E4 P16_MFMA(S, I, 5) E5 P16_MFMA(S, I, 6) E6 P16_MFMA(S, I, 7) E7
// Fragment reads of substep KS (0, 1) from stage ST into set T: W block F
// (16 rows) at base pwKS + 2048 F, X block F at pxKS + 2048 F.
#define P16_RW(T, F, KS, ST) "ds_read_b128 %[" #T "w" #F "], %[pw" #KS "] offset:32768*" #ST "+2048*" #F "\n"
#define P16_RX(T, F, KS, ST) "ds_read_b128 %[" #T "x" #F "], %[px" #KS "] offset:32768*" #ST "+2048*" #F "\n"
// A substep of set S; rows 0..3 read the 16 fragments of substep KS / stage
// ST into set T at their even slots; L0..L15 go to the odd slots 1 and 5 of
// rows 0..7.
#define P16_SUB(S, T, KS, ST, L0, L1, L2, L3, L4, L5, L6, L7, L8, L9, L10, L11, L12, L13, L14, L15)            \
    P16_ROW(S, 0, P16_RW(T, 0, KS, ST), L0, P16_RW(T, 1, KS, ST), "", P16_RW(T, 2, KS, ST), L1,                \
            P16_RW(T, 3, KS, ST), "")                                                                        \
    P16_ROW(S, 1, P16_RW(T, 4, KS, ST), L2, P16_RW(T, 5, KS, ST), "", P16_RW(T, 6, KS, ST), L3,                \
            P16_RW(T, 7, KS, ST), "")                                                                        \
    P16_ROW(S, 2, P16_RX(T, 0, KS, ST), L4, P16_RX(T, 1, KS, ST), "", P16_RX(T, 2, KS, ST), L5,                \
            P16_RX(T, 3, KS, ST), "")                                                                        \
    P16_ROW(S, 3, P16_RX(T, 4, KS, ST), L6, P16_RX(T, 5, KS, ST), "", P16_RX(T, 6, KS, ST), L7,                \
            P16_RX(T, 7, KS, ST), "")                                                                        \
    P16_ROW(S, 4, "", L8, "", "", "", L9, "", "")                                                             \
    P16_ROW(S, 5, "", L10, "", "", "", L11, "", "")                                                           \
    P16_ROW(S, 6, "", L12, "", "", "", L13, "", "")                                                           \
    P16_ROW(S, 7, "", L14, "", "", "", L15, "", "")
#define P16_SUB_EXP(...) P16_SUB(__VA_ARGS__)
#define P16_NONE "", "", "", "", "", "", "", "", "", "", "", "", "", "", "", ""
// One K tile in stage ST: substep 0 (set a) reads substep 1 of this tile
// into set b; the barrier; substep 1 (set b) reads substep 0 of the next tile
// (stage OT) into set a and loads the tile two ahead into ST.
#define P16_TILE(ST, OT)                                                                                      \
    P16_SUB_EXP(a, b, 1, ST, P16_NONE)                                                                        \
    "s_waitcnt vmcnt(0) lgkmcnt(0)\n"                                                                         \
    "s_barrier\n"                                                                                             \
    "s_min_u32 %[kc], %[kn], %[kmax]\n"                                                                       \
    "s_add_u32 %[kn], %[kn], 128\n"                                                                           \
    P16_SUB_EXP(b, a, 0, OT, PIPE_X8(ST), PIPE_W8(ST))                                                        \
    "s_waitcnt lgkmcnt(0)\n"

#define P16_ACC8(I) [c##I##0] "+a"(c[I][0]), [c##I##1] "+a"(c[I][1]), [c##I##2] "+a"(c[I][2]),               \
    [c##I##3] "+a"(c[I][3]), [c##I##4] "+a"(c[I][4]), [c##I##5] "+a"(c[I][5]), [c##I##6] "+a"(c[I][6]),      \
    [c##I##7] "+a"(c[I][7])
#define P16_SET(S) [S##w0] "=&v"(S##f[0]), [S##w1] "=&v"(S##f[1]), [S##w2] "=&v"(S##f[2]),                    \
    [S##w3] "=&v"(S##f[3]), [S##w4] "=&v"(S##f[4]), [S##w5] "=&v"(S##f[5]), [S##w6] "=&v"(S##f[6]),          \
    [S##w7] "=&v"(S##f[7]), [S##x0] "=&v"(S##f[8]), [S##x1] "=&v"(S##f[9]), [S##x2] "=&v"(S##f[10]),          \
    [S##x3] "=&v"(S##f[11]), [S##x4] "=&v"(S##f[12]), [S##x5] "=&v"(S##f[13]), [S##x6] "=&v"(S##f[14]),      \
    [S##x7] "=&v"(S##f[15])

// First row and column of output tile pid: bands of PIPE_GROUP_M row tiles sweep
// the columns together.
__device__ inline void pipe_tile(const GemmArgs &a, unsigned pid, unsigned &m0, unsigned &n0) {
    // A last band of fewer rows, not even bands: 8193 rows, 5376 -> 28672 -> 5376 (33 row
    // tiles) 2.87 ms against 2.93 in nine bands of three or four.
    const unsigned tiles_m = (a.m + TM - 1) / TM, tiles_n = a.n / TN;
    const unsigned band = pid / (PIPE_GROUP_M * tiles_n), first_m = band * PIPE_GROUP_M;
    const unsigned rows_in_band = min(tiles_m - first_m, (unsigned)PIPE_GROUP_M);
    const unsigned tm = first_m + (pid % (PIPE_GROUP_M * tiles_n)) % rows_in_band;
    const unsigned tn = (pid % (PIPE_GROUP_M * tiles_n)) / rows_in_band;
    m0 = __builtin_amdgcn_readfirstlane(tm * TM);
    n0 = __builtin_amdgcn_readfirstlane(tn * TN);
}

// Output row `row`, columns col0 .. col0 + 127 of a wave: accumulator block i of
// a lane holds columns col0 + 16 i + 4 q4 + 0..3. Blocks i and i + 1 go out
// together as 16-byte stores: v_permlane16_swap hands the odd lane rows' block-i
// values to the even rows and the even rows' block-(i+1) values to the odd rows,
// so each lane holds eight consecutive columns.
template <int EPI>
__device__ inline void pipe_store(const GemmArgs &a, unsigned row, unsigned col0, unsigned q4, const f32x4 *c) {
    if constexpr (EPI & 8) {
        // Blocks 2 i and 2 i + 1 are gate and up of output columns col0 / 2 + 16 i + 4 q4
        // + 0..3: both rounded to BF16, as the separate SwiGLU reads them.
        uint16_t *dst = a.y + (size_t)row * (a.n / 2);
#pragma unroll
        for (int ip = 0; ip < 2; ip++) {
            unsigned w[2][2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                u16x4 out;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    out[e] = f32_to_bf16(swiglu_fast(bf16_to_f32(f32_to_bf16(c[4 * ip + 2 * h][e])),
                                                     bf16_to_f32(f32_to_bf16(c[4 * ip + 2 * h + 1][e]))));
                w[h][0] = out[0] | ((unsigned)out[1] << 16);
                w[h][1] = out[2] | ((unsigned)out[3] << 16);
            }
            const auto s0 = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
            const auto s1 = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
            const unsigned col = col0 / 2 + 32 * ip + ((q4 & 1) ? 16 + 4 * (q4 - 1) : 4 * q4);
            u32x4 v = {s0[0], s1[0], s0[1], s1[1]};
            *reinterpret_cast<u32x4 *>(dst + col) = v;
        }
        return;
    }
    uint16_t *dst = a.y + (size_t)row * a.n;
#pragma unroll
    for (int ip = 0; ip < 4; ip++) {
        unsigned w[2][2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int i = 2 * ip + h;
            const unsigned col = col0 + i * 16 + 4 * q4;
            u16x4 out;
            u16x4 bias4 = {};
            if constexpr (EPI & 1) bias4 = *reinterpret_cast<const u16x4 *>(a.bias + col);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float x = c[i][e];
                if constexpr (EPI & 4) x *= a.alpha[0];
                if constexpr (EPI & 1) x += bf16_to_f32(bias4[e]);
                uint16_t b = f32_to_bf16(x);
                if constexpr (EPI & 2) b = f32_to_bf16(gelu_tanh(bf16_to_f32(b)));
                out[e] = b;
            }
            w[h][0] = out[0] | ((unsigned)out[1] << 16);
            w[h][1] = out[2] | ((unsigned)out[3] << 16);
        }
        const auto s0 = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
        const auto s1 = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
        const unsigned col = col0 + 2 * ip * 16 + ((q4 & 1) ? 16 + 4 * (q4 - 1) : 4 * q4);
        u32x4 v = {s0[0], s1[0], s0[1], s1[1]};
        *reinterpret_cast<u32x4 *>(dst + col) = v;
    }
}

// SPLIT: the launch has split tiles (compiled out of the others, where the extra
// prologue and epilogue code cost 1%: 32400 rows, 5120 -> 13824 + GELU, 3.38 against
// 3.42 ms).
template <int EPI, bool SPLIT>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(1, 1)))
void gemm_bf16_pipe(GemmArgs a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const unsigned tid = threadIdx.x, lane = tid % 64, n16 = lane % 16, q4 = lane / 16;
    const unsigned wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const unsigned wm = wave / 2, wn = wave % 2;
    // K units: stage pairs.
    unsigned units = a.k / (2 * TK);
    TileShare t{};
    if constexpr (SPLIT) t = tile_share(a.tile, units);
    else t.pid = xcd_remap(blockIdx.x, gridDim.x);
    const unsigned k0 = t.first * 2 * TK, ksteps = units * 2;
    unsigned m0, n0;
    pipe_tile(a, t.pid, m0, n0);

    const uint64_t xbase = (uint64_t)(a.x + (size_t)m0 * a.k + k0);
    const unsigned wrow = EPI & 8 ? n0 / 2 : n0, wrows = EPI & 8 ? a.n / 2 + TN / 2 : TN;
    const uint64_t wbase = (uint64_t)((const uint16_t *)a.w + (size_t)wrow * a.k + k0);
    const unsigned xrows = min(a.m - m0, (unsigned)TM);
    const i32x4 sx = {(int)__builtin_amdgcn_readfirstlane((unsigned)xbase),
                      (int)__builtin_amdgcn_readfirstlane((unsigned)(xbase >> 32)),
                      (int)__builtin_amdgcn_readfirstlane((xrows * a.k - k0) * 2), 0x00020000};
    const i32x4 sw = {(int)__builtin_amdgcn_readfirstlane((unsigned)wbase),
                      (int)__builtin_amdgcn_readfirstlane((unsigned)(wbase >> 32)),
                      (int)__builtin_amdgcn_readfirstlane((wrows * a.k - k0) * 2), 0x00020000};
    const unsigned lrow = 8 * wave + lane / 8;
    // X and W tiles share the lane offsets: row lrow + 32 t, swizzled chunk.
    unsigned o[8];
#pragma unroll
    for (int t = 0; t < 8; t++) o[t] = (lrow + 32 * t) * a.k * 2 + swz(lrow, lane % 8) * 16;
    // SwiGLU: weight row 16 b + r of the tile (b < 16) is gate (b even) or up (b odd)
    // row n0 / 2 + 16 (b / 2) + r, so that a lane's accumulator blocks 2 i and 2 i + 1
    // hold both for the same columns.
    unsigned ow[8];
#pragma unroll
    for (int t = 0; t < 8; t++)
        ow[t] = EPI & 8 ? (lrow / 16 * (a.n / 2) + 16 * t + lrow % 16) * a.k * 2 + swz(lrow, lane % 8) * 16 : o[t];
    const unsigned mb = __builtin_amdgcn_readfirstlane(wave * 1024);
    unsigned kn = 2 * TK * 2, kc = 0;
    const unsigned kmax = __builtin_amdgcn_readfirstlane((ksteps - 1) * TK * 2);
    unsigned pairs = __builtin_amdgcn_readfirstlane(ksteps / 2);
    // Fragment bases of substep ks (32 K) in stage 0: row n16 of the wave's
    // 128-row half, logical chunk 4 ks + q4.
    unsigned pw[2], px[2];
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        const unsigned part = n16 * ROW_BYTES + swz(n16, 4 * ks + q4) * 16;
        pw[ks] = 2 * TILE_BYTES + wn * 128 * ROW_BYTES + part;
        px[ks] = wm * 128 * ROW_BYTES + part;
    }
    f32x4 c[8][8];
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) c[i][j] = f32x4{};
    bf16x8 af[16], bf[16];
    // Prologue: tiles 0 and 1 into stages 0 and 1, substep 0 of tile 0 into
    // set a. Then the tiles in stage pairs; the last pair's loads are clamped
    // reloads of the last tile into a stage nobody reads again, and its
    // closing reads land in registers nobody uses.
    asm volatile(
        "s_mov_b32 %[kc], 0\n" PIPE_LOADS_X(0) PIPE_LOADS_W(0)
        "s_mov_b32 %[kc], 128\n" PIPE_LOADS_X(1) PIPE_LOADS_W(1)
        "s_waitcnt vmcnt(0)\n"
        "s_barrier\n"
        P16_RW(a, 0, 0, 0) P16_RW(a, 1, 0, 0) P16_RW(a, 2, 0, 0) P16_RW(a, 3, 0, 0)
        P16_RW(a, 4, 0, 0) P16_RW(a, 5, 0, 0) P16_RW(a, 6, 0, 0) P16_RW(a, 7, 0, 0)
        P16_RX(a, 0, 0, 0) P16_RX(a, 1, 0, 0) P16_RX(a, 2, 0, 0) P16_RX(a, 3, 0, 0)
        P16_RX(a, 4, 0, 0) P16_RX(a, 5, 0, 0) P16_RX(a, 6, 0, 0) P16_RX(a, 7, 0, 0)
        "s_waitcnt lgkmcnt(0)\n"
        "p16_loop_%=:\n"
        P16_TILE(0, 1)
        P16_TILE(1, 0)
        "s_sub_u32 %[pairs], %[pairs], 1\n"
        "s_cmp_lg_u32 %[pairs], 0\n"
        "s_cbranch_scc1 p16_loop_%=\n"
        "s_waitcnt vmcnt(0) lgkmcnt(0)\n"
        // The last MFMAs' results are complete before the epilogue reads the
        // accumulators (hipcc does not see the MFMAs inside this block).
        "s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n"
        : P16_ACC8(0), P16_ACC8(1), P16_ACC8(2), P16_ACC8(3), P16_ACC8(4), P16_ACC8(5), P16_ACC8(6), P16_ACC8(7),
          P16_SET(a), P16_SET(b),
          [kc] "+s"(kc), [kn] "+s"(kn), [pairs] "+s"(pairs)
        : [sx] "s"(sx), [sw] "s"(sw), [o0] "v"(o[0]), [o1] "v"(o[1]), [o2] "v"(o[2]), [o3] "v"(o[3]),
          [o4] "v"(o[4]), [o5] "v"(o[5]), [o6] "v"(o[6]), [o7] "v"(o[7]), [w0] "v"(ow[0]), [w1] "v"(ow[1]),
          [w2] "v"(ow[2]), [w3] "v"(ow[3]), [w4] "v"(ow[4]), [w5] "v"(ow[5]), [w6] "v"(ow[6]), [w7] "v"(ow[7]),
          [mb] "s"(mb), [kmax] "s"(kmax), [pw0] "v"(pw[0]), [pw1] "v"(pw[1]), [px0] "v"(px[0]), [px1] "v"(px[1])
        : "m0", "scc", "memory");

    if (SPLIT && t.partial) {
        // Partial sums of (split tile, share): element (i, j) of thread t at
        // ((8 j + i) * 256 + t), so that every store instruction is contiguous.
        f32x4 *dst = reinterpret_cast<f32x4 *>(a.tile.part) +
                     ((size_t)t.tile * a.tile.split + t.share) * (TM * TN / 4) + tid;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (m0 + wm * 128 + j * 16 >= a.m) break;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                hold(c[i][j]);
                dst[(8 * j + i) * 256] = c[i][j];
            }
        }
        return;
    }
    // Block (i, j): lane holds output row m0 + wm*128 + j*16 + n16 and columns
    // n0 + wn*128 + i*16 + 4*q4 + 0..3.
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const unsigned row = m0 + wm * 128 + j * 16 + n16;
        if (row >= a.m) continue;
        f32x4 block[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            hold(c[i][j]);
            block[i] = c[i][j];
        }
        pipe_store<EPI>(a, row, n0 + wn * 128, q4, block);
    }
}

// The split tiles' shares added in order, and the pipe kernel's epilogue. One
// workgroup per (tile, accumulator row j); HBM-bound.
template <int EPI>
__global__ __launch_bounds__(256) void gemm_pipe_reduce(GemmArgs a) {
    const unsigned tile = blockIdx.x / 8, j = blockIdx.x % 8, tid = threadIdx.x;
    const unsigned lane = tid % 64, wave = tid / 64, n16 = lane % 16, q4 = lane / 16;
    unsigned m0, n0;
    pipe_tile(a, split_tile(a.tile, tile), m0, n0);
    const unsigned row = m0 + (wave / 2) * 128 + j * 16 + n16;
    if (row >= a.m) return;
    const f32x4 *src = reinterpret_cast<const f32x4 *>(a.tile.part) + (size_t)tile * a.tile.split * (TM * TN / 4) + 8 * j * 256 + tid;
    f32x4 block[8];
#pragma unroll
    for (int i = 0; i < 8; i++) block[i] = src[i * 256];
#pragma unroll 4
    for (unsigned s = 1; s < a.tile.split; s++) {
        src += TM * TN / 4;
#pragma unroll
        for (int i = 0; i < 8; i++) block[i] += src[i * 256];
    }
    pipe_store<EPI>(a, row, n0 + (wave % 2) * 128, q4, block);
}

template <int EPI>
int launch_pipe(h3_gpu *g, GemmArgs a, unsigned split, bool timed) {
    constexpr size_t shared = PIPE_LDS;
    static bool configured = false;
    if (!configured) {
        for (const void *kernel : {(const void *)gemm_bf16_pipe<EPI, false>, (const void *)gemm_bf16_pipe<EPI, true>})
            if (!h3_hip_check(g, hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shared),
                              "GEMM shared memory"))
                return 0;
        configured = true;
    }
    const unsigned tiles = (a.m + TM - 1) / TM * (a.n / TN);
    a.tile = split_last_wave(g, tiles, split, a.k / (2 * TK), TM * TN);
    const unsigned rest = tiles - a.tile.full;
    h3_note_kernel(g, "gemm_bf16_pipe", 0, a.tile.split);
    hipEvent_t timing = timed ? h3_kernel_timing_begin(g) : nullptr;
    if (!rest) {
        hipLaunchKernelGGL((gemm_bf16_pipe<EPI, false>), dim3(tiles), dim3(256), shared, g->compute, a);
    } else {
        hipLaunchKernelGGL((gemm_bf16_pipe<EPI, true>), dim3(a.tile.full + rest * a.tile.split), dim3(256), shared, g->compute, a);
        if (h3_launch_status(g, "BF16 GEMM"))
            hipLaunchKernelGGL(gemm_pipe_reduce<EPI>, dim3(rest * 8), dim3(256), 0, g->compute, a);
    }
    h3_kernel_timing_end(g, timing);
    return h3_launch_status(g, "BF16 GEMM");
}

bool pipe_fits(const GemmArgs &a) {
    return a.n % TN == 0 && a.k % (2 * TK) == 0 && a.m >= 32 && (size_t)a.m * a.k * 2 < (1ull << 31) &&
           (size_t)a.n * a.k * 2 < (1ull << 31);
}
// epi: bit 0 bias, 1 GELU, 2 alpha, 3 SwiGLU.
int launch_pipe_epi(h3_gpu *g, const GemmArgs &a, int epi, unsigned split, bool timed) {
    switch (epi) {
    case 0: return launch_pipe<0>(g, a, split, timed);
    case 1: return launch_pipe<1>(g, a, split, timed);
    case 2: return launch_pipe<2>(g, a, split, timed);
    case 3: return launch_pipe<3>(g, a, split, timed);
    case 8: return launch_pipe<8>(g, a, split, timed);
    default: return launch_pipe<4>(g, a, split, timed);
    }
}

// W8A16 weights -> BF16 values w = bf16(code * scale[row, k / group]), the
// reconstruction of gemm_mid and of the reference's Metal kernel
// (shaders.metal:825-827), written once per projection call for
// gemm_bf16_pipe. HBM-bound: each thread reads 16 codes (one 16-byte load)
// and writes 32 bytes. group is a multiple of 16, so one scale covers them.
__global__ __launch_bounds__(256) void q8_dequant_bf16(const int8_t *codes, const float *scales, uint16_t *out,
                                                     unsigned k, unsigned group, unsigned groups, size_t chunks) {
    const size_t c = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= chunks) return;
    const size_t first = c * 16;
    const unsigned row = (unsigned)(first / k), col = (unsigned)(first % k);
    const float s = scales[(size_t)row * groups + col / group];
    const i32x4 q = *reinterpret_cast<const i32x4 *>(codes + first);
    bf16x8 half[2];
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        const int word = q[e / 4];
        f32x2 f = {(float)(int8_t)(word >> (8 * (e % 4))) * s, (float)(int8_t)(word >> (8 * (e % 4 + 1))) * s};
        bf16x2 b = __builtin_convertvector(f, bf16x2);
        half[e / 8][e % 8] = b[0];
        half[e / 8][e % 8 + 1] = b[1];
    }
    *reinterpret_cast<bf16x8 *>(out + first) = half[0];
    *reinterpret_cast<bf16x8 *>(out + first + 8) = half[1];
}

// Any-shape fallback (short sums of few rows, unaligned projections): one lane per
// column, FP32 accumulation in k order. Same weight reconstruction as the tiled
// kernel. A workgroup of 64 columns and 4 * SMALL_R rows stages SMALL_K values of
// its weight rows in LDS as BF16 (16-byte loads where K and the rows allow them:
// VEC), so that memory is read in whole lines; the lane rows are padded by 16 bytes,
// which spreads a wave's 16-byte LDS reads over all banks. Bound by the FMA chain
// and the LDS latency in it. Measured (one thread per output with strided two-byte
// loads before): 2 rows, 256 -> 5376: 8.3 us (58); 31 rows, int8: 17 us (214).
constexpr unsigned SMALL_K = 128, SMALL_R = 4, SMALL_ROW = SMALL_K * 2 + 16;

template <bool Q8, bool VEC>
__global__ __launch_bounds__(256) void gemm_small(GemmArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t ws[64 * SMALL_ROW];
    __shared__ __attribute__((aligned(16))) float xs[4 * SMALL_R][SMALL_K];
    const unsigned tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const unsigned row_blocks = (a.m + 4 * SMALL_R - 1) / (4 * SMALL_R);
    const unsigned n0 = blockIdx.x / row_blocks * 64, m0 = blockIdx.x % row_blocks * 4 * SMALL_R, col = n0 + lane;
    float acc[SMALL_R] = {};
    for (unsigned k0 = 0; k0 < a.k; k0 += SMALL_K) {
        const unsigned kn = min(SMALL_K, a.k - k0);
        __syncthreads();
        if constexpr (VEC) {
            // 8 values per chunk, 16 chunks per row.
            for (unsigned c = tid; c < 64 * SMALL_K / 8; c += 256) {
                const unsigned r = c / (SMALL_K / 8), at = c % (SMALL_K / 8) * 8;
                const size_t row = min(n0 + r, a.n - 1);
                if (at >= kn) continue;
                bf16x8 v;
                if constexpr (Q8) {
                    const i32x2 q = *reinterpret_cast<const i32x2 *>((const int8_t *)a.w + row * a.k + k0 + at);
                    const float sc = a.scales[row * a.groups + (k0 + at) / a.group];
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] = (__bf16)((float)(int8_t)(q[e / 4] >> (8 * (e % 4))) * sc);
                } else {
                    v = *reinterpret_cast<const bf16x8 *>((const uint16_t *)a.w + row * a.k + k0 + at);
                }
                *reinterpret_cast<bf16x8 *>(ws + r * SMALL_ROW + at * 2) = v;
            }
        } else {
            for (unsigned c = tid; c < 64 * SMALL_K; c += 256) {
                const unsigned r = c / SMALL_K, at = c % SMALL_K;
                const size_t row = min(n0 + r, a.n - 1);
                if (at >= kn) continue;
                uint16_t v;
                if constexpr (Q8)
                    v = f32_to_bf16((float)((const int8_t *)a.w)[row * a.k + k0 + at] *
                                    a.scales[row * a.groups + (k0 + at) / a.group]);
                else
                    v = ((const uint16_t *)a.w)[row * a.k + k0 + at];
                *reinterpret_cast<uint16_t *>(ws + r * SMALL_ROW + at * 2) = v;
            }
        }
        for (unsigned c = tid; c < 4 * SMALL_R * SMALL_K; c += 256) {
            const unsigned r = c / SMALL_K, at = c % SMALL_K;
            if (at < kn && m0 + r < a.m) xs[r][at] = bf16_to_f32(a.x[(size_t)(m0 + r) * a.k + k0 + at]);
        }
        __syncthreads();
        // Rows past M read what LDS holds; they are not stored.
        const uint8_t *wr = ws + lane * SMALL_ROW;
        unsigned kk = 0;
        for (; kk + 8 <= kn; kk += 8) {
            const u16x8 w = *reinterpret_cast<const u16x8 *>(wr + kk * 2);
#pragma unroll
            for (unsigned r = 0; r < SMALL_R; r++) {
                if (m0 + wave + 4 * r >= a.m) break;
                const float *x = xs[wave + 4 * r] + kk;
#pragma unroll
                for (int e = 0; e < 8; e++) acc[r] = fmaf(x[e], bf16_to_f32(w[e]), acc[r]);
            }
        }
        for (; kk < kn; kk++) {
            const float w = bf16_to_f32(*reinterpret_cast<const uint16_t *>(wr + kk * 2));
#pragma unroll
            for (unsigned r = 0; r < SMALL_R; r++) acc[r] = fmaf(xs[wave + 4 * r][kk], w, acc[r]);
        }
    }
    if (col >= a.n) return;
#pragma unroll
    for (unsigned r = 0; r < SMALL_R; r++) {
        const unsigned row = m0 + wave + 4 * r;
        if (row >= a.m) return;
        float v = acc[r];
        if (a.alpha) v *= a.alpha[0];
        if (a.bias) v += bf16_to_f32(a.bias[col]);
        uint16_t b = f32_to_bf16(v);
        if (a.gelu) b = f32_to_bf16(gelu_tanh(bf16_to_f32(b)));
        a.y[(size_t)row * a.n + col] = b;
    }
}

int launch_small(h3_gpu *g, const GemmArgs &a, bool q8) {
    const bool vec = a.k % 8 == 0 && (!q8 || a.group % 8 == 0);
    h3_note_kernel(g, "gemm_small");
    // One grid dimension, rows first: the others end at 65535 blocks (4.19 million columns).
    const dim3 grid((a.m + 4 * SMALL_R - 1) / (4 * SMALL_R) * ((a.n + 63) / 64));
    if (q8 && vec) hipLaunchKernelGGL((gemm_small<true, true>), grid, dim3(256), 0, g->compute, a);
    else if (q8) hipLaunchKernelGGL((gemm_small<true, false>), grid, dim3(256), 0, g->compute, a);
    else if (vec) hipLaunchKernelGGL((gemm_small<false, true>), grid, dim3(256), 0, g->compute, a);
    else hipLaunchKernelGGL((gemm_small<false, false>), grid, dim3(256), 0, g->compute, a);
    return h3_launch_status(g, "small GEMM");
}

// ------------------------------------------------------------ choice of the kernel
// The fastest of the kernels that take this projection, by gemm_last_wave with rates fitted
// to the measured times of all plans of eight projections (K, N 5120 to 28672) of 33 to 24000
// rows and of ten narrow or short ones (K 256 to 5376, N 64 to 5376) of 33 to 24000 rows: BF16,
// int8 with one scale per column and int8 of group 64. The plan taken is 0.5% (narrow: 1.6%)
// slower than the best one in the mean, and never 2% slower than whole tiles of the pipe
// kernel for the wide ones. Converting a weight to BF16 first takes 0.4 to 1.2 us per million
// values, most for a long K, whose rows share the cache with the weight. What is not the pipe
// kernel on whole tiles must promise 2%. Measured, in microseconds, the runner-up in brackets:
// 729 rows, 7168 -> 5376, BF16: pipe in 4 shares 61 (whole 113); 729 rows, 5376 -> 28672, int8
// of group 64: mid 256 in 3 shares 260 (pipe in 3 281), per column: q8 in 3 shares 213 (mid
// 240); 729 rows, 5120 -> 13824, group 64: pipe 122 (mid 151); 1800 rows, 14336 -> 5376, per
// column: q8 292 (pipe 315); 64 rows, 5376 -> 28672, BF16: mid 64 in 2 shares 61 (pipe 114); 256
// rows, 5376 -> 64, BF16: mid 64 in 10 shares 12.5 (mid 128 in 16 14.7).
GemmPlan choose(const h3_gpu *g, const GemmArgs &a, bool q8, bool may_convert) {
    static constexpr GemmRates PIPE{2.68f, 1.93f, 1.61f, .58f, 8.7f, .048f, .33f};       // per 128 values of K
    static constexpr GemmRates CODES{1.55f, 1.1f, .93f, .51f, 15.9f, .018f, .83f};       // gemm_q8; per 64, as all below
    static constexpr GemmRates MID_BF16[3] = {{.6f, .41f, .19f, .15f, 5.5f, .104f, .16f},
                                              {.9f, .68f, .48f, .6f, 7.f, .088f, .09f},
                                              {1.73f, 1.02f, .61f, .15f, 7.9f, .06f, .02f}};
    static constexpr GemmRates MID_COLUMN[3] = {{.85f, .72f, .06f, .15f, 7.2f, .113f, .15f},
                                                {1.08f, .95f, .05f, .15f, 8.4f, .094f, .09f},
                                                {1.82f, 1.4f, .46f, .15f, 11.5f, .06f, .02f}};
    static constexpr GemmRates MID_GROUP[3] = {{1.07f, .91f, .11f, .15f, 7.3f, .108f, .15f},
                                               {1.23f, 1.06f, .18f, .15f, 8.3f, .091f, .09f},
                                               {1.91f, 1.48f, .45f, .15f, 11.5f, .059f, .03f}};
    GemmPlan best{3.4e38f, 0, 1, false};
    const float convert = q8 ? (float)a.n * a.k * (.4e-6f + 3e-11f * a.k) + 3.f : 0.f;
    auto consider = [&](GemmPlan p, unsigned tm, bool dequant) {
        p.tm = tm;
        p.dequant = dequant;
        if (dequant) p.us += convert;
        if (tm || p.split > 1) p.us *= 1.02f;
        if (p.us < best.us) best = p;
    };
    auto tiles = [&](unsigned rows) { return (a.m + rows - 1) / rows * ((a.n + TN - 1) / TN); };
    const bool pipe = pipe_fits(a);
    if (pipe && (!q8 || may_convert)) consider(gemm_last_wave(g, tiles(TM), a.k / (2 * TK), PIPE), 0, q8);
    if (q8 && h3_gemm_q8_fits(a)) consider(gemm_last_wave(g, tiles(TM), a.k / TK, CODES), GEMM_Q8, false);
    if (h3_gemm_mid_fits(a, q8))
        for (unsigned i = 0; i < 3; i++) {
            const unsigned tm = 64u << i;
            const GemmRates &codes = a.group == a.k ? MID_COLUMN[i] : MID_GROUP[i];
            if (q8) consider(gemm_last_wave(g, tiles(tm), a.k / TK, codes, tm / 256.f), tm, false);
            if ((i < 2 || !pipe) && (!q8 || may_convert))
                consider(gemm_last_wave(g, tiles(tm), a.k / TK, MID_BF16[i], tm / 256.f), tm, q8);
        }
    return best;
}

// Runs a projection that pipe or mid takes. Both kernels of a converted projection are
// inside one kernel-timing window.
int run(h3_gpu *g, const GemmArgs &a, bool q8, int epi) {
    // The context keeps the converted weight: none of 2 GiB or more, which the pipe kernel's
    // 32-bit offsets do not take either.
    const size_t weights = (size_t)a.n * a.k;
    GemmPlan p = choose(g, a, q8, weights * 2 < (1ull << 31));
    // No room for the converted weight: a kernel that reads the codes (gemm_mid takes all).
    if (p.dequant && !h3_buffer_try(g, &g->gemm_weights, weights * 2)) p = choose(g, a, q8, false);
    if (p.tm == GEMM_Q8) return h3_gemm_q8(g, a, p.split);
    if (!p.dequant) return p.tm ? h3_gemm_mid(g, a, q8, p.tm, p.split) : launch_pipe_epi(g, a, epi, p.split, true);
    const size_t chunks = weights / 16;
    hipEvent_t timing = h3_kernel_timing_begin(g);
    hipLaunchKernelGGL(q8_dequant_bf16, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, g->compute,
                       (const int8_t *)a.w, a.scales, (uint16_t *)g->gemm_weights.ptr, a.k, a.group, a.groups, chunks);
    GemmArgs b = a;
    b.w = g->gemm_weights.ptr;
    const int ok = h3_launch_status(g, "W8A16 dequantization") &&
                   (p.tm ? h3_gemm_mid(g, b, false, p.tm, p.split, false) : launch_pipe_epi(g, b, epi, p.split, false));
    h3_kernel_timing_end(g, timing);
    g->last.converted = true;
    return ok;
}

bool tiled(const GemmArgs &a, bool q8) {
    return !(a.m < 32 && a.k <= H3_GEMM_SHORT_K) && h3_gemm_mid_fits(a, q8);
}

}  // namespace

// y[M,N] = bf16(alpha[0] * x[M,K] . w[N,K]^T) with BF16 device operands and a
// device scalar alpha (the NVFP4 projections' dequantized operands).
int h3_gemm_bf16_alpha(h3_gpu *g, uint16_t *y, const uint16_t *x, const uint16_t *w, const float *alpha, uint32_t m,
                       uint32_t k, uint32_t n) {
    GemmArgs a{};
    a.y = y; a.x = x; a.w = w; a.alpha = alpha; a.m = m; a.n = n; a.k = k; a.group = 1; a.groups = 1;
    if (h3_gemm_skinny_fits(a, false)) return h3_gemm_skinny(g, a, false);
    return tiled(a, false) ? run(g, a, false, 4) : launch_small(g, a, false);
}

static GemmArgs gemm_args(uint16_t *y, const uint16_t *x, const h3_gpu_tensor *w, const uint16_t *bias, uint32_t m,
                          uint32_t k, uint32_t n, int activation) {
    GemmArgs a{};
    a.y = y; a.x = x; a.w = w->data; a.bias = bias; a.m = m; a.n = n; a.k = k; a.gelu = activation;
    a.scales = w->q8 ? w->q8_scales : nullptr;
    a.group = w->q8 ? w->q8_group : 1;
    a.groups = w->q8 ? (k + a.group - 1) / a.group : 1;
    return a;
}

bool h3_gemm_swiglu_fits(const h3_gpu_tensor *w, uint32_t m, uint32_t k, uint32_t hidden) {
    if (hidden > UINT32_MAX / 2) return false;
    const GemmArgs a = gemm_args(nullptr, nullptr, w, nullptr, m, k, 2 * hidden, H3_GEMM_SWIGLU);
    return !h3_gemm_skinny_fits(a, w->q8 != 0) && tiled(a, w->q8 != 0);
}

int h3_gemm(h3_gpu *g, uint16_t *y, const uint16_t *x, const h3_gpu_tensor *w, const uint16_t *bias, uint32_t m,
            uint32_t k, uint32_t n, int activation) {
    const bool q8 = w->q8 != 0;
    const GemmArgs a = gemm_args(y, x, w, bias, m, k, n, activation);
    if (!h3_tensor_acquire(g, w)) return 0;
    const int epi = (bias ? 1 : 0) | (activation == H3_GEMM_GELU ? 2 : 0) | (activation == H3_GEMM_SWIGLU ? 8 : 0);
    const int ok = h3_gemm_skinny_fits(a, q8) ? h3_gemm_skinny(g, a, q8)
                   : tiled(a, q8)             ? run(g, a, q8, epi)
                                              : launch_small(g, a, q8);
    if (ok) {
        g->stats.linear_dispatches++;
        if (q8) { g->stats.q8_dispatches++; g->stats.quant_projection_dispatches++; }
    }
    return ok && h3_tensor_release(g, w);
}
