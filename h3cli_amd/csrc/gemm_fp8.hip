// FP8 W8A8 projection GEMM: y[M,N] = bf16(sx sw sum_k x8[m,k] w8[n,k]), E4M3 codes,
// FP32 accumulation, on v_mfma_f32_32x32x64_f8f6f4.
//
// The schedule is gemm_bf16_pipe's (gemm.hip): a 256 x 256 output tile per workgroup,
// four waves of 128 x 128 (one per SIMD), each 4 x 4 accumulator blocks of 32 x 32 in
// AGPRs, so one fragment read from LDS feeds four MFMAs. The whole K loop is one
// inline-asm block, because its value is the order of the instructions; with one wave
// per SIMD nothing else hides a stall:
//  * a K tile is 128 bytes, two substeps of sixteen MFMAs (64 K each); the eight 32-byte
//    fragments of the next substep are read in the first eight MFMA slots of the
//    current one, two ds_read_b128 each, into the other register set;
//  * the sixteen global -> LDS loads of a K tile (1 KB each) are issued two tiles ahead,
//    one per MFMA of the second substep, into the stage this tile has finished reading;
//  * one barrier per tile, between the substeps.
// LDS (128 KB): X stages at 0 and 32 KB, W stages at 64 and 96 KB; rows of 128 codes with
// XOR-swizzled 16-byte chunks. Fixed registers: fragment set S in v[64 + 64 S ..], W block
// I at + 8 I, X block J at + 32 + 8 J.
//
// Bound by the MFMAs and the power they draw: 2.5 PFLOP/s at 18225 rows, 5376 -> 21504.
// Measured against eight compiler-scheduled waves of 128 x 64 (two per SIMD), activation
// packing included: 8193 rows, 5376 -> 21504: 780 us (925); 18225 rows: 1.69 ms (2.07);
// 700 rows, 14336 -> 5376: 75 us (200); 60 rows, 5376 -> 21504: 36 us (74). Results equal
// that kernel's bit for bit but for split tiles. Row tiles per band (18225 rows / 8193
// rows, 5376 -> 21504, in us): 2: 1686 / 804, 3: 1840 / 753, 4: 1690 / 832, 6: 1834 / 831,
// 8: 1910 / 841; 4, spread evenly, is taken.
#include "common.h"
#include "internal.h"
#include "gemm.h"
#include "gemm_fp8.h"
#include <algorithm>

namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int TM = 256, TN = 256, TK = 128, TILE = 256 * TK, LDS = 4 * TILE;
constexpr int GROUP_M = 4;

__device__ inline unsigned swz(unsigned row, unsigned ch) { return ch ^ ((row >> 1) & 7); }

// Load T (0..7) of a K tile's X or W into stage ST: LDS block wave + 4 T, rows 8 wave +
// lane / 8 + 32 T. kc: the tile's K byte offset.
#define F8_LX(ST, T) "s_add_u32 m0, %[mb], 32768*" #ST "+4096*" #T "\n"                                             \
    "buffer_load_dwordx4 %[o" #T "], %[sx], %[kc] offen lds\n"
#define F8_LW(ST, T) "s_add_u32 m0, %[mb], 65536+32768*" #ST "+4096*" #T "\n"                                       \
    "buffer_load_dwordx4 %[o" #T "], %[sw], %[kc] offen lds\n"
#define F8_LOADS(ST) F8_LX(ST, 0), F8_LW(ST, 0), F8_LX(ST, 1), F8_LW(ST, 1), F8_LX(ST, 2), F8_LW(ST, 2), F8_LX(ST, 3), \
    F8_LW(ST, 3), F8_LX(ST, 4), F8_LW(ST, 4), F8_LX(ST, 5), F8_LW(ST, 5), F8_LX(ST, 6), F8_LW(ST, 6), F8_LX(ST, 7),     \
    F8_LW(ST, 7)
#define F8_NONE "", "", "", "", "", "", "", "", "", "", "", "", "", "", "", ""
#define F8_MFMA(S, I, J)                                                                                            \
    "v_mfma_f32_32x32x64_f8f6f4 %[c" #I #J "], v[64+64*" #S "+8*" #I ":64+64*" #S "+8*" #I "+7], "                   \
    "v[64+64*" #S "+32+8*" #J ":64+64*" #S "+32+8*" #J "+7], %[c" #I #J "]\n"
// Fragment F of substep KS, stage ST, into set T: its two 16-byte halves.
#define F8_RW(T, F, KS, ST)                                                                                         \
    "ds_read_b128 v[64+64*" #T "+8*" #F ":64+64*" #T "+8*" #F "+3], %[w" #KS "0] offset:32768*" #ST "+4096*" #F "\n"     \
    "ds_read_b128 v[64+64*" #T "+8*" #F "+4:64+64*" #T "+8*" #F "+7], %[w" #KS "1] offset:32768*" #ST "+4096*" #F "\n"
#define F8_RX(T, F, KS, ST)                                                                                         \
    "ds_read_b128 v[64+64*" #T "+32+8*" #F ":64+64*" #T "+32+8*" #F "+3], %[x" #KS "0] offset:32768*" #ST "+4096*" #F "\n" \
    "ds_read_b128 v[64+64*" #T "+32+8*" #F "+4:64+64*" #T "+32+8*" #F "+7], %[x" #KS "1] offset:32768*" #ST "+4096*" #F "\n"
// A substep of set S that reads substep KS of stage ST into set T; L0..L15 behind its MFMAs.
#define F8_SUB(S, T, KS, ST, L0, L1, L2, L3, L4, L5, L6, L7, L8, L9, L10, L11, L12, L13, L14, L15)                    \
    F8_MFMA(S, 0, 0) F8_RW(T, 0, KS, ST) L0 F8_MFMA(S, 0, 1) F8_RX(T, 0, KS, ST) L1                                  \
    F8_MFMA(S, 0, 2) F8_RX(T, 1, KS, ST) L2 F8_MFMA(S, 0, 3) F8_RX(T, 2, KS, ST) L3                                  \
    F8_MFMA(S, 1, 0) F8_RX(T, 3, KS, ST) L4 F8_MFMA(S, 1, 1) F8_RW(T, 1, KS, ST) L5                                  \
    F8_MFMA(S, 1, 2) F8_RW(T, 2, KS, ST) L6 F8_MFMA(S, 1, 3) F8_RW(T, 3, KS, ST) L7                                  \
    F8_MFMA(S, 2, 0) L8 F8_MFMA(S, 2, 1) L9 F8_MFMA(S, 2, 2) L10 F8_MFMA(S, 2, 3) L11                                \
    F8_MFMA(S, 3, 0) L12 F8_MFMA(S, 3, 1) L13 F8_MFMA(S, 3, 2) L14 F8_MFMA(S, 3, 3) L15
#define F8_SUB_EXP(...) F8_SUB(__VA_ARGS__)
#define F8_TILE(ST, OT)                                                                                             \
    F8_SUB_EXP(0, 1, 1, ST, F8_NONE)                                                                                 \
    "s_waitcnt vmcnt(0) lgkmcnt(0)\n"                                                                               \
    "s_barrier\n"                                                                                                   \
    "s_min_u32 %[kc], %[kn], %[kmax]\n"                                                                             \
    "s_add_u32 %[kn], %[kn], 128\n"                                                                                 \
    F8_SUB_EXP(1, 0, 0, OT, F8_LOADS(ST))                                                                            \
    "s_waitcnt lgkmcnt(0)\n"
#define F8_FIRST(ST, KC) "s_mov_b32 %[kc], " KC "\n" F8_LX(ST, 0) F8_LW(ST, 0) F8_LX(ST, 1) F8_LW(ST, 1) F8_LX(ST, 2)      \
    F8_LW(ST, 2) F8_LX(ST, 3) F8_LW(ST, 3) F8_LX(ST, 4) F8_LW(ST, 4) F8_LX(ST, 5) F8_LW(ST, 5) F8_LX(ST, 6)             \
    F8_LW(ST, 6) F8_LX(ST, 7) F8_LW(ST, 7)
#define F8_ACC4(I) [c##I##0] "+a"(c[I][0]), [c##I##1] "+a"(c[I][1]), [c##I##2] "+a"(c[I][2]), [c##I##3] "+a"(c[I][3])
#define F8_CL10(x) "v" #x "0", "v" #x "1", "v" #x "2", "v" #x "3", "v" #x "4", "v" #x "5", "v" #x "6", "v" #x "7",     \
    "v" #x "8", "v" #x "9"

__device__ inline void fp8_tile(const Fp8GemmArgs &a, unsigned pid, unsigned &m0, unsigned &n0) {
    unsigned tm, tn;
    band_tile((a.m + TM - 1) / TM, (a.n + TN - 1) / TN, GROUP_M, pid, tm, tn);
    m0 = __builtin_amdgcn_readfirstlane(tm * TM);
    n0 = __builtin_amdgcn_readfirstlane(tn * TN);
}

// Output row `row`, accumulator block of 32 columns from col: register group g of lane
// half hf holds columns 8 g + 4 hf + 0..3. Groups g and g + 1 go out together as 16-byte
// stores: v_permlane32_swap gives the low half both halves of group g, the high half
// those of group g + 1.
__device__ inline void fp8_store(const Fp8GemmArgs &a, unsigned row, unsigned col, unsigned hf, const f32x4 *c, float scale) {
    if (col >= a.n) return;     // N is a multiple of 128: the last tile may be half full
    uint16_t *dst = a.y + (size_t)row * a.n + col;
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
        unsigned w[2][2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            u16x4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = f32_to_bf16(c[g + h][e] * scale);
            w[h][0] = o[0] | ((unsigned)o[1] << 16);
            w[h][1] = o[2] | ((unsigned)o[3] << 16);
        }
        const auto s0 = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
        *reinterpret_cast<u32x4 *>(dst + 8 * (g + hf)) = u32x4{s0[0], s1[0], s0[1], s1[1]};
    }
}

// SPLIT: the tiles of the last, incomplete wave are shared over K, as in gemm_bf16_pipe.
template <bool SPLIT>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(1, 1)))
void fp8_gemm_pipe(Fp8GemmArgs a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const unsigned tid = threadIdx.x, lane = tid % 64, n32 = lane % 32, hf = lane / 32;
    const unsigned wave = __builtin_amdgcn_readfirstlane(tid / 64), wm = wave / 2, wn = wave % 2;
    unsigned ksteps = a.k / TK;
    TileShare t{};
    if constexpr (SPLIT) t = tile_share(a.tile, ksteps);
    else t.pid = xcd_remap(blockIdx.x, gridDim.x);
    const unsigned k0 = t.first * TK;
    unsigned m0, n0;
    fp8_tile(a, t.pid, m0, n0);
    const uint64_t xbase = (uint64_t)(a.x + (size_t)m0 * a.k + k0), wbase = (uint64_t)(a.w + (size_t)n0 * a.k + k0);
    const unsigned xrows = min(a.m - m0, (unsigned)TM), wrows = min(a.n - n0, (unsigned)TN);
    // Rows past M or N are past the resources' size and load zeros.
    const i32x4 sx = {(int)__builtin_amdgcn_readfirstlane((unsigned)xbase),
                      (int)__builtin_amdgcn_readfirstlane((unsigned)(xbase >> 32)),
                      (int)__builtin_amdgcn_readfirstlane(xrows * a.k - k0), 0x00020000};
    const i32x4 sw = {(int)__builtin_amdgcn_readfirstlane((unsigned)wbase),
                      (int)__builtin_amdgcn_readfirstlane((unsigned)(wbase >> 32)),
                      (int)__builtin_amdgcn_readfirstlane(wrows * a.k - k0), 0x00020000};
    const unsigned lrow = 8 * wave + lane / 8;
    // From K = 2^24 on, rows of 128 and more are past M and N (h3_gemm_fp8) and their offsets
    // would wrap: out of range instead.
    const unsigned past = a.k >> 24 ? BUFFER_OOB : 0u;
    unsigned o[8];
#pragma unroll
    for (int t = 0; t < 8; t++) o[t] = (lrow + 32 * t) * a.k + swz(lrow, lane % 8) * 16 | (t < 4 ? 0u : past);
    const unsigned mb = __builtin_amdgcn_readfirstlane(wave * 1024);
    const unsigned kmax = __builtin_amdgcn_readfirstlane((ksteps - 1) * TK);
    const unsigned kone = min(kmax, (unsigned)TK);
    unsigned kn = 2 * TK, kc = 0, steps = __builtin_amdgcn_readfirstlane(ksteps);
    // Fragment bases in stage 0: row n32 of the wave's half, bytes 32 hf .. + 31 of substep
    // s, that is chunks 4 s + 2 hf and the next one.
    unsigned pw[2][2], px[2][2];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const unsigned part = n32 * TK + swz(n32, 4 * s + 2 * hf + h) * 16;
            pw[s][h] = 2 * TILE + wn * 128 * TK + part;
            px[s][h] = wm * 128 * TK + part;
        }
    f32x16 c[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) c[i][j] = f32x16{};
    // Prologue: tiles 0 and 1 into stages 0 and 1, substep 0 of tile 0 into set 0. The loop
    // body is two tiles, left after the first where their count is odd; loads past the
    // end reload the last tile into a stage nobody reads again.
    asm volatile(
        F8_FIRST(0, "0") F8_FIRST(1, "%[kone]")
        "s_waitcnt vmcnt(0)\n"
        "s_barrier\n"
        F8_RW(0, 0, 0, 0) F8_RW(0, 1, 0, 0) F8_RW(0, 2, 0, 0) F8_RW(0, 3, 0, 0)
        F8_RX(0, 0, 0, 0) F8_RX(0, 1, 0, 0) F8_RX(0, 2, 0, 0) F8_RX(0, 3, 0, 0)
        "s_waitcnt lgkmcnt(0)\n"
        "f8_loop_%=:\n"
        F8_TILE(0, 1)
        "s_sub_u32 %[steps], %[steps], 1\n"
        "s_cmp_eq_u32 %[steps], 0\n"
        "s_cbranch_scc1 f8_end_%=\n"
        F8_TILE(1, 0)
        "s_sub_u32 %[steps], %[steps], 1\n"
        "s_cmp_lg_u32 %[steps], 0\n"
        "s_cbranch_scc1 f8_loop_%=\n"
        "f8_end_%=:\n"
        "s_waitcnt vmcnt(0) lgkmcnt(0)\n"
        // The last MFMAs' results are complete before the epilogue reads the accumulators
        // (hipcc does not see the MFMAs inside this block).
        "s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7\n"
        : F8_ACC4(0), F8_ACC4(1), F8_ACC4(2), F8_ACC4(3), [kc] "+s"(kc), [kn] "+s"(kn), [steps] "+s"(steps)
        : [sx] "s"(sx), [sw] "s"(sw), [o0] "v"(o[0]), [o1] "v"(o[1]), [o2] "v"(o[2]), [o3] "v"(o[3]),
          [o4] "v"(o[4]), [o5] "v"(o[5]), [o6] "v"(o[6]), [o7] "v"(o[7]), [mb] "s"(mb), [kmax] "s"(kmax),
          [kone] "s"(kone), [w00] "v"(pw[0][0]), [w01] "v"(pw[0][1]), [w10] "v"(pw[1][0]), [w11] "v"(pw[1][1]),
          [x00] "v"(px[0][0]), [x01] "v"(px[0][1]), [x10] "v"(px[1][0]), [x11] "v"(px[1][1])
        : "v64", "v65", "v66", "v67", "v68", "v69", F8_CL10(7), F8_CL10(8), F8_CL10(9), F8_CL10(10), F8_CL10(11),
          F8_CL10(12), F8_CL10(13), F8_CL10(14), F8_CL10(15), F8_CL10(16), F8_CL10(17), F8_CL10(18), "v190", "v191",
          "m0", "scc", "memory");

    // Block (i, j): lane holds output row m0 + 128 wm + 32 j + n32.
    const float scale = a.sx[0] * a.sw[0];
    if (SPLIT && t.partial) {
        f32x4 *dst = reinterpret_cast<f32x4 *>(a.tile.part) +
                     ((size_t)t.tile * a.tile.split + t.share) * (TM * TN / 4) + tid;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (m0 + wm * 128 + j * 32 >= a.m) break;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                hold(c[i][j]);
#pragma unroll
                for (int g = 0; g < 4; g++)
                    dst[((j * 4 + i) * 4 + g) * 256] =
                        f32x4{c[i][j][4 * g], c[i][j][4 * g + 1], c[i][j][4 * g + 2], c[i][j][4 * g + 3]};
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const unsigned row = m0 + wm * 128 + j * 32 + n32;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            f32x4 block[4];
            hold(c[i][j]);
#pragma unroll
            for (int g = 0; g < 4; g++)
                block[g] = f32x4{c[i][j][4 * g], c[i][j][4 * g + 1], c[i][j][4 * g + 2], c[i][j][4 * g + 3]};
            if (row < a.m) fp8_store(a, row, n0 + wn * 128 + i * 32, hf, block, scale);
        }
    }
}

// The split tiles' shares added in order, and the epilogue. One workgroup per (tile,
// accumulator block).
__global__ __launch_bounds__(256) void fp8_gemm_reduce(Fp8GemmArgs a) {
    const unsigned tile = blockIdx.x / 16, j = blockIdx.x % 16 / 4, i = blockIdx.x % 4;
    const unsigned tid = threadIdx.x, wave = tid / 64, lane = tid % 64, n32 = lane % 32, hf = lane / 32;
    unsigned m0, n0;
    fp8_tile(a, split_tile(a.tile, tile), m0, n0);
    const unsigned row = m0 + wave / 2 * 128 + j * 32 + n32;
    if (row >= a.m) return;
    const f32x4 *src = reinterpret_cast<const f32x4 *>(a.tile.part) + (size_t)tile * a.tile.split * (TM * TN / 4) +
                       (j * 4 + i) * 4 * 256 + tid;
    f32x4 block[4];
#pragma unroll
    for (int g = 0; g < 4; g++) block[g] = src[g * 256];
#pragma unroll 4
    for (unsigned s = 1; s < a.tile.split; s++) {
        src += TM * TN / 4;
#pragma unroll
        for (int g = 0; g < 4; g++) block[g] += src[g * 256];
    }
    fp8_store(a, row, n0 + wave % 2 * 128 + i * 32, hf, block, a.sx[0] * a.sw[0]);
}

}  // namespace

// Packed weights have N and K multiples of 128 (h3_gpu_quant_load); any M.
int h3_gemm_fp8(h3_gpu *g, Fp8GemmArgs a) {
    static bool configured = false;
    if (!configured) {
        for (const void *kernel : {(const void *)fp8_gemm_pipe<false>, (const void *)fp8_gemm_pipe<true>})
            if (!h3_hip_check(g, hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS),
                              "FP8 GEMM shared memory"))
                return 0;
        configured = true;
    }
    // Offsets inside a tile's rows have 32 bits. N * K has no more (h3_gpu_quant_load), so from
    // K = 2^24 on the weight has 128 rows, and those of x are taken 128 at a time.
    if ((uint64_t)TM * a.k > UINT32_MAX && a.m > TM / 2) {
        Fp8GemmArgs part = a;
        for (unsigned row = 0; row < a.m; row += TM / 2) {
            part.x = a.x + (size_t)row * a.k;
            part.y = a.y + (size_t)row * a.n;
            part.m = std::min(a.m - row, TM / 2u);
            if (!h3_gemm_fp8(g, part)) return 0;
        }
        return 1;
    }
    const unsigned tiles = (a.m + TM - 1) / TM * ((a.n + TN - 1) / TN);
    // Shared over K where all tiles are at most half a wave, in shares of eight K tiles or
    // more, so that short sums keep one order (14336 -> 5376: 1024 rows, 84 tiles: 3 shares
    // 94 us, whole 136; 2048 rows, 168 tiles: whole 156, 3 shares 199).
    static constexpr GemmRates RATES{1.5f, 1.5f, 0.f, 1.f, 2.f, .09f, .9f};
    const unsigned split = tiles < g->cus ? gemm_last_wave(g, tiles, a.k / TK, RATES, 1.f, 8).split : 1;
    a.tile = split_last_wave(g, tiles, split, a.k / TK, TM * TN);
    const unsigned rest = tiles - a.tile.full;
    h3_note_kernel(g, "fp8_gemm_pipe", 0, a.tile.split);
    hipEvent_t timing = h3_kernel_timing_begin(g);
    if (!rest) {
        hipLaunchKernelGGL(fp8_gemm_pipe<false>, dim3(tiles), dim3(256), LDS, g->compute, a);
    } else {
        hipLaunchKernelGGL(fp8_gemm_pipe<true>, dim3(a.tile.full + rest * a.tile.split), dim3(256), LDS, g->compute, a);
        if (h3_launch_status(g, "native fp8 projection"))
            hipLaunchKernelGGL(fp8_gemm_reduce, dim3(rest * 16), dim3(256), 0, g->compute, a);
    }
    h3_kernel_timing_end(g, timing);
    return h3_launch_status(g, "native fp8 projection");
}
