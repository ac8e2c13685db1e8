// Shared by the projection GEMM translation units: arguments, epilogue math and
// the launchers that h3_gemm chooses between.
#pragma once
#include "common.h"
#include "internal.h"

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr unsigned GEMM_Q8 = 1;

struct GemmPlan {
    float us;             // modelled time
    unsigned tm;          // row tile of gemm_mid, 0: gemm_bf16_pipe, GEMM_Q8: gemm_q8_pipe
    unsigned split;       // K shares of each tile of the last, incomplete wave
    bool dequant;         // W8A16: convert the whole weight to BF16 first
};

// Measured rates of a kernel in microseconds, one workgroup on each CU: a K unit of a tile in
// a whole wave (full); in a wave that occupies a part f of the CUs, part + rise * max(0, f -
// knee), because fewer busy CUs draw less power and clock higher (7168 -> 5376, BF16, 84 /
// 168 / 252 tiles: 114 / 128 / 153); start per wave of workgroups; and for split tiles each
// share's 256 x 256 partial sums, written and read (sum), and each share added in turn (turn).
struct GemmRates {
    float full, part, rise, knee, start, sum, turn;
};

// The modelled time of `tiles` output tiles of `units` K units, `size` times 256 x 256 each, and
// the number of shares of the tiles of the last wave that it is least for. Shares run in one
// round of the CUs: half of a wave or more stays whole (7168 -> 5376, BF16: 84 tiles in 3
// shares 72 us (whole 114), in 4, so two rounds, 96; 168 tiles whole 128, in 3 shares 146).
// Behind one whole wave also two rounds (14336 -> 5376, 420 tiles: 3 shares 621, whole 658).
// Behind eight or more only long 256-row tiles. In us, split / whole: 8941 rows, 11264 ->
// 15104, 9 shares: 2300 / 2521; 7000 rows, 5376 -> 28672, 3: 1626 / 1664; 5742 rows, 8704 ->
// 23808, 2: 1948 / 2008 (of 34 such projections in two shares 32 are faster, by 1.3% in the
// mean). Short ones have nothing to gain (11772 rows, 2240 -> 26112, 3: 1444 / 1409), and
// 128-row tiles, slower there than their rates say, must not pass others by it (2572 rows,
// 12608 -> 25856: 1732, 256 rows 1628).
inline GemmPlan gemm_last_wave(const h3_gpu *g, unsigned tiles, unsigned units, const GemmRates &r, float size = 1.f,
                               unsigned least_units = 1) {
    const unsigned rest = tiles % g->cus, waves = tiles / g->cus, rounds_max = waves == 1 ? 2 : 1;
    auto unit = [&](float busy) { return r.part + r.rise * (busy > r.knee ? busy - r.knee : 0.f); };
    GemmPlan p{(float)waves * (units * r.full + r.start), 0, 1, false};
    if (!rest) return p;
    const float before = p.us;
    p.us += units * unit((float)rest / g->cus) + r.start;
    if (waves >= 8 && (size < 1.f || units * r.full < 85.f)) return p;
    for (unsigned s = 2; s <= 32 && s * least_units <= units && rest * s <= rounds_max * g->cus; s++) {
        const unsigned rounds = (rest * s + g->cus - 1) / g->cus;
        const float busy = (float)(rest * s) / (rounds * g->cus);
        const float t = before + rounds * ((units + s - 1) / s * unit(busy) + r.start) + rest * s * size * r.sum + s * r.turn;
        if (t < p.us) { p.us = t; p.split = s; }
    }
    return p;
}

// Split tiles of a launch. Tiles [0, full) are whole; each later one is taken by `split`
// workgroups, whose FP32 partial sums go to part.
struct TileSplit {
    unsigned tiles, full, split;
    float *part;
};

// Epilogue of h3_gemm after the bias. SwiGLU (no bias): the weight holds hidden gate
// rows, then hidden up rows, n = 2 * hidden, and y is [m, hidden]; only where
// h3_gemm_swiglu_fits.
enum { H3_GEMM_PLAIN = 0, H3_GEMM_GELU = 1, H3_GEMM_SWIGLU = 2 };

struct GemmArgs {
    uint16_t *y;
    const uint16_t *x;
    const void *w;            // bf16 [N,K] or int8 [N,K]
    const float *scales;      // q8: [N, groups]
    const uint16_t *bias;     // optional [N]
    const float *alpha;       // EPI bit 2: device scalar multiplying the accumulator
    unsigned m, n, k, group, groups;
    int gelu;                 // H3_GEMM_PLAIN, _GELU or (pipe and mid kernels) _SWIGLU
    TileSplit tile;           // all kernels but gemm_skinny and gemm_small
};

__device__ inline float gelu_tanh(float v) {
    // Reference h3_gelu_bf16, approximate form (src/cuda/cuda_kernels.cuh:879-902):
    // 0.5 v (1 + tanh(c (v + 0.044715 v^3))), c = sqrt(2 / pi), written as
    // v / (1 + exp(-2 c (v + 0.044715 v^3))) with the hardware exp and
    // reciprocal (no IEEE division, no branches). Large |v| saturate through
    // exp: to v (exp -> 0) or to a signed zero (exp -> inf, reciprocal 0).
    const float u = v * (1.5957691216057308f + 0.071354816272192f * v * v);
    return v * __builtin_amdgcn_rcpf(1.0f + __expf(-u));
}

// silu(gate) * up with the hardware exp and reciprocal, as gelu_tanh: large |gate|
// saturate through exp to gate * up or a signed zero. The reciprocal flushes results below
// the normal range, which 1 / (1 + exp(-gate)) reaches from gate = -87.4 on while exp is
// still finite: it is taken 16 times larger.
__device__ inline float swiglu_fast(float gate, float up) {
    return gate * (__builtin_amdgcn_rcpf(fmaf(__expf(-gate), 0.0625f, 0.0625f)) * 0.0625f) * up;
}

// Pins an accumulator to its AGPRs up to here. An epilogue that branches (whole tile or
// partial sums) reads all of them on both sides; without this hipcc moves the 256 reads in
// front of the branch and spills 8 to 32 registers of the kernel (729 rows, 5376 -> 28672,
// int8 of one scale per column: 246 us, without spills 213).
template <class V> __device__ inline void hold(V &acc) { asm volatile("" : "+a"(acc)); }

// The output tile (pid) of this workgroup, its place among the split ones (tile) and its
// share of the K units: `ksteps` of them from `first` on (on entry those of a whole tile).
// Behind whole waves tiles keep the places that they have in an unsplit launch, so that the
// whole tiles of an XCD meet in its L2 as they do there, and the split ones are its last
// (10000 rows, 5376 -> 28672, 17.5 waves: 2273 us unsplit; in two shares, whole and split
// tiles placed each among themselves, 2394). Without whole waves the shares of one K range
// are neighbours.
struct TileShare {
    unsigned pid, tile, share, first;
    bool partial;
};
__device__ inline unsigned split_tile(const TileSplit &s, unsigned tile) {
    return s.full ? xcd_remap(s.full + tile, s.tiles) : tile;
}
__device__ inline TileShare tile_share(const TileSplit &s, unsigned &ksteps) {
    if (blockIdx.x < s.full) return {xcd_remap(blockIdx.x, s.tiles), 0, 0, 0, false};
    const unsigned rest = s.tiles - s.full, at = s.full ? blockIdx.x - s.full : xcd_remap(blockIdx.x, gridDim.x);
    const unsigned tile = at % rest, share = at / rest;
    const unsigned first = share * ksteps / s.split;
    ksteps = (share + 1) * ksteps / s.split - first;
    return {split_tile(s, tile), tile, share, first, true};
}
// The tiles of a last, incomplete wave in `split` shares of their K units (each share has
// one or more) of `values` partial sums, or whole where there is no memory for those.
inline TileSplit split_last_wave(h3_gpu *g, unsigned tiles, unsigned split, unsigned units, size_t values) {
    const unsigned rest = tiles % g->cus, shares = split < units ? split : units;
    if (!rest || shares <= 1 || !h3_buffer_try(g, &g->gemm_partials, (size_t)rest * shares * values * 4))
        return {tiles, tiles, 1, nullptr};
    return {tiles, tiles - rest, shares, (float *)g->gemm_partials.ptr};
}

// Tile (row, column) of workgroup pid: bands of at most `rows` row tiles sweep the
// columns together, so that the workgroups an XCD runs at a time share both operands in
// its L2. The row tiles are spread evenly over the bands: a last band of one row would
// read the whole weight for it alone (FP8, 8193 rows, 5376 -> 21504, in bands of four:
// 832 us, in nine bands of three or four: 780 us).
__device__ inline void band_tile(unsigned tiles_m, unsigned tiles_n, unsigned rows, unsigned pid, unsigned &tm,
                                 unsigned &tn) {
    const unsigned bands = (tiles_m + rows - 1) / rows, band = ((pid / tiles_n + 1) * bands - 1) / tiles_m;
    const unsigned first = band * tiles_m / bands, count = (band + 1) * tiles_m / bands - first;
    const unsigned at = pid - first * tiles_n;
    tm = first + at % count;
    tn = at / count;
}

// 16 int8 codes of one scale group -> BF16 values w = bf16(code * scale), the
// reconstruction of the reference's Metal kernel (src/metal/shaders.metal:825-827).
__device__ inline void dequant16(const i32x4 &q, float s, bf16x8 *half) {
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        const int word = q[e / 4];
        f32x2 f = {(float)(int8_t)(word >> (8 * (e % 4))) * s, (float)(int8_t)(word >> (8 * (e % 4 + 1))) * s};
        bf16x2 b = __builtin_convertvector(f, bf16x2);
        half[e / 8][e % 8] = b[0];
        half[e / 8][e % 8 + 1] = b[1];
    }
}

int h3_gemm(h3_gpu *g, uint16_t *y, const uint16_t *x, const h3_gpu_tensor *w, const uint16_t *bias, uint32_t m,
            uint32_t k, uint32_t n, int activation);
bool h3_gemm_swiglu_fits(const h3_gpu_tensor *w, uint32_t m, uint32_t k, uint32_t hidden);

// gemm_skinny.hip: at most 16 rows. Sums of up to H3_GEMM_SHORT_K products stay with
// gemm_small: a chain of that length is short (2 rows, 256 -> 5376: 8.3 us against
// 3.2), and its sums, in K order, keep the timestep embedding's bits, which every
// block's modulation depends on.
constexpr unsigned H3_GEMM_SHORT_K = 256;
bool h3_gemm_skinny_fits(const GemmArgs &a, bool q8);
int h3_gemm_skinny(h3_gpu *g, const GemmArgs &a, bool q8);

// gemm_mid.hip: row tiles of tm = 64, 128 or 256, the last wave of tiles in split
// shares of K.
bool h3_gemm_mid_fits(const GemmArgs &a, bool q8);
int h3_gemm_mid(h3_gpu *g, const GemmArgs &a, bool q8, unsigned tm, unsigned split, bool timed = true);

// gemm_q8.hip: per-column W8A16 weights converted in a hand-scheduled loop, 256 x 256 tiles.
bool h3_gemm_q8_fits(const GemmArgs &a);
int h3_gemm_q8(h3_gpu *g, GemmArgs a, unsigned split);
