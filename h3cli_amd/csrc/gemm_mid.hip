// Projections with too few rows for gemm_bf16_pipe's 256 x 256 tiles, or of shapes
// it does not take (any N, K a multiple of 64): y[M,N] = x[M,K] . W[N,K]^T (+bias)
// (+GELU-tanh or SwiGLU), BF16 or W8A16 weights, FP32 accumulation.
//
// A workgroup of eight waves (two per SIMD, (TM / 2) x 64 outputs each, C^T = W . X^T
// on v_mfma_f32_32x32x16_bf16) computes TM x 256 outputs, TM = 64, 128 or 256. All
// operands go from memory to LDS without registers, as many 64-wide K steps ahead as
// LDS holds stages (64 rows: four), because a step of few rows is much shorter than a
// memory access; int8 weights are read as such, converted by the wave that loaded
// them a step before their products, and so are read once per row tile instead of
// being written and read again as BF16. The K range of the last wave of tiles is
// split as in gemm_bf16_pipe.
//
// Bound by memory latency and the int8 conversion at 64 rows, by the LDS-fed products
// at 256. Measured against the pipe kernel with its conversion pass, int8 of group 64: 33
// rows, 5376 -> 28672: 58 us (171); 256 rows, 14336 -> 5376: 65 us (113); 729 rows, 5376 ->
// 28672: 263 us (281); without one, BF16: 128 rows, 5120 -> 5120: 21 us (29); and against
// one thread per output: 729 rows, 5376 -> 96: 15 us (337).
#include "common.h"
#include "internal.h"
#include "gemm.h"

namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int TN = 256, TK = 64, T = 512;
constexpr int ROW_BYTES = TK * 2;               // 128 B per BF16 tile row
constexpr int W_BYTES = TN * ROW_BYTES;         // 32 KB
constexpr int W8_BYTES = TN * TK;               // 16 KB int8 tile
constexpr int GROUP_M = 8;

__device__ inline unsigned swz(unsigned row, unsigned ch) { return ch ^ ((row >> 1) & 7); }
// Chunk c (0..1023) of a 256 x 64 int8 tile -> (row, 16-byte part): eight consecutive
// lanes take rows of one parity, so their LDS stores hit eight different chunks.
__device__ inline unsigned w_row(unsigned c) { const unsigned l = c % 16; return (c / 64) * 16 + 2 * (l % 8) + l / 8; }
__device__ inline unsigned w_part(unsigned c) { return (c / 16) % 4; }

// Weight formats: BF16, int8 with one scale per output column, int8 with a scale per
// column and group of K values (a multiple of 16).
enum { BF16 = 0, CHANNEL = 1, GROUPED = 2 };
// Stages of the operands as they come from memory: as many as LDS holds. Grouped
// scales come through LDS with them where that is more than two (512 threads x 2).
template <int W, int TM> constexpr int depth() { return TM == 64 ? (W == GROUPED ? 3 : 4) : TM == 128 && W != GROUPED ? 3 : 2; }
template <int W, int TM> constexpr int x_bytes() { return TM * ROW_BYTES; }
template <int W, int TM> constexpr int scale_bytes() { return W == GROUPED && depth<W, TM>() > 2 ? T * 8 : 0; }
template <int W, int TM> constexpr int lds_bytes() {
    return depth<W, TM>() * (x_bytes<W, TM>() + (W == BF16 ? W_BYTES : W8_BYTES) + scale_bytes<W, TM>()) +
           (W == BF16 ? 0 : 2 * W_BYTES);
}

// Waits for all but N of this wave's vector-memory loads and for its LDS accesses,
// then for the other waves. In asm because hipcc's own barrier and fences wait for
// every load to LDS, those of later steps included.
template <int N> __device__ inline void step_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

__device__ inline __amdgpu_buffer_rsrc_t uniform_resource(const void *p, unsigned bytes) {
    const uint64_t v = (uint64_t)p;
    // readfirstlane returns int: through uint32_t, so that the low word's sign stays out
    // of the high one.
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    const uint64_t u = lo | (uint64_t)hi << 32;
    return __builtin_amdgcn_make_buffer_rsrc((void *)u, (short)0, (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

template <int TM>
__device__ inline void mid_tile(const GemmArgs &a, unsigned pid, unsigned &m0, unsigned &n0) {
    unsigned tm, tn;
    band_tile((a.m + TM - 1) / TM, (a.n + TN - 1) / TN, GROUP_M, pid, tm, tn);
    m0 = __builtin_amdgcn_readfirstlane(tm * TM);
    n0 = __builtin_amdgcn_readfirstlane(tn * TN);
}

// Row of the weight that tile row r holds. SwiGLU: 32 gate rows and the 32 up rows of
// the same columns alternate, so that a lane's two accumulator blocks hold both.
__device__ inline unsigned weight_row(const GemmArgs &a, unsigned r) {
    return a.gelu == H3_GEMM_SWIGLU ? r / 32 % 2 * (a.n / 2) + r / 64 * 32 + r % 32 : r;
}

// Four columns of output row `row`. width: columns of y. alpha: 1 without one (exact).
__device__ inline void store4(uint16_t *y, unsigned row, unsigned col, unsigned width, u16x4 out) {
    uint16_t *dst = y + (size_t)row * width + col;
    if (width % 4 == 0) *reinterpret_cast<u16x4 *>(dst) = out;
    else
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (col + e < width) dst[e] = out[e];
}
__device__ inline void mid_store(const GemmArgs &a, unsigned row, unsigned col, f32x4 v, float alpha) {
    if (row >= a.m || col >= a.n) return;
    v *= alpha;
    if (a.bias) {
        u16x4 b;
        if (a.n % 4 == 0) b = *reinterpret_cast<const u16x4 *>(a.bias + col);
        else
#pragma unroll
            for (int e = 0; e < 4; e++) b[e] = a.bias[min(col + e, a.n - 1)];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] += bf16_to_f32(b[e]);
    }
    u16x4 out;
#pragma unroll
    for (int e = 0; e < 4; e++) out[e] = f32_to_bf16(v[e]);
    if (a.gelu)
#pragma unroll
        for (int e = 0; e < 4; e++) out[e] = f32_to_bf16(gelu_tanh(bf16_to_f32(out[e])));
    store4(a.y, row, col, a.n, out);
}
// Blocks 0 and 1 of a wave (64 columns from col0), register group g, lane half hf.
__device__ inline void mid_store_pair(const GemmArgs &a, unsigned row, unsigned col0, unsigned g, unsigned hf, f32x4 v0,
                                      f32x4 v1, float alpha) {
    if (a.gelu == H3_GEMM_SWIGLU) {
        const unsigned col = col0 / 2 + g * 8 + hf * 4;
        if (row >= a.m || col >= a.n / 2) return;
        u16x4 out;
#pragma unroll
        for (int e = 0; e < 4; e++)
            out[e] = f32_to_bf16(swiglu_fast(bf16_to_f32(f32_to_bf16(v0[e])), bf16_to_f32(f32_to_bf16(v1[e]))));
        store4(a.y, row, col, a.n / 2, out);
        return;
    }
    mid_store(a, row, col0 + g * 8 + hf * 4, v0, alpha);
    mid_store(a, row, col0 + 32 + g * 8 + hf * 4, v1, alpha);
}

template <int W, int TM>
__global__ __attribute__((amdgpu_flat_work_group_size(T, T), amdgpu_waves_per_eu(2, 2)))
void gemm_mid(GemmArgs a) {
    constexpr bool Q8 = W != BF16, LDS_SCALES = scale_bytes<W, TM>() > 0;
    constexpr int NBM = TM / 64, NBN = 2, D = depth<W, TM>(), X_BYTES = x_bytes<W, TM>();
    constexpr int RAW = Q8 ? W8_BYTES : W_BYTES;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    // LDS: D stages of x, D of the weight as stored, D of scales; two of dequantized weight.
    uint8_t *const ws_raw = lds + D * X_BYTES, *const scs = ws_raw + D * RAW;
    uint8_t *const ws_deq = scs + D * scale_bytes<W, TM>();
    const unsigned tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const unsigned n32 = lane % 32, hf = lane / 32, wm = wave / 4, wn = wave % 4;
    unsigned ksteps = a.k / TK;
    const TileShare t = tile_share(a.tile, ksteps);
    const unsigned k0 = __builtin_amdgcn_readfirstlane(t.first * TK);
    ksteps = __builtin_amdgcn_readfirstlane(ksteps);
    unsigned m0, n0;
    mid_tile<TM>(a, t.pid, m0, n0);

    // Rows past M or N are past the resources' size and load zeros (SwiGLU: up rows
    // past the end; gate rows past it are up rows, whose columns are not stored).
    const unsigned xrows = min(a.m - m0, (unsigned)TM), first = a.gelu == H3_GEMM_SWIGLU ? n0 / 2 : n0;
    const unsigned wrows = a.gelu == H3_GEMM_SWIGLU ? a.n - first : min(a.n - n0, (unsigned)TN);
    constexpr unsigned WB = Q8 ? 1 : 2;
    const __amdgpu_buffer_rsrc_t xr = uniform_resource(a.x + (size_t)m0 * a.k + k0, (xrows * a.k - k0) * 2);
    const __amdgpu_buffer_rsrc_t wr =
        uniform_resource((const char *)a.w + ((size_t)first * a.k + k0) * WB, (wrows * a.k - k0) * WB);
    // BF16 operand block b = wave + 8 t: rows 8 b + lane / 8, 16-byte chunk lane % 8 (swizzled).
    const unsigned lrow = 8 * wave + lane / 8;
    const uint32_t off = (lrow * a.k + swz(lrow, lane % 8) * 8) * 2, off_step = 64 * a.k * 2;
    // int8 chunks tid + 512 j: tile row w_row(tid) + 128 j, part w_part(tid).
    const unsigned wrow = w_row(tid), wpart = w_part(tid);
    uint32_t woff[4];
#pragma unroll
    for (int t = 0; t < (Q8 ? 2 : 4); t++)
        woff[t] = Q8 ? weight_row(a, wrow + 128 * t) * a.k + wpart * 16
                     : (weight_row(a, lrow + 64 * t) * a.k + swz(lrow, lane % 8) * 8) * 2;
    // Rows past N read the last row's scales; their codes are zero.
    const float *sp[2];
    if constexpr (Q8)
#pragma unroll
        for (int j = 0; j < 2; j++) sp[j] = a.scales + (size_t)min(first + weight_row(a, wrow + 128 * j), a.n - 1) * a.groups;

    f32x16 acc[NBN][NBM];
#pragma unroll
    for (int i = 0; i < NBN; i++)
#pragma unroll
        for (int j = 0; j < NBM; j++) acc[i][j] = f32x16{};

    // Loads of step kt into stage st; steps past the end reload the last one into a
    // stage that nobody reads again.
    auto load_x = [&](unsigned kt, unsigned st) {
        kt = __builtin_amdgcn_readfirstlane(min(kt, ksteps - 1));
#pragma unroll
        for (int t = 0; t < NBM; t++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                xr, (__attribute__((address_space(3))) void *)(lds + st * X_BYTES + (wave + 8 * t) * 1024), 16,
                off + t * off_step, kt * TK * 2, 0, 0);
    };
    auto load_w = [&](unsigned kt, unsigned st) {
        kt = __builtin_amdgcn_readfirstlane(min(kt, ksteps - 1));
        uint8_t *dst = ws_raw + st * RAW;
        if constexpr (Q8) {
#pragma unroll
            for (int j = 0; j < 2; j++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    wr, (__attribute__((address_space(3))) void *)(dst + (wave + 8 * j) * 1024), 16, woff[j], kt * TK, 0, 0);
        } else {
#pragma unroll
            for (int t = 0; t < 4; t++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    wr, (__attribute__((address_space(3))) void *)(dst + (wave + 8 * t) * 1024), 16, woff[t], kt * TK * 2,
                    0, 0);
        }
        if constexpr (LDS_SCALES)
#pragma unroll
            for (int j = 0; j < 2; j++)
                __builtin_amdgcn_global_load_lds(
                    (const __attribute__((address_space(1))) void *)(sp[j] + (k0 + kt * TK + wpart * 16) / a.group),
                    (__attribute__((address_space(3))) void *)(scs + st * T * 8 + (wave + 8 * j) * 256), 4, 0, 0);
    };
    float wscale[2] = {};
    auto load_scale = [&](unsigned kt) {
        kt = min(kt, ksteps - 1);
        if constexpr (Q8 && !LDS_SCALES)
#pragma unroll
            for (int j = 0; j < 2; j++) wscale[j] = sp[j][W == CHANNEL ? 0 : (k0 + kt * TK + wpart * 16) / a.group];
    };
    // int8 stage st (this thread's own chunks and scales) -> BF16 stage at & 1.
    auto dequant = [&](unsigned st, unsigned at) {
        if constexpr (Q8) {
            const uint8_t *src = ws_raw + st * RAW;
            uint8_t *ws = ws_deq + (at & 1) * W_BYTES;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const unsigned row = wrow + 128 * j;
                const float s = LDS_SCALES ? *reinterpret_cast<const float *>(scs + st * T * 8 + (tid + T * j) * 4) : wscale[j];
                bf16x8 half[2];
                dequant16(*reinterpret_cast<const i32x4 *>(src + (tid + T * j) * 16), s, half);
                *reinterpret_cast<bf16x8 *>(ws + row * ROW_BYTES + swz(row, wpart * 2) * 16) = half[0];
                *reinterpret_cast<bf16x8 *>(ws + row * ROW_BYTES + swz(row, wpart * 2 + 1) * 16) = half[1];
            }
        }
    };
    auto frags = [&](unsigned st, unsigned at, int ks, bf16x8 *wf, bf16x8 *xf) {
        const uint8_t *xs = lds + st * X_BYTES, *ws = Q8 ? ws_deq + (at & 1) * W_BYTES : ws_raw + st * RAW;
#pragma unroll
        for (int i = 0; i < NBN; i++) {
            const unsigned r = wn * 64 + i * 32 + n32;
            wf[i] = *reinterpret_cast<const bf16x8 *>(ws + r * ROW_BYTES + swz(r, ks * 2 + hf) * 16);
        }
#pragma unroll
        for (int j = 0; j < NBM; j++) {
            const unsigned r = wm * (TM / 2) + j * 32 + n32;
            xf[j] = *reinterpret_cast<const bf16x8 *>(xs + r * ROW_BYTES + swz(r, ks * 2 + hf) * 16);
        }
    };

    // Step kt issues the loads of step kt + D - 1 (int8 weights one step further on,
    // since they are dequantized a step ahead of their products) and ends waiting
    // for those of step kt + 1: D - 2 steps' loads stay in flight. An int8 chunk is
    // loaded and dequantized by the same wave, so its wait needs no barrier.
    constexpr int GROUP = NBM + (Q8 ? 2 : 4) + (LDS_SCALES ? 2 : 0), AHEAD = (D - 2) * GROUP;
    load_scale(0);
#pragma unroll
    for (int s = 0; s < D - 1; s++) {
        load_w(s, s);
        load_x(s, s);
    }
    if constexpr (Q8) load_w(D - 1, D - 1);
    step_barrier<0>();
    dequant(0, 0);
    if constexpr (W == GROUPED) load_scale(1);
    if constexpr (Q8) step_barrier<0>();

    // One barrier per step: the next step's first fragments are read behind it,
    // before the last MFMAs of this one (the sched_barrier keeps them there).
    bf16x8 wf[2][NBN], xf[2][NBM];
    frags(0, 0, 0, wf[0], xf[0]);
    unsigned cur = 0;                                     // kt % D
    for (unsigned kt = 0; kt < ksteps; kt++) {
        const unsigned next = cur + 1 == D ? 0 : cur + 1, last = cur == 0 ? D - 1 : cur - 1;
        if constexpr (Q8) load_w(kt + D, cur);
        else load_w(kt + D - 1, last);
        load_x(kt + D - 1, last);
#pragma unroll
        for (int ks = 0; ks < TK / 16; ks++) {
            if (ks + 1 < TK / 16) {
                frags(cur, kt, ks + 1, wf[(ks + 1) & 1], xf[(ks + 1) & 1]);
            } else {
                step_barrier<AHEAD>();
                frags(next, kt + 1, 0, wf[0], xf[0]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NBN; i++)
#pragma unroll
                for (int j = 0; j < NBM; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[ks & 1][i], xf[ks & 1][j], acc[i][j], 0, 0, 0);
            if (ks == 0) {
                dequant(next, kt + 1);
                if constexpr (W == GROUPED) load_scale(kt + 2);
            }
        }
        cur = next;
    }
    wait_vm_loads();   // LDS must not be written after the workgroup has ended

    // Lane: output row m0 + wm * TM / 2 + 32 j + n32, columns n0 + 64 wn + 32 i + 8 g + 4 hf + 0..3.
    auto part4 = [&](int i, int j, int g) {
        return f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
    };
    if (t.partial) {
        f32x4 *dst = reinterpret_cast<f32x4 *>(a.tile.part) +
                     ((size_t)t.tile * a.tile.split + t.share) * (TM * TN / 4) + tid;
#pragma unroll
        for (int j = 0; j < NBM; j++) {
            if (m0 + wm * (TM / 2) + j * 32 >= a.m) break;
#pragma unroll
            for (int i = 0; i < NBN; i++)
#pragma unroll
                for (int g = 0; g < 4; g++) dst[((j * NBN + i) * 4 + g) * T] = part4(i, j, g);
        }
        return;
    }
    const float alpha = a.alpha ? a.alpha[0] : 1.f;
#pragma unroll
    for (int j = 0; j < NBM; j++)
#pragma unroll
        for (int g = 0; g < 4; g++)
            mid_store_pair(a, m0 + wm * (TM / 2) + j * 32 + n32, n0 + wn * 64, g, hf, part4(0, j, g), part4(1, j, g), alpha);
}

// The split tiles' shares added in order, and the epilogue. One workgroup per (tile,
// row block j, register group g).
template <int TM>
__global__ __launch_bounds__(T) void gemm_mid_reduce(GemmArgs a) {
    constexpr unsigned BLOCKS = TM / 64 * 4;
    const unsigned tile = blockIdx.x / BLOCKS, j = blockIdx.x % BLOCKS / 4, g = blockIdx.x % 4;
    const unsigned tid = threadIdx.x, wave = tid / 64, lane = tid % 64, n32 = lane % 32, hf = lane / 32;
    unsigned m0, n0;
    mid_tile<TM>(a, split_tile(a.tile, tile), m0, n0);
    const unsigned row = m0 + wave / 4 * (TM / 2) + j * 32 + n32;
    if (row >= a.m) return;
    const f32x4 *src = reinterpret_cast<const f32x4 *>(a.tile.part) +
                       (size_t)tile * a.tile.split * (TM * TN / 4) + (j * 8 + g) * T + tid;
    f32x4 v0 = src[0], v1 = src[4 * T];
#pragma unroll 4
    for (unsigned s = 1; s < a.tile.split; s++) {
        src += TM * TN / 4;
        v0 += src[0];
        v1 += src[4 * T];
    }
    mid_store_pair(a, row, n0 + wave % 4 * 64, g, hf, v0, v1, a.alpha ? a.alpha[0] : 1.f);
}

template <int W, int TM>
int launch(h3_gpu *g, GemmArgs a, unsigned split, bool timed) {
    constexpr int shared = lds_bytes<W, TM>();
    static_assert(shared <= 160 * 1024, "LDS of a CU");
    static bool configured = false;
    auto kernel = gemm_mid<W, TM>;
    if (!configured) {
        if (!h3_hip_check(g, hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, shared),
                          "GEMM shared memory"))
            return 0;
        configured = true;
    }
    const unsigned tiles = (a.m + TM - 1) / TM * ((a.n + TN - 1) / TN);
    a.tile = split_last_wave(g, tiles, split, a.k / TK, TM * TN);
    const unsigned rest = tiles - a.tile.full;
    h3_note_kernel(g, "gemm_mid", TM, a.tile.split);
    hipEvent_t timing = timed ? h3_kernel_timing_begin(g) : nullptr;
    hipLaunchKernelGGL(kernel, dim3(a.tile.full + rest * a.tile.split), dim3(T), shared, g->compute, a);
    if (rest && h3_launch_status(g, "GEMM"))
        hipLaunchKernelGGL(gemm_mid_reduce<TM>, dim3(rest * (TM / 64) * 4), dim3(T), 0, g->compute, a);
    h3_kernel_timing_end(g, timing);
    return h3_launch_status(g, "GEMM");
}

}  // namespace

bool h3_gemm_mid_fits(const GemmArgs &a, bool q8) {
    // 32-bit offsets inside a tile's rows; SwiGLU reaches from gate to up rows.
    const size_t reach = a.gelu == H3_GEMM_SWIGLU ? (size_t)a.n : 256;
    return a.k % TK == 0 && (!q8 || a.group % 16 == 0) && reach * a.k * 2 < (1ull << 31) && (size_t)256 * a.k * 2 < (1ull << 31);
}

template <int W>
static int launch_tm(h3_gpu *g, const GemmArgs &a, unsigned tm, unsigned split, bool timed) {
    return tm == 64    ? launch<W, 64>(g, a, split, timed)
           : tm == 128 ? launch<W, 128>(g, a, split, timed)
                       : launch<W, 256>(g, a, split, timed);
}

int h3_gemm_mid(h3_gpu *g, const GemmArgs &a, bool q8, unsigned tm, unsigned split, bool timed) {
    if (!q8) return launch_tm<BF16>(g, a, tm, split, timed);
    return a.group == a.k ? launch_tm<CHANNEL>(g, a, tm, split, timed) : launch_tm<GROUPED>(g, a, tm, split, timed);
}
