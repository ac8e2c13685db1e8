// Projections of at most 16 rows (timestep and modulation projections, a few
// conditioning rows): y[M,N] = x[M,K] . W[N,K]^T (+bias) (+GELU-tanh), BF16 or
// W8A16 weights, FP32 accumulation.
//
// Reading W once is all the work there is, so the split is made for memory: a
// workgroup takes 16 * NB output columns and its waves take the K steps in turn
// (64 values a step), so that together they read 128 * WAVES consecutive bytes of
// every weight row; their FP32 partial sums meet in LDS, added in wave order.
// The products run on v_mfma_f32_16x16x32_bf16 (C^T = W . X^T), so the VALU is left with the int8 conversion; x comes from
// L2, which all workgroups share.
//
// HBM-bound. Measured (one thread per output, its predecessor, in brackets):
// 2 rows, 5376 -> 32256, BF16: 61 us, 5.6 TB/s (1268 us, 0.27 TB/s); 9 rows, int8:
// 54 us. From 17 rows on every workgroup's reading of x weighs as much as the
// weights, and gemm_mid is faster (31 rows: 68 us against 77).
#include "common.h"
#include "internal.h"
#include "gemm.h"

namespace {

constexpr int STEP = 64;      // K values per step

template <bool Q8, int NB, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void gemm_skinny(GemmArgs a) {
    constexpr int U = 4;          // K steps in flight per wave
    const unsigned tid = threadIdx.x, wave = tid / 64, lane = tid % 64, n16 = lane % 16, q4 = lane / 16;
    const unsigned n0 = blockIdx.x * 16 * NB, steps = a.k / STEP;
    // MFMA operand element j of lane quarter q4 holds K value 16 q4 + j of the
    // step (first product) or 16 q4 + 8 + j (second), the same for W and X.
    const uint16_t *xp = a.x + (size_t)min(n16, a.m - 1) * a.k + 16 * q4;
    const char *wp[NB];
    const float *sp[NB];
#pragma unroll
    for (int n = 0; n < NB; n++) {
        const size_t row = min(n0 + 16 * n + n16, a.n - 1);   // columns past N repeat the last one; not stored
        wp[n] = (const char *)a.w + (row * a.k + 16 * q4) * (Q8 ? 1 : 2);
        if constexpr (Q8) sp[n] = a.scales + row * a.groups;
    }
    f32x4 acc[NB];
#pragma unroll
    for (int n = 0; n < NB; n++) acc[n] = f32x4{};

    auto run = [&](unsigned s, auto count) {
        constexpr int C = decltype(count)::value;
        bf16x8 x[C][2], w[C][NB][2];
        i32x4 q[C][NB];
        float sc[C][NB];
#pragma unroll
        for (int c = 0; c < C; c++) {
            const size_t k = (size_t)(s + c * WAVES) * STEP;
#pragma unroll
            for (int n = 0; n < NB; n++) {
                if constexpr (Q8) {
                    q[c][n] = *reinterpret_cast<const i32x4 *>(wp[n] + k);
                    sc[c][n] = sp[n][(unsigned)(k + 16 * q4) / a.group];
                } else {
                    w[c][n][0] = *reinterpret_cast<const bf16x8 *>(wp[n] + k * 2);
                    w[c][n][1] = *reinterpret_cast<const bf16x8 *>(wp[n] + k * 2 + 16);
                }
            }
            x[c][0] = *reinterpret_cast<const bf16x8 *>(xp + k);
            x[c][1] = *reinterpret_cast<const bf16x8 *>(xp + k + 8);
        }
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int n = 0; n < NB; n++) {
                if constexpr (Q8) dequant16(q[c][n], sc[c][n], w[c][n]);
#pragma unroll
                for (int h = 0; h < 2; h++)
                    acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[c][n][h], x[c][h], acc[n], 0, 0, 0);
            }
    };
    unsigned s = wave;
    for (; s + (U - 1) * WAVES < steps; s += U * WAVES) run(s, std::integral_constant<int, U>{});
    for (; s < steps; s += WAVES) run(s, std::integral_constant<int, 1>{});

    __shared__ f32x4 part[WAVES][NB][64];
#pragma unroll
    for (int n = 0; n < NB; n++) part[wave][n][lane] = acc[n];
    __syncthreads();
    // Lane of block n: row n16, columns n0 + 16 n + 4 q4 + 0..3.
    if (wave >= NB || n16 >= a.m) return;
    f32x4 v = part[0][wave][lane];
#pragma unroll
    for (int w = 1; w < WAVES; w++) v += part[w][wave][lane];
    const unsigned col = n0 + 16 * wave + 4 * q4;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (col + e >= a.n) break;
        float f = v[e];
        if (a.alpha) f *= a.alpha[0];
        if (a.bias) f += bf16_to_f32(a.bias[col + e]);
        uint16_t o = f32_to_bf16(f);
        if (a.gelu) o = f32_to_bf16(gelu_tanh(bf16_to_f32(o)));
        a.y[(size_t)n16 * a.n + col + e] = o;
    }
}

template <bool Q8, int NB, int WAVES>
int launch(h3_gpu *g, const GemmArgs &a) {
    h3_note_kernel(g, "gemm_skinny");
    hipLaunchKernelGGL((gemm_skinny<Q8, NB, WAVES>), dim3((a.n + 16 * NB - 1) / (16 * NB)), dim3(64 * WAVES), 0,
                       g->compute, a);
    return h3_launch_status(g, "skinny GEMM");
}

// Column blocks per workgroup: x is small beside the weights, and the more workgroups
// the better (5376 -> 32256, 2 rows, BF16: NB 1 / 2 / 4 take 61 / 66 / 68 us; 5376 ->
// 256, 5 rows: 8.6 / 13 / 22 us), except for int8 weights of many columns, whose
// half-size loads meet as many loads of x (9 rows: 63 / 54 / 57 us).
template <bool Q8>
int choose(h3_gpu *g, const GemmArgs &a) {
    if constexpr (Q8)
        if (a.n >= 8192) return launch<Q8, 2, 4>(g, a);
    return launch<Q8, 1, 8>(g, a);
}

}  // namespace

bool h3_gemm_skinny_fits(const GemmArgs &a, bool q8) {
    // Up to 32 threads a column, less than 2^32 in all.
    return a.m <= 16 && a.k > H3_GEMM_SHORT_K && a.k % STEP == 0 && (!q8 || a.group % 16 == 0) && a.n < (1u << 27);
}

int h3_gemm_skinny(h3_gpu *g, const GemmArgs &a, bool q8) { return q8 ? choose<true>(g, a) : choose<false>(g, a); }
