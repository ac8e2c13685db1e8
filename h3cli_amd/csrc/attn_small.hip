// Dense BF16 attention for few query rows (D = 128, non-causal), one launch.
//
// Semantics as attn_bf16.hip: softmax(scale * Q K^T) V with FP32 scores, running max
// and sums, P rounded to BF16 for P.V, FP32 accumulation, BF16 output. With few
// (head, 256-query) tiles that file's kernels leave most of the chip idle and pay
// two more launches (the V transpose and the recomputation); here a workgroup of four
// waves takes 32 * NQ queries, its waves take the 64-key tiles in turn, and their
// partial results meet in LDS:
//  * each wave keeps its own K and V tile in LDS (32 KB, global -> LDS directly, 16-byte
//    chunks XOR-swizzled) and waits for its own loads only, so the key loop has no
//    barrier; the next K tile loads during the softmax and P.V, the next V tile during
//    the next scores;
//  * scores are transposed, S^T = K Q^T, so a lane owns a query column and its P,
//    rounded to BF16, is the B operand of O^T += V^T P^T; V^T fragments come from the
//    row-major V tile by transposing LDS reads (ds_read_b64_tr_b16), in the key order
//    that P has;
//  * a running max per tile, raised when a tile's max passes it by more than 8 (log2
//    units). P is taken 8 below it, so that P <= 1 in every wave, whichever key it has seen
//    first, and a partial O is at most the keys' sum of |V|.
#include "common.h"
#include "internal.h"
#include "attn_common.h"

namespace {

constexpr int D = 128, BN = 64, TILE = BN * D * 2, WAVES = 4;
constexpr float RESCALE_SLACK = 8.0f;

struct SmallArgs {
    uint16_t *out;
    const uint16_t *q, *k, *v;
    unsigned seq, heads;
    float scale_log2;
    int head_major;
    unsigned *fault;
};

// 16-byte chunk swizzle of a 256-byte row.
__device__ inline unsigned chunk(unsigned key, unsigned ch) { return ch ^ (key & 15); }

// The largest exponent field seen, in place (bits 30:23 of a float): non-finite from
// 0x7f800000 on. A running maximum costs no mask registers.
__device__ inline void note_bf16(unsigned &worst, const void *values, int words) {
    const uint32_t *w = static_cast<const uint32_t *>(values);
#pragma unroll
    for (int i = 0; i < words; i++) worst = max(max(worst, w[i] & 0x7f800000u), w[i] << 16 & 0x7f800000u);
}

template <int N> __device__ inline void wait_vm_lds() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory"); }

typedef short i16x4 __attribute__((ext_vector_type(4)));

template <int NQ>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WAVES, 64 * WAVES), amdgpu_waves_per_eu(NQ == 1 ? 2 : 1, NQ == 1 ? 2 : 1)))
void attn_small(SmallArgs a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    __shared__ float mpart[WAVES][NQ][32], lpart[WAVES][NQ][32];
    const unsigned tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const unsigned n = lane % 32, hf = lane / 32;
    const unsigned nqb = (a.seq + 32 * NQ - 1) / (32 * NQ);
    const unsigned id = xcd_remap(blockIdx.x, gridDim.x);
    const unsigned head = __builtin_amdgcn_readfirstlane(id / nqb), qb = __builtin_amdgcn_readfirstlane(id % nqb);
    const unsigned q0 = qb * 32 * NQ, count = (a.seq + BN - 1) / BN;
    const size_t stride = (size_t)a.heads * D;
    const float c = a.scale_log2;
    uint8_t *const kt = smem + wave * 2 * TILE, *const vt = kt + TILE;

    // Tile loads: 1 KB block b of a tile holds keys 4 b + lane / 16, chunk lane % 16
    // (swizzled; the swizzle depends on key % 16, that is on b % 4 and the lane). Rows
    // past S take BUFFER_OOB and load zeros.
    const unsigned size = __builtin_amdgcn_readfirstlane((unsigned)(a.seq * stride * 2));
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc((void *)a.k, (short)0, (int)size, 0x00020000);
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc((void *)a.v, (short)0, (int)size, 0x00020000);
    const unsigned kstride = (unsigned)(stride * 2);
    unsigned off[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const unsigned key = 4 * j + lane / 16;
        off[j] = key * kstride + chunk(key, lane % 16) * 16;
    }
    auto load = [&](const __amdgpu_buffer_rsrc_t &r, uint8_t *dst, unsigned tile) {
        // Not unrolled in full, here and below: a call this short pays for every
        // instruction line it fetches.
        unsigned so = __builtin_amdgcn_readfirstlane(tile * BN * kstride + head * D * 2);
        unsigned left = a.seq - min(a.seq, tile * BN + lane / 16);   // rows from this lane's first one on
#pragma unroll 1
        for (int b = 0; b < 16; b += 4) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    r, (__attribute__((address_space(3))) void *)(dst + (b + j) * 1024), 16,
                    left > 4u * (b + j) ? off[j] : BUFFER_OOB, so, 0, 0);
            so = __builtin_amdgcn_readfirstlane(so + 16 * kstride);
        }
    };
    // Inf and NaN in this wave's copy of a tile.
    unsigned worst = 0;
    auto screen_tile = [&](const uint8_t *tile) {
#pragma unroll 1
        for (int b = 0; b < 16; b++) {
            const i32x4 w = *reinterpret_cast<const i32x4 *>(tile + (b * 64 + lane) * 16);
            note_bf16(worst, &w, 4);
        }
    };

    // Q fragments (rows past S repeat the last row).
    bf16x8 qf[NQ][8];
#pragma unroll
    for (int b = 0; b < NQ; b++) {
        const unsigned row = min(q0 + b * 32 + n, a.seq - 1);
        const uint16_t *p = a.q + (size_t)row * stride + (size_t)head * D + hf * 8;
#pragma unroll
        for (int ks = 0; ks < 8; ks++) qf[b][ks] = *reinterpret_cast<const bf16x8 *>(p + ks * 16);
    }
    unsigned t = wave;
    if (t < count) {
        load(kr, kt, t);
        load(vr, vt, t);
    }
    if (wave == 0)
#pragma unroll
        for (int b = 0; b < NQ; b++)
#pragma unroll
            for (int ks = 0; ks < 8; ks++) note_bf16(worst, &qf[b][ks], 4);
    f32x16 o[NQ][4];
    float m[NQ], l[NQ];
#pragma unroll
    for (int b = 0; b < NQ; b++) {
#pragma unroll
        for (int md = 0; md < 4; md++) o[b][md] = f32x16{};
        m[b] = -1e30f;
        l[b] = 0.f;
    }
    // V^T fragment reads: lane p of a 16-lane group addresses key row p / 4 and channels
    // 4 (p % 4) of a 4 x 16 block and receives channel p of its four keys.
    const unsigned p16 = lane % 16, vrow = hf * 4 + p16 / 4, vch = 2 * (lane / 16 % 2) + p16 % 4 / 2;

    for (; t < count; t += WAVES) {
        const bool more = t + WAVES < count;
        const unsigned key0 = t * BN;
        // Each tile's K and V are screened for Inf and NaN by one of the head's workgroups.
        const bool screen = t % nqb == qb;
        wait_vm_lds<16>();                  // K(t); V(t), loaded after it, may be in flight
        f32x16 s[NQ][2];
#pragma unroll
        for (int b = 0; b < NQ; b++) s[b][0] = s[b][1] = f32x16{};
        {
            bf16x8 kf[16];
#pragma unroll
            for (int x = 0; x < 16; x++) {
                const unsigned key = x % 2 * 32 + n;
                kf[x] = *reinterpret_cast<const bf16x8 *>(kt + key * 256 + chunk(key, x / 2 * 2 + hf) * 16);
            }
            if (screen) screen_tile(kt);
            wait_vm_lds<16>();              // this wave's reads: the tile may be overwritten
            if (more) load(kr, kt, t + WAVES);
#pragma unroll
            for (int ks = 0; ks < 8; ks++)
#pragma unroll
                for (int b = 0; b < NQ; b++)
#pragma unroll
                    for (int mb = 0; mb < 2; mb++)
                        s[b][mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks * 2 + mb], qf[b][ks], s[b][mb], 0, 0, 0);
        }
        if (key0 + BN > a.seq)
#pragma unroll
            for (int b = 0; b < NQ; b++)
#pragma unroll
                for (int mb = 0; mb < 2; mb++)
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        if (key0 + mb * 32 + (r / 4) * 8 + hf * 4 + r % 4 >= a.seq) s[b][mb][r] = -INFINITY;
        bf16x8 pb[NQ][4];
#pragma unroll
        for (int b = 0; b < NQ; b++) {
            float mx0 = -INFINITY, mx1 = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                mx0 = fmaxf(fmaxf(mx0, s[b][0][r]), s[b][0][r + 1]);
                mx1 = fmaxf(fmaxf(mx1, s[b][1][r]), s[b][1][r + 1]);
            }
            const float mx = half_max_swap(fmaxf(mx0, mx1)) * c;
            if (__builtin_amdgcn_ballot_w64(mx > m[b] + RESCALE_SLACK)) {
                const float mnew = fmaxf(m[b], mx), alpha = exp2f_fast(m[b] - mnew);
                m[b] = mnew;
                l[b] *= alpha;
#pragma unroll
                for (int md = 0; md < 4; md++) o[b][md] *= alpha;
            }
            const float neg = -m[b] - RESCALE_SLACK;
            float sum = 0.f;
#pragma unroll
            for (int mb = 0; mb < 2; mb++)
#pragma unroll
                for (int r = 0; r < 16; r += 2) {
                    const float p0 = exp2f_fast(fmaf(s[b][mb][r], c, neg)), p1 = exp2f_fast(fmaf(s[b][mb][r + 1], c, neg));
                    sum += p0 + p1;
                    pb[b][mb * 2 + r / 8][r % 8] = (__bf16)p0;
                    pb[b][mb * 2 + r / 8][r % 8 + 1] = (__bf16)p1;
                }
            l[b] += sum;
        }
        if (more) wait_vm_lds<16>();        // V(t); the next K tile may be in flight
        else wait_vm_lds<0>();
        bf16x8 vf[16];
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int md = 0; md < 4; md++) {
                // Keys 16 kk + 4 hf + 0..3 and 8 further on: the order of P's registers.
                i16x4 half[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const unsigned row = 16 * kk + 8 * h + vrow;
                    half[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) i16x4 *)(vt + row * 256 + chunk(row, md * 4 + vch) * 16 +
                                                                     p16 % 2 * 8));
                }
                vf[kk * 4 + md] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7));
            }
        if (screen) screen_tile(vt);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (more) load(vr, vt, t + WAVES);
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int md = 0; md < 4; md++)
#pragma unroll
                for (int b = 0; b < NQ; b++)
                    o[b][md] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[kk * 4 + md], pb[b][kk], o[b][md], 0, 0, 0);
    }
    wait_vm_loads();

    // The waves' partial results, brought to the common max and added in wave order:
    // wave w finishes channels 32 w .. 32 w + 31. O^T blocks go through the tile memory
    // (16 KB per block of 32 queries).
    if (hf == 0)
#pragma unroll
        for (int b = 0; b < NQ; b++) mpart[wave][b][n] = m[b];
    __syncthreads();
    float *const ob = reinterpret_cast<float *>(smem + wave * 2 * TILE);
#pragma unroll
    for (int b = 0; b < NQ; b++) {
        float top = mpart[0][b][n];
#pragma unroll
        for (int w = 1; w < WAVES; w++) top = fmaxf(top, mpart[w][b][n]);
        const float alpha = exp2f_fast(m[b] - top), sum = half_sum_swap(l[b]) * alpha;
        if (hf == 0) lpart[wave][b][n] = sum;
#pragma unroll
        for (int md = 0; md < 4; md++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *reinterpret_cast<f32x4 *>(ob + ((b * 16 + md * 4 + g) * 64 + lane) * 4) =
                    f32x4{o[b][md][4 * g] * alpha, o[b][md][4 * g + 1] * alpha, o[b][md][4 * g + 2] * alpha,
                          o[b][md][4 * g + 3] * alpha};
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < NQ; b++) {
        const unsigned q = q0 + b * 32 + n;
        float total = lpart[0][b][n];
#pragma unroll
        for (int w = 1; w < WAVES; w++) total += lpart[w][b][n];
        const float inv = total > 0.f ? 1.f / total : 0.f;
        uint16_t *dst = a.out + (a.head_major ? ((size_t)head * a.seq + q) * D : ((size_t)q * a.heads + head) * D);
#pragma unroll
        for (int g = 0; g < 4; g++) {
            f32x4 x{};
#pragma unroll
            for (int w = 0; w < WAVES; w++)
                x += *reinterpret_cast<const f32x4 *>(smem + w * 2 * TILE + ((b * 16 + wave * 4 + g) * 64 + lane) * 16);
            u16x4 out;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float y = x[e] * inv;
                worst = max(worst, __builtin_bit_cast(uint32_t, y) & 0x7f800000u);   // rows past S repeat the last one
                out[e] = f32_to_bf16(y);
            }
            if (q < a.seq) *reinterpret_cast<u16x4 *>(dst + wave * 32 + g * 8 + hf * 4) = out;
        }
    }
    if (worst >= 0x7f800000u) a.fault[0] = 1u;
}

template <int NQ>
int launch(h3_gpu *g, const SmallArgs &a) {
    constexpr size_t shared = WAVES * 2 * TILE;
    static bool configured = false;
    if (!configured) {
        if (!h3_hip_check(g, hipFuncSetAttribute((const void *)attn_small<NQ>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)shared), "attention shared memory"))
            return 0;
        configured = true;
    }
    h3_note_kernel(g, "attn_small", 32 * NQ);
    hipEvent_t timing = h3_kernel_timing_begin(g);
    hipLaunchKernelGGL(attn_small<NQ>, dim3((a.seq + 32 * NQ - 1) / (32 * NQ) * a.heads), dim3(64 * WAVES), shared,
                       g->compute, a);
    h3_kernel_timing_end(g, timing);
    return h3_launch_status(g, "BF16 attention");
}

}  // namespace

// Workgroup rounds and modelled microseconds: the kernels here by 64-key tiles per
// wave, the 256-query tile kernel by 128-key groups, the V transpose and the
// recomputation launch included. Measured, calls back to back (it in brackets): 1024
// keys x 8 heads, one block 15.2, two 22.0 (34.8); 300 x 4: 10.6, 15.9 (23.8); 2048 x
// 8: 41.7, 36.0 (53.1); 4200 x 2: 69.2, 58.9 (87.2); 384 x 40: 20.1, 16.8 (27.1); 1024
// x 24: 39.2, 42.8 (40.6); 729 x 56: 57.8, 54.7 (41.2). A second round is counted in
// full though it starts beside the first, so that just past one round the tile kernel
// runs where one block is faster: 448 x 40: 22.9, 28.4 (30.3); 512 x 40: 25.9, 31.1 (31.4).
int h3_attention_small_blocks(const h3_gpu *g, uint32_t seq, uint32_t heads) {
    // Every other variant is one of the tile kernels (15: the default one).
    if (g->attention_variant || (size_t)seq * heads * D * 2 >= (1ull << 32)) return 0;   // 32-bit buffer offsets
    const float tiles = (float)((seq + BN * WAVES - 1) / (BN * WAVES));   // of the busiest wave
    auto rounds = [&](uint32_t queries) {
        return (float)(((uint64_t)((seq + queries - 1) / queries) * heads + g->cus - 1) / g->cus);
    };
    const float one = rounds(32) * (8.f + 2.2f * tiles), two = rounds(64) * (12.f + 3.f * tiles);
    const float wide = 15.f + rounds(256) * (2.f + 2.13f * (float)((seq + 127) / 128));
    return one <= two ? (one < wide ? 1 : 0) : (two < wide ? 2 : 0);
}

int h3_launch_attention_small(h3_gpu *g, int blocks, uint16_t *out, const uint16_t *q, const uint16_t *k,
                              const uint16_t *v, uint32_t seq, uint32_t heads, float scale, bool head_major) {
    const SmallArgs a{out, q, k, v, seq, heads, scale * 1.4426950408889634f, head_major ? 1 : 0, g->fault};
    return blocks == 2 ? launch<2>(g, a) : launch<1>(g, a);
}
