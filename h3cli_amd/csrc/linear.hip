// Projection entry points of the operator surface: BF16 / W8A16 linear, the
// fused QKV projection + norm/RoPE, the SwiGLU MLP, and q8 weight tensors.
#include "common.h"
#include "internal.h"
#include "gemm.h"
#include <algorithm>
#include <cerrno>
#include <cmath>
#include <fcntl.h>
#include <new>
#include <unistd.h>
#include <vector>

// activation: H3_GEMM_PLAIN, _GELU or (n = 2 * hidden, where it fits) _SWIGLU.
static int linear(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in, const h3_gpu_tensor *w,
                  const h3_gpu_tensor *bias, uint32_t rows, uint32_t k, uint32_t n, int activation) {
    if (!h3_launch_ready(g)) return 0;
    if (!rows || !k || !n || !w || w->owner != g)
        return h3_set_error(g, "linear %ux%ux%u: invalid shape or weight", rows, n, k);
    if (!h3_require(g, in, H3_GPU_BF16, (size_t)rows * k, "linear input") ||
        !h3_require(g, out, H3_GPU_BF16, (size_t)rows * (activation == H3_GEMM_SWIGLU ? n / 2 : n), "linear output") ||
        (bias && !h3_require(g, bias, H3_GPU_BF16, n, "linear bias")))
        return 0;
    if (w->quant_mode) {
        // Reference gpu_cuda.cu:928-930: packed FP8 weights take no bias or epilogue.
        if (bias || activation) return h3_set_error(g, "unsupported quantized projection offset/bias/type");
        if (out == in) return h3_set_error(g, "linear: output aliases input");
        return h3_quant_gemm(g, out, in, w, rows, k, n);
    }
    if (w->q8) {
        if (w->q8_rows != n || w->q8_cols != k)
            return h3_set_error(g, "linear: q8 weight is %ux%u, need %ux%u", w->q8_rows, w->q8_cols, n, k);
    } else if (w->dtype != H3_GPU_BF16 || w->elements < (size_t)n * k) {
        return h3_set_error(g, "linear %ux%ux%u: weight must be BF16 with %zu elements", rows, n, k, (size_t)n * k);
    }
    if (out == in) return h3_set_error(g, "linear: output aliases input");
    return h3_gemm(g, (uint16_t *)out->data, (const uint16_t *)in->data, w,
                   bias ? (const uint16_t *)bias->data : nullptr, rows, k, n, activation);
}

extern "C" int h3_gpu_linear_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in, const h3_gpu_tensor *w,
                                  const h3_gpu_tensor *bias, uint32_t rows, uint32_t k, uint32_t n) {
    return g && linear(g, out, in, w, bias, rows, k, n, H3_GEMM_PLAIN);
}

extern "C" int h3_hip_linear_gelu_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in, const h3_gpu_tensor *w,
                                       const h3_gpu_tensor *bias, uint32_t rows, uint32_t k, uint32_t n) {
    return g && linear(g, out, in, w, bias, rows, k, n, H3_GEMM_GELU);
}

extern "C" int h3_gpu_grouped_qkv_linear_rope_bf16(h3_gpu *g, h3_gpu_tensor *q, h3_gpu_tensor *k, h3_gpu_tensor *v,
                                                   h3_gpu_tensor *qkv, const h3_gpu_tensor *in, const h3_gpu_tensor *w,
                                                   const h3_gpu_tensor *qw, const h3_gpu_tensor *kw,
                                                   const h3_gpu_tensor *c, const h3_gpu_tensor *s, uint32_t rows,
                                                   uint32_t width, uint32_t heads, uint32_t dim, uint32_t half, float eps) {
    return g && h3_gpu_linear_bf16(g, qkv, in, w, nullptr, rows, width, heads * dim * 3) &&
           h3_gpu_grouped_qkv_rope_bf16(g, q, k, v, qkv, qw, kw, c, s, rows, heads, dim, half, eps);
}

// The MLP's intermediates stay in a grow-only workspace of the context: allocating
// and freeing them in each call waits for the GPU (8193 rows, 5376 -> 14336 -> 5376,
// alone: 20.0 ms a call, of which 3.4 ms computing). The context keeps no more than this;
// calls with more rows than it holds run in parts of the rows.
constexpr size_t MLP_WORKSPACE = (size_t)1 << 30;

// A BF16 tensor over workspace memory, for the operators of one call.
static h3_gpu_tensor workspace_tensor(h3_gpu *g, void *data, size_t elements) {
    h3_gpu_tensor t{};
    t.owner = g; t.data = data; t.elements = elements; t.bytes = t.bytes_alloc = elements * 2;
    t.dtype = H3_GPU_BF16; t.storage = H3_GPU_DEVICE_ONLY;
    return t;
}

// Workspace of `rows` rows: the activated rows and, where SwiGLU is not fc1's epilogue, the
// 2 * hidden wide product, each with the slack of h3_gpu_tensor_alloc behind it.
struct MlpPart {
    bool fused;
    size_t act, both;
};
static MlpPart mlp_part(const h3_gpu_tensor *w1, size_t rows, uint32_t width, uint32_t hidden) {
    const bool fused = w1 && !w1->quant_mode && h3_gemm_swiglu_fits(w1, (uint32_t)rows, width, hidden);
    const auto slack = [](size_t bytes) { return (bytes + 511) & ~(size_t)255; };
    return {fused, slack(rows * hidden * 2), fused ? 0 : slack(rows * hidden * 4)};
}

// fc1 (2*hidden, gate rows then up rows) -> SwiGLU -> fc2, as src/cuda/gpu_cuda.cu:1108-1112.
// Where the projection kernel takes it, SwiGLU is fc1's epilogue and the 2 * hidden
// wide product is never written.
extern "C" int h3_gpu_mlp_bf16(h3_gpu *g, h3_gpu_tensor *out, const h3_gpu_tensor *in, const h3_gpu_tensor *w1,
                               const h3_gpu_tensor *w2, uint32_t rows, uint32_t width, uint32_t hidden, uint32_t output_dim) {
    if (!g) return 0;
    // Its intermediates cannot be allocated for a graph, nor may a graph keep the workspace.
    if (h3_capturing(g)) return h3_set_error(g, "MLP: the compute stream is being captured");
    if (!rows || !hidden || hidden > UINT32_MAX / 2 ||
        !h3_require(g, in, H3_GPU_BF16, (size_t)rows * width, "MLP input") ||
        !h3_require(g, out, H3_GPU_BF16, (size_t)rows * output_dim, "MLP output"))
        return rows && hidden && hidden <= UINT32_MAX / 2 ? 0 : h3_set_error(g, "MLP: invalid shape %ux%u", rows, hidden);
    // Parts of whole 256-row tiles, even ones. A packed weight sees all rows at once: the
    // scale of its quantized activations is the tensor's.
    size_t most = rows;
    if (!(w1 && w1->quant_mode) && !(w2 && w2->quant_mode)) {
        const size_t row_bytes = (size_t)hidden * (mlp_part(w1, rows, width, hidden).fused ? 2 : 6);
        most = std::max(MLP_WORKSPACE / row_bytes / 256, (size_t)1) * 256;
    }
    const size_t parts = (rows + most - 1) / most;
    const size_t step = parts == 1 ? rows : ((rows + parts - 1) / parts + 255) / 256 * 256;
    const size_t last = rows - (rows - 1) / step * step;
    const MlpPart a = mlp_part(w1, step, width, hidden), b = mlp_part(w1, last, width, hidden);
    const size_t bytes = std::max(a.act + a.both, b.act + b.both);
    h3_gpu_tensor *own = nullptr;
    char *workspace = nullptr;
    if (bytes <= MLP_WORKSPACE + 1024 && h3_buffer_try(g, &g->mlp_workspace, bytes)) workspace = (char *)g->mlp_workspace.ptr;
    else if ((own = h3_gpu_tensor_new_bf16(g, bytes / 2))) workspace = (char *)own->data;
    int ok = workspace != nullptr;
    // Last part first where the output of a part could reach the input of a later one.
    const bool backward = out->data == in->data && output_dim > width;
    const size_t count = (rows + step - 1) / step;
    for (size_t i = 0; ok && i < count; i++) {
        const size_t first = (backward ? count - 1 - i : i) * step, m = std::min(step, rows - first);
        const MlpPart p = m == step ? a : b;
        h3_gpu_tensor act = workspace_tensor(g, workspace, m * hidden);
        h3_gpu_tensor both = workspace_tensor(g, workspace + p.act, p.fused ? 0 : m * hidden * 2);
        h3_gpu_tensor x = workspace_tensor(g, (uint16_t *)in->data + first * width, m * width);
        h3_gpu_tensor y = workspace_tensor(g, (uint16_t *)out->data + first * output_dim, m * output_dim);
        ok = p.fused ? linear(g, &act, &x, w1, nullptr, (uint32_t)m, width, hidden * 2, H3_GEMM_SWIGLU)
                     : linear(g, &both, &x, w1, nullptr, (uint32_t)m, width, hidden * 2, H3_GEMM_PLAIN) &&
                           h3_gpu_swiglu_bf16(g, &act, &both, (uint32_t)m, hidden);
        ok = ok && linear(g, &y, &act, w2, nullptr, (uint32_t)m, hidden, output_dim, H3_GEMM_PLAIN);
    }
    h3_gpu_tensor_free(own);
    return ok;
}

// ------------------------------------------------------------------ q8 weights
static h3_gpu_tensor *q8_tensor(h3_gpu *g, uint32_t rows, uint32_t cols, uint32_t group) {
    if (!rows || !cols || !group || group > cols) { h3_set_error(g, "q8: invalid %ux%u group %u", rows, cols, group); return nullptr; }
    h3_gpu_tensor *t = h3_gpu_tensor_alloc(g, (size_t)rows * cols, H3_GPU_I8, H3_GPU_DEVICE_ONLY);
    if (!t) return nullptr;
    size_t groups = (cols + group - 1) / group, sbytes = (size_t)rows * groups * 4;
    if (!h3_hip_check(g, hipMalloc(&t->q8_scales, sbytes), "q8 scales")) { t->q8_scales = nullptr; h3_gpu_tensor_free(t); return nullptr; }
    t->q8 = 1; t->q8_rows = rows; t->q8_cols = cols; t->q8_group = group;
    g->stats.q8_weights++;
    g->stats.q8_storage_bytes += t->bytes + sbytes;
    return t;
}

extern "C" h3_gpu_tensor *h3_hip_q8_new(h3_gpu *g, uint32_t rows, uint32_t cols, uint32_t group) {
    return g ? q8_tensor(g, rows, cols, group) : nullptr;
}

extern "C" h3_gpu_tensor *h3_hip_q8_from_packed(h3_gpu *g, const int8_t *codes, const float *scales, uint32_t rows,
                                                uint32_t cols, uint32_t group) {
    if (!g || !codes || !scales) return nullptr;
    h3_gpu_tensor *t = q8_tensor(g, rows, cols, group);
    if (!t) return nullptr;
    size_t groups = (cols + group - 1) / group;
    if (!h3_hip_check(g, hipMemcpy(t->data, codes, (size_t)rows * cols, hipMemcpyHostToDevice), "q8 codes upload") ||
        !h3_hip_check(g, hipMemcpy(t->q8_scales, scales, (size_t)rows * groups * 4, hipMemcpyHostToDevice), "q8 scales upload")) {
        h3_gpu_tensor_free(t);
        return nullptr;
    }
    return t;
}

// Reference q8 packing (src/weights/q8.c:26-56), restated on the device: one
// thread per (row, 64-wide group): scale = max|w| / 127 (IEEE division; 1 for an
// all-zero group, floored at FLT_MIN), code = round-half-to-even(w / scale)
// clamped to +-127. Bit-identical to h3_q8_pack_rows. A non-finite weight sets
// bad[0] (the whole tensor is then rejected, as the reference does).
__global__ __launch_bounds__(256) void q8_pack_kernel(const uint16_t *src, int8_t *codes, float *scales, uint32_t rows,
                                                      uint32_t cols, uint32_t groups, unsigned *bad) {
    const size_t id = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= (size_t)rows * groups) return;
    const uint32_t r = (uint32_t)(id / groups), gi = (uint32_t)(id % groups);
    const uint32_t begin = gi * 64, end = min(begin + 64, cols);
    const uint16_t *row = src + (size_t)r * cols;
    float amax = 0.f;
    bool finite = true;
    for (uint32_t c = begin; c < end; c++) {
        const float w = bf16_to_f32(row[c]);
        finite &= finite_f32(w);
        amax = fmaxf(amax, fabsf(w));
    }
    if (!finite) { bad[0] = 1u; return; }
    const float scale = amax == 0.f ? 1.f : fmaxf(__fdiv_rn(amax, 127.f), 1.17549435e-38f);
    scales[id] = scale;
    int8_t *out = codes + (size_t)r * cols;
    for (uint32_t c = begin; c < end; c++) {
        const float q = rintf(__fdiv_rn(bf16_to_f32(row[c]), scale));
        out[c] = (int8_t)fminf(fmaxf(q, -127.f), 127.f);
    }
}

extern "C" int h3_q8_layout(uint32_t rows, uint32_t columns, size_t *offset, size_t *bytes);

// Reads rows x columns BF16 at `offset` of `path` and packs it on the device.
extern "C" h3_gpu_tensor *h3_gpu_q8_load(h3_gpu *g, const char *path, uint64_t offset, uint32_t rows, uint32_t columns) {
    if (!g || !path || !rows || !columns) return nullptr;
    size_t layout_offset, layout_bytes;
    if (!h3_q8_layout(rows, columns, &layout_offset, &layout_bytes)) {
        h3_set_error(g, "q8 load %s: invalid shape %ux%u", path, rows, columns);
        return nullptr;
    }
    const size_t n = (size_t)rows * columns, groups = (columns + 63) / 64;
    std::vector<uint16_t> src(n);
    int fd = open(path, O_RDONLY | O_CLOEXEC);
    if (fd < 0) { h3_set_error(g, "q8 load %s: %s", path, strerror(errno)); return nullptr; }
    size_t got = 0;
    while (got < n * 2) {
        ssize_t r = pread(fd, (char *)src.data() + got, n * 2 - got, (off_t)(offset + got));
        if (r < 0 && errno == EINTR) continue;
        if (r <= 0) { close(fd); h3_set_error(g, "q8 load %s: short read", path); return nullptr; }
        got += (size_t)r;
    }
    close(fd);
    h3_gpu_tensor *t = q8_tensor(g, rows, columns, 64);
    if (!t) return nullptr;
    void *staging = nullptr;
    const size_t flag_at = (n * 2 + 255) & ~(size_t)255;
    unsigned bad = 0;
    bool ok = h3_hip_check(g, hipMalloc(&staging, flag_at + 4), "q8 load staging") &&
              h3_hip_check(g, hipMemcpy(staging, src.data(), n * 2, hipMemcpyHostToDevice), "q8 load upload") &&
              h3_hip_check(g, hipMemset((char *)staging + flag_at, 0, 4), "q8 load flag");
    if (ok) {
        const size_t threads = (size_t)rows * groups;
        hipLaunchKernelGGL(q8_pack_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, nullptr,
                           (const uint16_t *)staging, (int8_t *)t->data, (float *)t->q8_scales, rows, columns,
                           (uint32_t)groups, (unsigned *)((char *)staging + flag_at));
        ok = h3_hip_check(g, hipGetLastError(), "q8 pack") &&
             h3_hip_check(g, hipMemcpy(&bad, (char *)staging + flag_at, 4, hipMemcpyDeviceToHost), "q8 pack flag");
    }
    if (staging) hipFree(staging);
    if (ok && bad) { h3_set_error(g, "q8 load %s: non-finite weight or invalid shape", path); ok = false; }
    if (!ok) { h3_gpu_tensor_free(t); return nullptr; }
    g->stats.q8_source_bytes += n * 2;
    return t;
}
