"""DiT block operators on the GPU vs the CPU oracle: BF16 and W8A16 projections,
fused GELU, AdaLN, gates, Q/K norm + RoPE, activations and Euler."""
import ctypes as C
import math
import os
import tempfile

import numpy as np
import pytest

from h3cli_amd import synth
from h3cli_amd._lib import GpuStats
from h3cli_amd.runtime import Gpu
from oracle import oracle
from tests.helpers import GEMM_REL_L2, bf16, metrics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    g = Gpu()
    yield g
    g.close()


def ulp_diff(a, b, floor=2.0 ** -17):
    """|a - b| in units of the BF16 ulp at the larger magnitude of the pair, with
    the ulp floored at `floor`: outputs that cancel to near zero (fma(x, 1+scale,
    shift) with x*(1+scale) ~ -shift) inherit the absolute error of the O(1) terms,
    not the tiny ulp of the result."""
    fa, fb = bf16(a).astype(np.float64), bf16(b).astype(np.float64)
    mag = np.maximum(np.maximum(np.abs(fa), np.abs(fb)), 2.0 ** -126)
    ulp = np.maximum(2.0 ** (np.floor(np.log2(mag)) - 7), floor)
    return np.abs(fa - fb) / ulp


def run(gpu, fn, *args):
    gpu.begin()
    ok = fn(gpu.handle, *args)
    if not ok:
        err = gpu.error()
        gpu.cancel()
        raise RuntimeError(err)
    gpu.submit()


def q8_weight(gpu, codes, scales, n, k, group):
    c = np.ascontiguousarray(codes, np.int8)
    s = np.ascontiguousarray(scales, np.float32)
    h = gpu.lib.h3_hip_q8_from_packed(gpu.handle, c.ctypes.data, s.ctypes.data, n, k, group)
    assert h, gpu.error()
    from h3cli_amd.runtime import Tensor
    t = Tensor(gpu, h, n * k, 2)
    gpu.tensors.append(t)
    return t


def synthetic_q8(seed, n, k, group):
    """BASELINE config 4 weights: int8 uniform in [-127, 127], per-output-channel
    (group = k) or per-group fp32 scales uniform in [1e-3, 1e-2]."""
    rng = np.random.default_rng(seed)
    codes = rng.integers(-127, 128, size=n * k, dtype=np.int8)
    scales = rng.uniform(1e-3, 1e-2, size=n * ((k + group - 1) // group)).astype(np.float32)
    return codes, scales


@pytest.mark.parametrize("m,k,n,group,bias,gelu", [
    (300, 512, 256, 512, False, False),     # per-channel, ragged M
    (513, 1024, 512, 64, True, False),      # reference q8 recipe (group 64) + bias
    (256, 768, 768, 768, False, True),      # fused GELU-tanh epilogue
    (33, 256, 256, 256, False, False),      # M smaller than a tile
    (300, 1024, 512, 1024, True, False),    # split tiles, bias epilogue
    (300, 1024, 512, 1024, True, True),     # split tiles, bias + GELU-tanh epilogue
    (50, 100, 30, 100, True, False),        # unaligned shape: small-GEMM path
])
def test_w8a16_linear(gpu, m, k, n, group, bias, gelu):
    print(f"[w8a16] m={m} k={k} n={n} group={group} bias={bias} gelu={gelu}", flush=True)
    codes, scales = synthetic_q8(m + n, n, k, group)
    x = synth.normal_bf16(m * 3 + 1, m * k)
    b = synth.normal_bf16(7, n, scale=0.1) if bias else None
    w = q8_weight(gpu, codes, scales, n, k, group)
    tx, ty = gpu.from_bf16(x), gpu.empty(m * n)
    tb = gpu.from_bf16(b) if bias else None
    fn = gpu.lib.h3_hip_linear_gelu_bf16 if gelu else gpu.lib.h3_gpu_linear_bf16
    run(gpu, fn, ty.handle, tx.handle, w.handle, tb.handle if tb else None, m, k, n)
    got = ty.read()
    ref, ref64 = oracle.linear_q8(x, codes, scales, m, k, n, group, bias=b, gelu=gelu)
    met = metrics(bf16(got), ref64)
    assert met["rel_l2"] <= GEMM_REL_L2, met
    # Reference gate for its q8 kernel (tests/metal_q8.c:156).
    assert met["rel_l2"] < 0.006, met
    # Nearly every element equals the FP64 reference rounded to BF16.
    assert np.mean(ulp_diff(got, ref) <= 1) > 0.99


@pytest.mark.parametrize("m,k,n,group,bias,gelu", [
    (1, 64, 16, 0, False, False),       # one K step: seven of the eight waves have none
    (2, 576, 30, 0, True, False),       # nine steps, a ragged column block
    (16, 320, 8200, 0, False, True),    # the most rows of one row block
    (17, 2176, 48, 0, True, True),      # two row blocks, 34 steps
    (32, 192, 8200, 0, True, False),    # four column blocks per workgroup, the last one ragged
    (5, 640, 37, 16, False, False),     # W8A16, smallest scale group
    (16, 320, 8200, 64, True, False),   # W8A16, two column blocks per workgroup
    (31, 1088, 8200, 1088, False, True),
])
def test_few_rows_linear(gpu, m, k, n, group, bias, gelu):
    """At most 32 rows against FP64: one BF16 rounding (two with the GELU) of the
    result plus the FP32 sum's k 2^-24 sum |x w|."""
    print(f"[few rows] m={m} k={k} n={n} group={group} bias={bias} gelu={gelu}", flush=True)
    x = synth.normal_bf16(m + 3, m * k)
    b = synth.normal_bf16(7, n, scale=0.1) if bias else None
    if group:
        codes, scales = synthetic_q8(m + n, n, k, group)
        w = q8_weight(gpu, codes, scales, n, k, group)
        wide = np.repeat(scales.reshape(n, -1), group, axis=1)[:, :k]
        wv = bf16(synth.f32_to_bf16(codes.reshape(n, k).astype(np.float32) * wide)).astype(np.float64)
    else:
        bits = synth.normal_bf16(m + 4, n * k, scale=1 / math.sqrt(k))
        w, wv = gpu.from_bf16(bits), bf16(bits).reshape(n, k).astype(np.float64)
    tx, tb, out = gpu.from_bf16(x), gpu.from_bf16(b) if bias else None, gpu.empty(m * n)
    fn = gpu.lib.h3_hip_linear_gelu_bf16 if gelu else gpu.lib.h3_gpu_linear_bf16
    run(gpu, fn, out.handle, tx.handle, w.handle, tb.handle if bias else None, m, k, n)
    got = bf16(out.read()).reshape(m, n).astype(np.float64)
    xv = bf16(x).reshape(m, k).astype(np.float64)
    want = xv @ wv.T + (bf16(b).astype(np.float64) if bias else 0.0)
    bound = 2.0 ** -8 * np.abs(want) + k * 2.0 ** -24 * (np.abs(xv) @ np.abs(wv).T)
    if gelu:
        # |gelu'| <= 1.13; the second rounding, and the hardware exp and reciprocal.
        want = 0.5 * want * (1 + np.tanh(math.sqrt(2 / math.pi) * (want + 0.044715 * want ** 3)))
        bound = 1.13 * bound + 2.0 ** -8 * np.abs(want) + 2.0 ** -20
    assert np.all(np.abs(got - want) <= bound), float(np.max(np.abs(got - want) / bound))
    for t in (tx, out, w) + ((tb,) if bias else ()):
        gpu.free(t)


@pytest.mark.parametrize("m,k,n,q8,bias,gelu", [
    (600, 4096, 512, False, False, False),    # six tiles, all split; the last row tile ragged
    (600, 4224, 512, True, True, True),       # 33 stage pairs in uneven shares, every epilogue
    (33, 2048, 256, False, True, False),      # one tile of 33 rows
    (300, 1024, 33280, False, False, False),  # 260 tiles: 256 whole ones and four split ones
])
def test_linear_split_over_k(gpu, m, k, n, q8, bias, gelu):
    """Tiles of an incomplete wave, whose K shares a second launch adds, against
    FP64 within the bound of test_few_rows_linear."""
    print(f"[split K] m={m} k={k} n={n} q8={q8} bias={bias} gelu={gelu}", flush=True)
    x = synth.normal_bf16(m + 3, m * k)
    b = synth.normal_bf16(7, n, scale=0.1) if bias else None
    if q8:
        codes, scales = synthetic_q8(m + n, n, k, k)
        w = q8_weight(gpu, codes, scales, n, k, k)
        wv = bf16(synth.f32_to_bf16(codes.reshape(n, k).astype(np.float32) * scales[:, None]))
    else:
        bits = synth.normal_bf16(m + 4, n * k, scale=1 / math.sqrt(k))
        w, wv = gpu.from_bf16(bits), bf16(bits).reshape(n, k)
    tx, tb, out = gpu.from_bf16(x), gpu.from_bf16(b) if bias else None, gpu.empty(m * n)
    fn = gpu.lib.h3_hip_linear_gelu_bf16 if gelu else gpu.lib.h3_gpu_linear_bf16
    run(gpu, fn, out.handle, tx.handle, w.handle, tb.handle if bias else None, m, k, n)
    got = bf16(out.read()).reshape(m, n)
    rows = np.unique(np.concatenate([np.arange(0, m, 37), [m - 1, min(255, m - 1), min(256, m - 1)]]))
    xv = bf16(x).reshape(m, k)[rows].astype(np.float64)
    for at in range(0, n, 4096):
        wt = wv[at:at + 4096].astype(np.float64)
        want = xv @ wt.T + (bf16(b)[at:at + 4096].astype(np.float64) if bias else 0.0)
        bound = 2.0 ** -8 * np.abs(want) + k * 2.0 ** -24 * (np.abs(xv) @ np.abs(wt).T)
        if gelu:
            want = 0.5 * want * (1 + np.tanh(math.sqrt(2 / math.pi) * (want + 0.044715 * want ** 3)))
            bound = 1.13 * bound + 2.0 ** -8 * np.abs(want) + 2.0 ** -20
        assert np.all(np.abs(got[rows, at:at + 4096] - want) <= bound)
    for t in (tx, out, w) + ((tb,) if bias else ()):
        gpu.free(t)


@pytest.mark.parametrize("m,k", [(2, 8), (20, 4)])
def test_any_shape_linear_of_many_columns(gpu, m, k):
    """More blocks of columns than the second and third grid dimensions hold (65535)."""
    n = 64 * 65536 + 33
    print(f"[many columns] m={m} k={k} n={n}", flush=True)
    x, w = synth.normal_bf16(m, m * k), synth.normal_bf16(m + 1, n * k)
    tx, tw, out = gpu.from_bf16(x), gpu.from_bf16(w), gpu.empty(m * n)
    run(gpu, gpu.lib.h3_gpu_linear_bf16, out.handle, tx.handle, tw.handle, None, m, k, n)
    assert gpu.last_kernel() == "gemm_small"
    cols = np.r_[0:n:9973, n - 70:n]
    xv, wv = bf16(x).reshape(m, k).astype(np.float64), bf16(w).reshape(n, k)[cols].astype(np.float64)
    want = xv @ wv.T
    bound = 2.0 ** -8 * np.abs(want) + k * 2.0 ** -24 * (np.abs(xv) @ np.abs(wv).T)
    assert np.all(np.abs(bf16(out.read()).reshape(m, n)[:, cols] - want) <= bound)
    for t in (tx, tw, out):
        gpu.free(t)


def test_large_q8_weight_is_not_converted(gpu):
    """A weight of 2 GiB or more in BF16 is multiplied from its codes, however many rows
    would pay for the conversion: the context keeps no buffer of that size."""
    m, k, n, group = 12288, 8256, 131072, 64
    print(f"[large q8] m={m} k={k} n={n}", flush=True)
    tx, out = gpu.empty(m * k), gpu.empty(m * n)
    w = gpu.lib.h3_hip_q8_new(gpu.handle, n, k, group)
    run(gpu, gpu.lib.h3_hip_fill_normal_bf16, tx.handle, 3, C.c_float(1.0), m * k)
    run(gpu, gpu.lib.h3_hip_fill_q8_random, w, 5, C.c_float(1e-4), C.c_float(3e-4))
    run(gpu, gpu.lib.h3_gpu_linear_bf16, out.handle, tx.handle, w, None, m, k, n)
    assert gpu.last_kernel().startswith("gemm_mid rows=256") and "converted" not in gpu.last_kernel()
    cols = np.r_[0:n:16381, n - 2:n].astype(np.uint64)
    base, kk = np.uint64(5 << 40), np.arange(k, dtype=np.uint64)
    codes = (synth.splitmix64(base + cols[:, None] * np.uint64(k) + kk) % np.uint64(255)).astype(np.float32) - 127
    at = cols[:, None] * np.uint64(k // group) + np.arange(k // group, dtype=np.uint64)
    unit = (synth.splitmix64(base + np.uint64(1 << 39) + at) >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
    scales = (1e-4 + 2e-4 * unit).astype(np.float32)
    wv = bf16(synth.f32_to_bf16((codes * np.repeat(scales, group, axis=1)).reshape(-1))).reshape(len(cols), k)
    xv = bf16(tx.read(k)).astype(np.float64)
    want = wv.astype(np.float64) @ xv
    # One BF16 rounding, the FP32 sum, and weights whose scale differs in the last place.
    bound = 2.0 ** -8 * np.abs(want) + k * 2.0 ** -24 * (np.abs(wv) @ np.abs(xv)) + 2.0 ** -8 * np.sqrt((wv ** 2) @ (xv ** 2))
    assert np.all(np.abs(bf16(out.read(n))[cols.astype(np.int64)] - want) <= bound)
    gpu.lib.h3_gpu_tensor_free(w)
    for t in (tx, out):
        gpu.free(t)


@pytest.mark.parametrize("m,k,n,group,bias,gelu", [
    (17, 64, 30, 0, False, False),        # one K step, a ragged column tile of odd width
    (64, 1088, 256, 0, True, False),      # 17 steps, split
    (65, 128, 300, 64, True, True),       # W8A16, two steps, one row past a 64-row tile
    (64, 2176, 512, 16, False, False),    # W8A16, smallest scale group
    (129, 640, 4096, 640, False, True),   # W8A16 per channel
    (300, 1088, 2562, 64, True, False),   # width not a multiple of four
    (513, 2112, 768, 2112, False, False), # K of 64 only
    (1000, 192, 90, 0, False, False),     # many rows, few columns
])
def test_mid_rows_linear(gpu, m, k, n, group, bias, gelu):
    """Row tiles of 64 to 256 and their remainders against FP64, bound as in
    test_few_rows_linear."""
    test_few_rows_linear(gpu, m, k, n, group, bias, gelu)


PIPE_WHOLE, PIPE_SPLIT = (2255, 128, 3840), (1690, 256, 9472)     # 135 and 256 + 3 tiles, ragged rows


@pytest.mark.parametrize("m,k,n,group,bias,gelu,kernel", [
    *[(*shape, 0, bias, gelu, kernel)
      for shape, kernel in ((PIPE_WHOLE, "gemm_bf16_pipe"), (PIPE_SPLIT, "gemm_bf16_pipe shares=2"))
      for bias in (False, True) for gelu in (False, True)],
    (600, 7168, 5376, 0, True, True, "gemm_bf16_pipe shares=4"),              # no whole wave
    (8400, 4096, 16128, 0, False, False, "gemm_bf16_pipe shares=4"),          # 31 tiles behind eight waves
    (1163, 128, 8192, 64, True, True, "gemm_bf16_pipe converted"),
    (2786, 512, 6144, 64, True, False, "gemm_bf16_pipe shares=4 converted"),
    (1076, 128, 7424, 128, False, True, "gemm_bf16_pipe converted"),
    (3316, 256, 4928, 0, True, True, "gemm_mid rows=256 shares=4"),
    (8571, 64, 817, 0, True, False, "gemm_mid rows=256"),                     # odd width, one K step
    (960, 6080, 2578, 6080, False, True, "gemm_mid rows=256 shares=5"),
    (303, 192, 30464, 192, True, False, "gemm_mid rows=256"),
    (748, 5824, 2825, 64, True, True, "gemm_mid rows=256 shares=7"),          # odd width
    (309, 192, 32256, 64, False, False, "gemm_mid rows=256"),
    (1458, 64, 5478, 64, True, True, "gemm_mid rows=256 converted"),
    (729, 5376, 28672, 64, False, False, "gemm_mid rows=256 shares=3"),
    (1275, 4096, 1545, 0, True, False, "gemm_mid rows=128 shares=3"),
    (2976, 64, 1408, 0, False, True, "gemm_mid rows=128"),
    (589, 3968, 2176, 3968, True, True, "gemm_mid rows=128 shares=5"),
    (1244, 64, 3254, 64, True, False, "gemm_mid rows=128"),
    (210, 2240, 5632, 64, False, False, "gemm_mid rows=128 shares=5"),
    (1242, 128, 3324, 64, True, True, "gemm_mid rows=128"),
    (81, 192, 64, 0, True, True, "gemm_mid rows=64 shares=3"),
    (179, 64, 30, 0, True, False, "gemm_mid rows=64"),
    (296, 128, 43, 128, True, False, "gemm_mid rows=64 shares=2"),
    (51, 320, 62, 64, False, True, "gemm_mid rows=64 shares=5"),
    (75, 128, 5720, 64, True, True, "gemm_mid rows=64"),
    (755, 2304, 5504, 2304, True, True, "gemm_q8_pipe shares=3"),
    (653, 960, 11264, 960, False, False, "gemm_q8_pipe"),
])
def test_linear_plans(gpu, m, k, n, group, bias, gelu, kernel):
    """Each kernel of many rows with whole and split tiles, each weight format and epilogue,
    and that it is the one that ran; bound as in test_few_rows_linear, rows at the edges of
    tiles and between."""
    print(f"[plans] m={m} k={k} n={n} group={group} bias={bias} gelu={gelu} {kernel}", flush=True)
    x = synth.normal_bf16(m + 3, m * k)
    b = synth.normal_bf16(7, n, scale=0.1) if bias else None
    if group:
        codes, scales = synthetic_q8(m + n, n, k, group)
        w = q8_weight(gpu, codes, scales, n, k, group)
    else:
        bits = synth.normal_bf16(m + 4, n * k, scale=1 / math.sqrt(k))
        w = gpu.from_bf16(bits)
    tx, tb, out = gpu.from_bf16(x), gpu.from_bf16(b) if bias else None, gpu.empty(m * n)
    fn = gpu.lib.h3_hip_linear_gelu_bf16 if gelu else gpu.lib.h3_gpu_linear_bf16
    run(gpu, fn, out.handle, tx.handle, w.handle, tb.handle if bias else None, m, k, n)
    assert gpu.last_kernel() == kernel
    edges = np.arange(64, m, 64)
    rows = np.unique(np.r_[0:m:max(1, m // 16), edges[:8], edges[:8] - 1, edges[-2:], edges[-2:] - 1, m - 1])
    got = bf16(out.read().reshape(m, n)[rows])
    xv = bf16(x.reshape(m, k)[rows]).astype(np.float64)
    for at in range(0, n, 4096):
        cols = slice(at, min(at + 4096, n))
        if group:
            wide = np.repeat(scales.reshape(n, -1)[cols], group, axis=1)[:, :k]
            wt = bf16(synth.f32_to_bf16(codes.reshape(n, k)[cols].astype(np.float32) * wide)).astype(np.float64)
        else:
            wt = bf16(bits.reshape(n, k)[cols]).astype(np.float64)
        want = xv @ wt.T + (bf16(b)[cols].astype(np.float64) if bias else 0.0)
        bound = 2.0 ** -8 * np.abs(want) + k * 2.0 ** -24 * (np.abs(xv) @ np.abs(wt).T)
        if gelu:
            want = 0.5 * want * (1 + np.tanh(math.sqrt(2 / math.pi) * (want + 0.044715 * want ** 3)))
            bound = 1.13 * bound + 2.0 ** -8 * np.abs(want) + 2.0 ** -20
        assert np.all(np.abs(got[:, cols] - want) <= bound), float(np.max(np.abs(got[:, cols] - want) / bound))
    for t in (tx, out, w) + ((tb,) if bias else ()):
        gpu.free(t)


@pytest.mark.parametrize("m,k,hidden,group,kernel", [
    (2255, 128, 1920, 0, "gemm_bf16_pipe"),
    (1690, 256, 4736, 0, "gemm_bf16_pipe shares=2"),
    (1163, 128, 4096, 64, "gemm_bf16_pipe converted"),
    (3316, 256, 2464, 0, "gemm_mid rows=256 shares=4"),          # gate and up rows ragged
    (309, 192, 16128, 64, "gemm_mid rows=256"),
    (1242, 128, 1662, 64, "gemm_mid rows=128"),                  # an even hidden width, not a multiple of four
    (653, 960, 5632, 960, "gemm_q8_pipe"),
    (755, 2304, 2752, 2304, "gemm_q8_pipe shares=3"),
])
def test_mlp_plans(gpu, m, k, hidden, group, kernel):
    """SwiGLU in the epilogue of each kernel, as test_mlp. The kernel of fc1, chosen by its
    sizes, is that of a projection of the same sizes."""
    tx, out = gpu.empty(m * k), gpu.empty(m * 2 * hidden)
    w = q8_weight(gpu, *synthetic_q8(1, 2 * hidden, k, group), 2 * hidden, k, group) if group else gpu.empty(2 * hidden * k)
    for t in (tx,) if group else (tx, w):
        run(gpu, gpu.lib.h3_hip_fill_normal_bf16, t.handle, 3, C.c_float(1.0), t.elements)
    run(gpu, gpu.lib.h3_gpu_linear_bf16, out.handle, tx.handle, w.handle, None, m, k, 2 * hidden)
    assert gpu.last_kernel() == kernel
    for t in (tx, out, w):
        gpu.free(t)
    test_mlp(gpu, m, k, hidden, 64, group)


@pytest.mark.parametrize("m,k,hidden,n,group", [
    (300, 512, 384, 256, 0),       # SwiGLU in fc1's epilogue, a ragged row tile
    (600, 4096, 256, 512, 4096),   # the same from split tiles, W8A16
    (33, 256, 128, 256, 64),       # one tile: 128 gate and 128 up rows
    (20, 320, 128, 192, 0),        # few rows: separate SwiGLU
    (70, 100, 30, 50, 0),          # unaligned
    (100, 640, 100, 64, 64),       # SwiGLU over 200 weight rows: gate and up rows ragged
    (200, 2048, 512, 300, 64),     # the same from split tiles, W8A16
])
def test_mlp(gpu, m, k, hidden, n, group):
    """fc1 -> SwiGLU -> fc2 against FP64. Gate, up, the activation and the result
    are rounded to BF16 once each (2^-9 relative at most, |silu'| <= 1.1), so the
    2-norms differ by at most about 4 * 2^-9."""
    print(f"[mlp] m={m} k={k} hidden={hidden} n={n} group={group}", flush=True)
    x = synth.normal_bf16(m + 5, m * k)
    ws, wv = [], []
    for seed, rows, cols in ((1, 2 * hidden, k), (2, n, hidden)):
        if group:
            gr = min(group, cols)
            codes, scales = synthetic_q8(m + seed, rows, cols, gr)
            scales /= 3 * math.sqrt(cols) / 10
            ws.append(q8_weight(gpu, codes, scales, rows, cols, gr))
            wide = np.repeat(scales.reshape(rows, -1), gr, axis=1)[:, :cols]
            wv.append(bf16(synth.f32_to_bf16(codes.reshape(rows, cols).astype(np.float32) * wide)).astype(np.float64))
        else:
            bits = synth.normal_bf16(m + seed, rows * cols, scale=1 / math.sqrt(cols))
            ws.append(gpu.from_bf16(bits))
            wv.append(bf16(bits).reshape(rows, cols).astype(np.float64))
    tx, out = gpu.from_bf16(x), gpu.empty(m * n)
    for _ in range(2):   # the second call finds the workspace in use by the first
        run(gpu, gpu.lib.h3_gpu_mlp_bf16, out.handle, tx.handle, ws[0].handle, ws[1].handle, m, k, hidden, n)
    got = bf16(out.read()).reshape(m, n)
    both = bf16(x).reshape(m, k).astype(np.float64) @ wv[0].T
    gate, up = both[:, :hidden], both[:, hidden:]
    want = (gate / (1 + np.exp(-gate)) * up) @ wv[1].T
    met = metrics(got, want)
    assert met["rel_l2"] <= 4 * 2.0 ** -9, met
    for t in (tx, out, *ws):
        gpu.free(t)


@pytest.mark.parametrize("m,k,hidden", [(64, 64, 64), (2255, 128, 1920), (653, 960, 5632)])
def test_mlp_gates_near_the_end_of_exp(gpu, m, k, hidden):
    """silu(gate) * up where 1 / (1 + exp(-gate)) is below the normal FP32 range and the
    product with a large up is not, in the mid, pipe and q8 kernels' epilogues: one input
    value, gates of one column each, ups of 2^100 and an fc2 that copies the first columns."""
    print(f"[mlp gates] m={m} k={k} hidden={hidden}", flush=True)
    gates = np.array([-60.0, -86.5, -87.0, -87.5, -88.0, -88.5, -1.0, 80.0], np.float32)
    x, w1, w2 = np.zeros((m, k), np.float32), np.zeros((2 * hidden, k), np.float32), np.zeros((64, hidden), np.float32)
    x[:, 0] = 1
    w1[:8, 0], w1[hidden:hidden + 8, 0] = gates, 2.0 ** 100
    w2[np.arange(8), np.arange(8)] = 1
    if hidden == 5632:      # codes of one scale per column
        scales = np.ones(2 * hidden, np.float32)
        scales[:8], scales[hidden:] = 0.5, 2.0 ** 100
        codes = np.zeros((2 * hidden, k), np.int8)
        gates = np.clip(gates, -63.5, 63.5)       # 127 codes of 0.5
        scales[1:6] = np.array([86.5, 87.0, 87.5, 88.0, 88.5], np.float32) / 100
        codes[:8, 0] = np.round(gates / 0.5)
        codes[1:6, 0] = -100
        codes[hidden:hidden + 8, 0] = 1
        t1 = q8_weight(gpu, codes.reshape(-1), scales, 2 * hidden, k, k)
        gates = bf16(synth.f32_to_bf16((codes[:8, 0] * scales[:8]).astype(np.float32)))
    else:
        t1 = gpu.from_bf16(synth.f32_to_bf16(w1.reshape(-1)))
    tx, t2, out = gpu.from_bf16(synth.f32_to_bf16(x.reshape(-1))), gpu.from_bf16(synth.f32_to_bf16(w2.reshape(-1))), gpu.empty(m * 64)
    run(gpu, gpu.lib.h3_gpu_mlp_bf16, out.handle, tx.handle, t1.handle, t2.handle, m, k, hidden, 64)
    got = bf16(out.read()).reshape(m, 64)[:, :8].astype(np.float64)
    gates = gates.astype(np.float64)
    want = gates / (1 + np.exp(-gates)) * 2.0 ** 100
    # One BF16 rounding of the activation, copied by fc2.
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want)), got[0] / want
    for t in (tx, t1, t2, out):
        gpu.free(t)


def test_mlp_in_parts():
    """More rows than the kept workspace holds (1 GiB of activated rows): parts of the
    rows, bit for bit what a call on a part's rows gives, with no tensor allocated in any
    call, and in place in both directions."""
    m, k, hidden, n, part = 16640, 64, 32768, 128, 8448
    print(f"[mlp parts] m={m} k={k} hidden={hidden} n={n}", flush=True)
    x = synth.normal_bf16(1, m * k)
    bits = [synth.normal_bf16(2, 2 * hidden * k, scale=1 / math.sqrt(k)),
            synth.normal_bf16(3, n * hidden, scale=1 / math.sqrt(hidden)),
            synth.normal_bf16(4, k // 2 * hidden, scale=1 / math.sqrt(hidden))]
    with Gpu() as gpu:
        tx, out, few = gpu.from_bf16(x), gpu.empty(m * n), gpu.empty(part * n)
        w1, w2, narrow = (gpu.from_bf16(b) for b in bits)
        place = gpu.empty(m * n)
        before, after = GpuStats(), GpuStats()
        gpu.lib.h3_gpu_get_stats(gpu.handle, C.byref(before))
        run(gpu, gpu.lib.h3_gpu_mlp_bf16, out.handle, tx.handle, w1.handle, w2.handle, m, k, hidden, n)
        got = out.read().reshape(m, n)
        for first in (0, part):
            rows = min(part, m - first)
            tp = gpu.from_bf16(x.reshape(m, k)[first:first + rows])
            run(gpu, gpu.lib.h3_gpu_mlp_bf16, few.handle, tp.handle, w1.handle, w2.handle, rows, k, hidden, n)
            assert np.array_equal(few.read(rows * n).reshape(rows, n), got[first:first + rows])
        rows = np.r_[0:m:997, part - 1, part, m - 1]
        xv, wv = bf16(x).reshape(m, k)[rows].astype(np.float64), [bf16(b).astype(np.float64) for b in bits]
        both = xv @ wv[0].reshape(-1, k).T
        want = (both[:, :hidden] / (1 + np.exp(-both[:, :hidden])) * both[:, hidden:]) @ wv[1].reshape(n, hidden).T
        met = metrics(bf16(got[rows]), want)
        assert met["rel_l2"] <= 4 * 2.0 ** -9, met
        # In place: wider output (last part first) and narrower output.
        for w, width in ((w2, n), (narrow, k // 2)):
            run(gpu, gpu.lib.h3_gpu_mlp_bf16, out.handle, tx.handle, w1.handle, w.handle, m, k, hidden, width)
            place_rows = np.zeros(m * n, np.uint16)
            place_rows[:m * k] = x
            gpu.check(gpu.lib.h3_gpu_tensor_write_bf16(place.handle, place_rows.ctypes.data, m * n), "write")
            run(gpu, gpu.lib.h3_gpu_mlp_bf16, place.handle, place.handle, w1.handle, w.handle, m, k, hidden, width)
            assert np.array_equal(place.read(m * width), out.read(m * width))
        gpu.lib.h3_gpu_get_stats(gpu.handle, C.byref(after))
        assert after.tensor_allocations - before.tensor_allocations == 2    # tp, twice


@pytest.mark.parametrize("m,k,n,hidden,bias,gelu", [
    (1000, 1472, 16192, 0, True, True),   # an odd K tile count, a quarter column tile
    (500, 1792, 32768, 0, True, False),   # an even one, a row tile of 244 rows
    (520, 4160, 8256, 0, False, True),    # 65 K tiles in two shares, 8 rows of the last row tile
    (513, 2112, 192, 9664, False, False), # SwiGLU, one row and half a column tile past whole ones
    (520, 4160, 128, 4128, False, False), # SwiGLU from split tiles, a quarter column tile
])
def test_per_channel_q8(gpu, m, k, n, hidden, bias, gelu):
    """W8A16 with one scale per channel, at sizes that convert the codes inside the
    hand-scheduled K loop; bounds as in test_few_rows_linear and test_mlp."""
    if hidden:
        test_mlp(gpu, m, k, hidden, n, k)
    else:
        test_few_rows_linear(gpu, m, k, n, k, bias, gelu)


def test_bf16_linear_exact_pattern(gpu):
    """tests/quant_native.c:31-50 power-of-two pattern: the BF16 GEMM output must
    equal bf16(exact sum) bit for bit, for several row counts."""
    n, k = 256, 256
    j = np.arange(n)[:, None]
    c = np.arange(k)[None, :]
    w = synth.f32_to_bf16(np.ldexp(1.0, (j % 3) - 1 + (c // 16) % 3).astype(np.float32))
    for rows in (1, 17, 129, 300):
        r = np.arange(rows)[:, None]
        x = synth.f32_to_bf16((np.where(r % 2, -1.0, 1.0) * np.ldexp(1.0, (r % 3) - 1 + (c // 16) % 2)).astype(np.float32))
        tw, tx, ty = gpu.from_bf16(w), gpu.from_bf16(x), gpu.empty(rows * n)
        run(gpu, gpu.lib.h3_gpu_linear_bf16, ty.handle, tx.handle, tw.handle, None, rows, k, n)
        exact = synth.bf16_to_f32(x).astype(np.float64) @ synth.bf16_to_f32(w).astype(np.float64).T
        assert np.array_equal(ty.read(), synth.f32_to_bf16(exact.astype(np.float32)).reshape(-1)), rows


def test_bf16_linear_random(gpu):
    m, k, n = 700, 1024, 512
    x = synth.normal_bf16(1, m * k)
    w = synth.normal_bf16(2, n * k, scale=0.03)
    tw, tx, ty = gpu.from_bf16(w), gpu.from_bf16(x), gpu.empty(m * n)
    run(gpu, gpu.lib.h3_gpu_linear_bf16, ty.handle, tx.handle, tw.handle, None, m, k, n)
    _, ref64 = oracle.linear_bf16(x, w, m, k, n)
    assert metrics(bf16(ty.read()), ref64)["rel_l2"] < 5e-3


def test_q8_load_from_file(gpu):
    """h3_gpu_q8_load packs BF16 weights from a file with the reference recipe."""
    n, k, m = 256, 320, 40
    w = synth.normal_bf16(3, n * k, scale=0.125)
    with tempfile.NamedTemporaryFile(delete=False) as f:
        f.write(b"\0" * 6 + w.tobytes())
        path = f.name
    try:
        h = gpu.lib.h3_gpu_q8_load(gpu.handle, path.encode(), 6, n, k)
        assert h, gpu.error()
        from h3cli_amd.runtime import Tensor
        t = Tensor(gpu, h, n * k, 2)
        gpu.tensors.append(t)
        x = synth.normal_bf16(4, m * k)
        tx, ty = gpu.from_bf16(x), gpu.empty(m * n)
        run(gpu, gpu.lib.h3_gpu_linear_bf16, ty.handle, tx.handle, t.handle, None, m, k, n)
        codes, scales = oracle.q8_pack(w, n, k, 64)
        _, ref64 = oracle.linear_q8(x, codes, scales, m, k, n, 64)
        assert metrics(bf16(ty.read()), ref64)["rel_l2"] < 0.006
    finally:
        os.unlink(path)


def test_q8_load_device_pack_bit_exact(gpu):
    """The device packer of h3_gpu_q8_load gives the codes and scales of the
    reference recipe bit for bit (vs the oracle and the host h3_q8_pack_rows):
    exact half ties, an all-zero group, a ragged last group (200 columns =
    64+64+64+8), large and tiny magnitudes. A NaN weight is rejected."""
    import ctypes as C
    n, k = 67, 200
    rng = np.random.default_rng(8)
    w = rng.standard_normal((n, k)).astype(np.float32)
    w[0, :64] = 0.0                                    # all-zero group -> scale 1
    w[1, :64] = np.arange(64) - 31.5                   # ties after scaling by 127/amax
    w[2] *= 1e30
    w[3] *= 1e-30
    w[4, 192:] = [127, -127, 63.5, -63.5, 0.5, -0.5, 1.5, 2.5]
    wb = synth.f32_to_bf16(w).reshape(-1)
    with tempfile.NamedTemporaryFile(delete=False) as f:
        f.write(b"\0" * 10 + wb.tobytes())
        path = f.name
    try:
        h = gpu.lib.h3_gpu_q8_load(gpu.handle, path.encode(), 10, n, k)
        assert h, gpu.error()
        from h3cli_amd.runtime import Tensor
        t = Tensor(gpu, h, n * k, 2)
        gpu.tensors.append(t)
        groups = (k + 63) // 64
        raw = np.zeros(n * k + n * groups * 4, np.uint8)
        assert gpu.lib.h3_hip_tensor_copy_to_host(h, raw.ctypes.data, raw.size), gpu.error()
        codes, scales = raw[:n * k].view(np.int8), raw[n * k:].view(np.float32)
        ref_codes, ref_scales = oracle.q8_pack(wb, n, k, 64)
        assert np.array_equal(codes, ref_codes) and np.array_equal(scales.view(np.uint32), ref_scales.view(np.uint32))
        host_codes, host_scales = np.zeros(n * k, np.int8), np.zeros(n * groups, np.float32)
        gpu.lib.h3_q8_pack_rows.restype = C.c_int
        assert gpu.lib.h3_q8_pack_rows(C.c_void_p(wb.ctypes.data), C.c_void_p(host_codes.ctypes.data),
                                       C.c_void_p(host_scales.ctypes.data), C.c_uint32(n), C.c_uint32(k))
        assert np.array_equal(codes, host_codes) and np.array_equal(scales, host_scales)
        bad = wb.copy()
        bad[5 * k + 7] = 0x7FC0
        with open(path, "r+b") as f:
            f.seek(10)
            f.write(bad.tobytes())
        assert not gpu.lib.h3_gpu_q8_load(gpu.handle, path.encode(), 10, n, k)
        assert "non-finite" in gpu.error()
    finally:
        os.unlink(path)


def test_linear_contract_errors(gpu):
    w = gpu.from_bf16(np.zeros(256 * 256, np.uint16))
    x = gpu.from_bf16(np.zeros(4 * 256, np.uint16))
    y = gpu.empty(4 * 256)
    gpu.begin()
    assert not gpu.lib.h3_gpu_linear_bf16(gpu.handle, y.handle, x.handle, w.handle, None, 4, 256, 257)
    assert not gpu.lib.h3_gpu_linear_bf16(gpu.handle, x.handle, x.handle, w.handle, None, 4, 256, 256)
    gpu.submit()


def modulation(seed, rows_map, slots, width):
    return synth.normal_bf16(seed, rows_map * slots * width, scale=0.3)


@pytest.mark.parametrize("rows,width", [(37, 512), (300, 5120), (5, 8192)])
def test_adaln(gpu, rows, width):
    x = synth.normal_bf16(rows, rows * width, scale=2.0)
    w = synth.normal_bf16(9, width, scale=0.5)
    mod = modulation(11, 3, 6, width)
    rmap = (np.arange(rows) % 3).astype(np.uint32)
    tx, tw, tm, tr, ty = gpu.from_bf16(x), gpu.from_bf16(w), gpu.from_bf16(mod), gpu.from_u32(rmap), gpu.empty(rows * width)
    run(gpu, gpu.lib.h3_gpu_adaln_bf16, ty.handle, tx.handle, tw.handle, tm.handle, tr.handle, rows, width, 6, 0, 1,
        C.c_float(1e-6))
    ref = oracle.adaln(x, w, mod, rmap, rows, width, 6, 0, 1, 1e-6)
    d = ulp_diff(ty.read(), ref)
    assert d.max() <= 1 and d.mean() < 0.02


@pytest.mark.parametrize("rows,width", [
    (1, 4096), (2048, 4104), (3, 6152),   # a workgroup per row: whole chunks, one left over
    (2049, 5376), (3, 4088),              # a wave per row: one row more, one chunk less
])
def test_adaln_row_split(gpu, rows, width):
    test_adaln(gpu, rows, width)


def test_gate_and_gate_adaln(gpu):
    rows, width = 129, 5120
    res = synth.normal_bf16(1, rows * width)
    br = synth.normal_bf16(2, rows * width)
    w = synth.normal_bf16(3, width, scale=0.5)
    mod = modulation(4, 2, 6, width)
    rmap = (np.arange(rows) >= 100).astype(np.uint32)
    t = {n: gpu.from_bf16(a) for n, a in (("res", res), ("br", br), ("w", w), ("mod", mod))}
    tr = gpu.from_u32(rmap)
    out, gated, norm = gpu.empty(rows * width), gpu.empty(rows * width), gpu.empty(rows * width)
    run(gpu, gpu.lib.h3_gpu_gate_bf16, out.handle, t["res"].handle, t["br"].handle, t["mod"].handle, tr.handle,
        rows, width, 6, 2)
    ref_gate = oracle.gate(res, br, mod, rmap, rows, width, 6, 2)
    assert np.array_equal(out.read(), ref_gate)
    run(gpu, gpu.lib.h3_gpu_gate_adaln_bf16, gated.handle, norm.handle, t["res"].handle, t["br"].handle,
        t["w"].handle, t["mod"].handle, t["mod"].handle, tr.handle, rows, width, 6, 2, 3, 4, C.c_float(1e-6))
    assert np.array_equal(gated.read(), ref_gate)
    ref_norm = oracle.adaln(ref_gate, w, mod, rmap, rows, width, 6, 3, 4, 1e-6)
    assert ulp_diff(norm.read(), ref_norm).max() <= 1


@pytest.mark.parametrize("grouped,norm,half,dim", [(0, False, 64, 128), (1, True, 48, 128), (0, True, 64, 128),
                                                   (1, False, 36, 72)])
def test_qkv_rope(gpu, grouped, norm, half, dim):
    seq, heads = 97, 5
    qkv = synth.normal_bf16(5, seq * heads * dim * 3)
    cos, sin = synth.rope_tables(27, 30, 40)
    cos = synth.f32_to_bf16(cos[:seq, :half].copy()).reshape(-1)
    sin = synth.f32_to_bf16(sin[:seq, :half].copy()).reshape(-1)
    qw = synth.normal_bf16(6, dim, scale=0.5) if norm else None
    kw = synth.normal_bf16(7, dim, scale=0.5) if norm else None
    tq, tk, tv = gpu.empty(seq * heads * dim), gpu.empty(seq * heads * dim), gpu.empty(seq * heads * dim)
    tin, tc, ts = gpu.from_bf16(qkv), gpu.from_bf16(cos), gpu.from_bf16(sin)
    tqw = gpu.from_bf16(qw) if norm else None
    tkw = gpu.from_bf16(kw) if norm else None
    fn = gpu.lib.h3_gpu_grouped_qkv_rope_bf16 if grouped else gpu.lib.h3_gpu_qkv_rope_bf16
    run(gpu, fn, tq.handle, tk.handle, tv.handle, tin.handle, tqw.handle if tqw else None,
        tkw.handle if tkw else None, tc.handle, ts.handle, seq, heads, dim, half, C.c_float(1e-6))
    rq, rk, rv = oracle.qkv_rope(qkv, qw, kw, cos, sin, seq, heads, dim, half, 1e-6, grouped)
    assert np.array_equal(tv.read(), rv)
    assert ulp_diff(tq.read(), rq).max() <= 1 and ulp_diff(tk.read(), rk).max() <= 1


def test_activations_and_euler(gpu):
    n = 100003
    x = synth.normal_bf16(1, n, scale=3.0)
    tx, ty = gpu.from_bf16(x), gpu.empty(n)
    for approx in (1, 0):
        run(gpu, gpu.lib.h3_gpu_gelu_bf16, ty.handle, tx.handle, n, approx)
        assert ulp_diff(ty.read(), oracle.gelu(x, bool(approx))).max() <= 1
    rows, width = 77, 640
    fused = synth.normal_bf16(2, rows * width * 2, scale=2.0)
    tf, to = gpu.from_bf16(fused), gpu.empty(rows * width)
    run(gpu, gpu.lib.h3_gpu_swiglu_bf16, to.handle, tf.handle, rows, width)
    assert ulp_diff(to.read(), oracle.swiglu(fused, rows, width)).max() <= 1
    sample = synth.normal(3, n + 10).astype(np.float32)
    last, prev = synth.normal_bf16(4, n), synth.normal_bf16(5, n)
    ts, tl, tp = gpu.from_f32(sample), gpu.from_bf16(last), gpu.from_bf16(prev)
    run(gpu, gpu.lib.h3_gpu_euler_bf16, ts.handle, C.c_size_t(7), tl.handle, tp.handle, n, C.c_float(-0.05),
        C.c_float(0.25))
    want = sample.copy()
    want[7:7 + n] = oracle.euler(sample[7:7 + n], last, prev, -0.05, 0.25)
    assert np.array_equal(ts.read(), want)


def test_adaln_offset_and_rms_norms(gpu):
    rows, width, off = 45, 1024, 3 * 1024 + 8
    x = synth.normal_bf16(21, off + rows * width, scale=2.0)
    w = synth.normal_bf16(22, width, scale=0.5)
    mod = modulation(23, 2, 6, width)
    rmap = (np.arange(rows) % 2).astype(np.uint32)
    tx, tw, tm, tr, ty = gpu.from_bf16(x), gpu.from_bf16(w), gpu.from_bf16(mod), gpu.from_u32(rmap), gpu.empty(rows * width)
    run(gpu, gpu.lib.h3_gpu_adaln_bf16_offset, ty.handle, tx.handle, off, tw.handle, tm.handle, tr.handle, rows, width,
        6, 3, 4, C.c_float(1e-6))
    ref = oracle.adaln(x[off:], w, mod, rmap, rows, width, 6, 3, 4, 1e-6)
    assert ulp_diff(ty.read(), ref).max() <= 1
    with pytest.raises(RuntimeError):  # offset not a multiple of 8
        run(gpu, gpu.lib.h3_gpu_adaln_bf16_offset, ty.handle, tx.handle, 3, tw.handle, tm.handle, tr.handle, rows,
            width, 6, 3, 4, C.c_float(1e-6))
    run(gpu, gpu.lib.h3_gpu_rms_norm_bf16, ty.handle, tx.handle, tw.handle, rows, width, C.c_float(1e-5))
    assert ulp_diff(ty.read(), oracle.rms_norm(x[:rows * width], w, rows, width, 1e-5)).max() <= 1
    seq, heads, dim = 131, 6, 128
    t = synth.normal_bf16(24, seq * heads * dim, scale=3.0)
    hw = synth.normal_bf16(25, dim, scale=0.5)
    tt, thw = gpu.from_bf16(t), gpu.from_bf16(hw)
    run(gpu, gpu.lib.h3_gpu_head_rms_norm_bf16, tt.handle, thw.handle, seq, heads, dim, C.c_float(1e-6))
    assert ulp_diff(tt.read(), oracle.head_rms_norm(t, hw, seq, heads, dim, 1e-6)).max() <= 1


def test_sub_silu_mul_copy(gpu):
    n = 70001
    a, b = synth.normal_bf16(31, n, scale=3.0), synth.normal_bf16(32, n, scale=3.0)
    ta, tb, to = gpu.from_bf16(a), gpu.from_bf16(b), gpu.empty(n)
    run(gpu, gpu.lib.h3_gpu_sub_bf16, to.handle, ta.handle, tb.handle, n)
    want = synth.f32_to_bf16(bf16(a) - bf16(b))  # one rounding of an exact FP32 difference
    assert np.array_equal(to.read(), want)
    run(gpu, gpu.lib.h3_gpu_silu_mul_bf16, to.handle, ta.handle, tb.handle, n)
    fa = bf16(a).astype(np.float64)
    ref = synth.f32_to_bf16((fa / (1 + np.exp(-fa)) * bf16(b)).astype(np.float32))
    assert ulp_diff(to.read(), ref).max() <= 1
    dst = gpu.empty(n + 100)
    run(gpu, gpu.lib.h3_gpu_copy_bf16, dst.handle, 100, ta.handle, 5, n - 5)
    assert np.array_equal(dst.read()[100:100 + n - 5], a[5:])
    with pytest.raises(RuntimeError):
        run(gpu, gpu.lib.h3_gpu_copy_bf16, dst.handle, 101, ta.handle, 0, n)  # destination range overflows


@pytest.mark.parametrize("m,k,n,mapped", [(33, 128, 320, False), (200, 48, 5120, False), (70, 100, 130, True)])
def test_patch_linear_bit_exact(gpu, m, k, n, mapped):
    """FP32 patch projection: bit-exact against the ordered-fma restatement."""
    rng = np.random.default_rng(m + k + n)
    x = rng.standard_normal(m * k).astype(np.float32)
    w = (rng.standard_normal(n * k) * 0.1).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    tx, tw, tb = gpu.from_f32(x), gpu.from_f32(w), gpu.from_f32(bias)
    if mapped:
        out_rows = m + 9
        rmap = rng.permutation(out_rows)[:m].astype(np.uint32)
        rmap[3] = out_rows + 4  # out-of-range entries are skipped
        tr = gpu.from_u32(rmap)
        zero = gpu.from_bf16(np.zeros(out_rows * n, np.uint16))
        run(gpu, gpu.lib.h3_gpu_patch_linear_bf16_map, zero.handle, tx.handle, tw.handle, tb.handle, tr.handle,
            out_rows, m, k, n)
        got = zero.read()
        want = oracle.patch_linear(x, w, bias, m, k, n, row_map=rmap, out_rows=out_rows)
    else:
        ty = gpu.empty(m * n)
        run(gpu, gpu.lib.h3_gpu_patch_linear_bf16, ty.handle, tx.handle, tw.handle, tb.handle, m, k, n)
        got = ty.read()
        want = oracle.patch_linear(x, w, bias, m, k, n)
    assert np.array_equal(got, want)


def test_tensor_load_files(gpu):
    vals = synth.normal(41, 1000).astype(np.float32)
    with tempfile.NamedTemporaryFile(delete=False) as f:
        f.write(b"\0" * 12 + vals.tobytes())
        path = f.name
    try:
        h = gpu.lib.h3_gpu_tensor_load_f32(gpu.handle, path.encode(), 12, 1000)
        assert h, gpu.error()
        from h3cli_amd.runtime import Tensor
        t = Tensor(gpu, h, 1000, 0)
        gpu.tensors.append(t)
        assert np.array_equal(t.read(), vals)
        assert not gpu.lib.h3_gpu_tensor_load_f32(gpu.handle, path.encode(), 12, 2000)  # short file
    finally:
        os.unlink(path)
