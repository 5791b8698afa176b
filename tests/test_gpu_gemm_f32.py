"""The f32-path quantized GEMM (tl_qtensor_matmul past four rows) at the edges of its tiles and
K ranges, against 64-bit sums over the oracle's exact dequantization; rows with infinities, NaN,
zeros and extreme magnitudes; and the form without a workspace it falls back to."""
import ctypes as C

import numpy as np
import pytest

import oracle
from tl_amd import GGML_Q4_0, GGML_Q4_K, GGML_Q6_K, GGML_Q8_0, QTensor, _lib
from tl_amd.llama import HipLlama, LlamaConfig, synthetic_prompt, synthetic_weights
from tl_amd.quant import random_q4_0_blocks, random_q4_k_blocks, random_q6_k_blocks, random_q8_0_blocks

pytestmark = pytest.mark.gpu

GEN = {GGML_Q4_0: random_q4_0_blocks, GGML_Q8_0: random_q8_0_blocks, GGML_Q4_K: random_q4_k_blocks,
       GGML_Q6_K: random_q6_k_blocks}


def bound(t, x, w, nb):
    """Per output: 2^-23 for X's two halves, one f32 rounding per unit and per term of its sum
    (each at most 2^-24 of the running magnitude), over the magnitudes that are added: |x| . |w|,
    and at most three times that for Q4_K, whose values are formed as d (q - o) + (d o - m)."""
    terms = 3 if t == GGML_Q4_K else 1
    return (2.0 ** -23 + (nb + 40) * 2.0 ** -24) * terms * (np.abs(x) @ np.abs(w).T) + 1e-37


@pytest.mark.parametrize("t", [GGML_Q4_0, GGML_Q8_0, GGML_Q4_K, GGML_Q6_K])
@pytest.mark.parametrize("m,n,k", [(5, 3, 256), (16, 129, 768), (17, 1000, 512), (33, 63, 1280), (64, 2049, 2048),
                                   (65, 130, 5632), (128, 250, 256), (200, 11008, 256), (301, 65, 4352),
                                   (512, 11264, 512), (129, 257, 34816)])
def test_gemm_f32_edges(dev, t, m, n, k):
    rng = np.random.default_rng(0x71590000 + m + n + k + t)
    raw = GEN[t](rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    y = dev.tl_qtensor_matmul(dev.tensor_new(x), QTensor(t, raw, (n, k))).to_numpy().astype(np.float64)
    w = oracle.dequantize(t, raw, n * k).reshape(n, k).astype(np.float64)
    assert np.all(np.abs(y - x.astype(np.float64) @ w.T) <= bound(t, x.astype(np.float64), w, k // 32))


@pytest.mark.parametrize("t", [GGML_Q4_0, GGML_Q8_0])
@pytest.mark.parametrize("k", [32, 96, 224, 1056])  # 1, 3, 7 and 33 units: iterations of 2 and 4 end inside
@pytest.mark.parametrize("m", [5, 20, 70])
def test_gemm_f32_odd_units(dev, t, k, m):
    rng = np.random.default_rng(0x71590400 + m + k + t)
    raw = GEN[t](rng, 77, k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    y = dev.tl_qtensor_matmul(dev.tensor_new(x), QTensor(t, raw, (77, k))).to_numpy().astype(np.float64)
    w = oracle.dequantize(t, raw, 77 * k).reshape(77, k).astype(np.float64)
    assert np.all(np.abs(y - x.astype(np.float64) @ w.T) <= bound(t, x.astype(np.float64), w, k // 32))


@pytest.mark.parametrize("t", [GGML_Q4_0, GGML_Q8_0, GGML_Q4_K, GGML_Q6_K])
@pytest.mark.parametrize("m", [7, 40, 130])
def test_gemm_f32_row_magnitudes(dev, t, m):
    """Rows are scaled one by one: each row's error is bounded by its own entries, from
    subnormal rows to rows near the f32 maximum; a row of zeros gives zeros, and a row with an
    infinity or NaN the products of a plain f32 sum."""
    n, k = 100, 1024
    rng = np.random.default_rng(0x71590800 + m + t)
    raw = GEN[t](rng, n, k)
    w = oracle.dequantize(t, raw, n * k).reshape(n, k).astype(np.float64)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[1] *= np.float32(1e-38)
    x[2] *= np.float32(1e34)
    x[3] = 0
    x[4, 5::7] *= np.float32(1e6)   # outliers over small entries
    bad = x.copy()
    bad[0, 17] = np.inf
    bad[5, 40] = np.nan
    bad[6, 3], bad[6, 900] = -np.inf, np.inf
    for a in (x, bad):
        q = QTensor(t, raw, (n, k))
        y = dev.tl_qtensor_matmul(dev.tensor_new(a), q).to_numpy()
        ok = np.isfinite(a).all(axis=1)
        a64 = a[ok].astype(np.float64)
        assert np.all(np.abs(y[ok].astype(np.float64) - a64 @ w.T) <= bound(t, a64, w, k // 32))
        assert not y[3].any()
        ref = oracle.qtensor_matmul(a, raw, t, n)
        assert np.array_equal(np.isnan(y), np.isnan(ref)) and np.array_equal(np.isinf(y), np.isinf(ref))
        assert np.array_equal(np.sign(y[np.isinf(ref)]), np.sign(ref[np.isinf(ref)]))


def zero_first_of_blocks(t, raw, n):
    """The same blocks with the first weight of each exactly 0."""
    b = raw.reshape(n, -1, {GGML_Q4_0: 18, GGML_Q8_0: 34, GGML_Q4_K: 144, GGML_Q6_K: 210}[t]).copy()
    if t == GGML_Q4_0:
        b[..., 2] = (b[..., 2] & 0xF0) | 8
    elif t == GGML_Q8_0:
        b[..., 2] = 0
    elif t == GGML_Q4_K:  # dmin = d, sub-block 0: scale 8, minimum 8 * 7, nibble 7
        b[..., 2:4] = b[..., 0:2]
        b[..., 4] = (b[..., 4] & 0xC0) | 8
        b[..., 8] = (b[..., 8] & 0xC0) | 56
        b[..., 16] = (b[..., 16] & 0xF0) | 7
    else:
        b[..., 0] &= 0xF0
        b[..., 128] = (b[..., 128] & 0xFC) | 2
    return b.reshape(raw.shape)


@pytest.mark.parametrize("t", [GGML_Q4_0, GGML_Q8_0, GGML_Q4_K, GGML_Q6_K])
@pytest.mark.parametrize("ratio", [1e5, 1e7, 1e8, 1e10, 1e12, 1e30])
@pytest.mark.parametrize("m", [7, 40, 130])
def test_gemm_f32_outliers_under_zero_weights(dev, t, ratio, m):
    """An entry far above the rest of its row whose weights are exactly 0 takes nothing from the
    precision of the others: the bound is over |x| . |w|, to which it adds nothing."""
    n, k = 70, 2048
    rng = np.random.default_rng(0x71590a00 + m + t + int(np.log10(ratio)))
    raw = zero_first_of_blocks(t, GEN[t](rng, n, k), n)
    w = oracle.dequantize(t, raw, n * k).reshape(n, k).astype(np.float64)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[:, 512] = np.float32(ratio) * np.where(np.arange(m) % 2, -1.0, 1.7).astype(np.float32)
    assert not w[:, 512].any()
    y = dev.tl_qtensor_matmul(dev.tensor_new(x), QTensor(t, raw, (n, k))).to_numpy().astype(np.float64)
    assert np.all(np.abs(y - x.astype(np.float64) @ w.T) <= bound(t, x.astype(np.float64), w, k // 32))


@pytest.mark.parametrize("t", [GGML_Q4_0, GGML_Q8_0, GGML_Q4_K, GGML_Q6_K])
@pytest.mark.parametrize("small", [1, 16, 17, 400])  # 16 such entries of a row are added one by one
@pytest.mark.parametrize("m,n,k", [(7, 70, 2048), (70, 200, 16384), (512, 11264, 768)])  # one K range, several; the widest tile
def test_gemm_f32_few_entries_far_below(dev, t, small, m, n, k):
    """Rows of zeros but for `small` entries of N(0, 1) and one of 2^40 or 2^-40 under zero weights
    (rows of the second kind lose nothing); the same bits from every call."""
    rng = np.random.default_rng(0x71590b00 + m + t + small)
    raw = zero_first_of_blocks(t, GEN[t](rng, n, k), n)
    w = oracle.dequantize(t, raw, n * k).reshape(n, k).astype(np.float64)
    x = np.zeros((m, k), np.float32)
    for r in range(m):
        at = rng.choice(k, small, replace=False)
        x[r, at] = rng.standard_normal(small)
        x[r, 512] = 2.0 ** (40 if r % 3 else -40)
    assert not w[:, 512].any()
    xt, q = dev.tensor_new(x), QTensor(t, raw, (n, k))
    y = dev.tl_qtensor_matmul(xt, q).to_numpy()
    assert np.all(np.abs(y - x.astype(np.float64) @ w.T) <= bound(t, x.astype(np.float64), w, k // 32))
    for _ in range(2):
        assert np.array_equal(dev.tl_qtensor_matmul(xt, q).to_numpy(), y)


@pytest.mark.parametrize("t", [GGML_Q4_0, GGML_Q4_K])
def test_gemm_f32_without_workspace(dev, t):
    """No memory for a workspace, or a call under capture: the plain FMA form, with the same
    bits from both and from every replay, as tl_hip_launch_quant_gemm_noalloc gives."""
    lib = _lib.load()
    hip = C.CDLL("libamdhip64.so.7")
    m, n, k = 24, 300, 1024
    rng = np.random.default_rng(0x71590c00 + t)
    raw = GEN[t](rng, n, k)
    w = QTensor(t, raw, (n, k))
    hw = w.upload(lib)
    x = rng.standard_normal((m, k)).astype(np.float32)
    xt, yt = dev.tensor_new(x), dev.tensor_new(np.full((m, n), np.nan, np.float32))
    stream = C.c_void_p(lib.tl_hip_stream())
    args = (hw, C.c_void_p(xt.data_ptr), C.c_void_p(yt.data_ptr), m, 0, stream)
    dev.synchronize()
    lib.tl_hip_debug_fail_alloc(0)
    try:
        rc = lib.tl_hip_launch_quant_gemm(*args)
    finally:
        lib.tl_hip_debug_fail_alloc(-1)
    assert rc == 0
    plain = yt.to_numpy()
    ref = oracle.qtensor_matmul(x, raw, t, n)
    assert float(np.max(np.abs(plain - ref)) / np.max(np.abs(ref))) <= 1e-4
    assert lib.tl_hip_launch_quant_gemm_noalloc(*args) == 0
    assert np.array_equal(yt.to_numpy(), plain)
    graph, gexec = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 1) == 0
    rc = lib.tl_hip_launch_quant_gemm(*args)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert rc == 0, lib.tl_hip_last_error()
    assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, C.c_size_t(0)) == 0
    nan = np.full((m, n), np.nan, np.float32)
    try:
        for _ in range(3):
            assert lib.tl_hip_memcpy_h2d(C.c_void_p(yt.data_ptr), nan.ctypes.data_as(C.c_void_p), nan.nbytes) == 0
            assert hip.hipGraphLaunch(gexec, stream) == 0
            assert hip.hipStreamSynchronize(stream) == 0
            assert np.array_equal(yt.to_numpy(), plain)
            assert lib.tl_hip_launch_quant_gemm(*args) == 0  # eager work between replays
            dev.synchronize()
    finally:
        hip.hipGraphExecDestroy(gexec)
        hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("t,f16", [(GGML_Q4_0, False), (GGML_Q8_0, False), (GGML_Q4_K, False), (GGML_Q6_K, False),
                                   (GGML_Q6_K, True)])
@pytest.mark.parametrize("m", [5, 16, 32, 64])
@pytest.mark.parametrize("n,k", [(1024, 768), (260, 11008), (2048, 2048)])
def test_gemm_one_launch_merge(dev, t, m, n, k, f16):
    """K slices added by a tile's last-arriving split (2 .. 16 of them) and by a launch of its own:
    the same order, so the same bits, call after call (the arrival counters return to zero)."""
    lib = _lib.load()
    rng = np.random.default_rng(0x71590e00 + m + n + k + t)
    q = QTensor(t, GEN[t](rng, n, k), (n, k))
    x = dev.tensor_new(rng.standard_normal((m, k)).astype(np.float32))
    run = lambda: (dev.tl_qtensor_matmul_f16 if f16 else dev.tl_qtensor_matmul)(x, q).to_numpy()  # noqa: E731
    prev = lib.tl_hip_debug_one_launch_merge(1)
    try:
        one = [run() for _ in range(3)]
        lib.tl_hip_debug_one_launch_merge(0)
        two = run()
    finally:
        lib.tl_hip_debug_one_launch_merge(prev)
    assert np.isfinite(two).all()
    for y in one:
        assert np.array_equal(y, two)


@pytest.mark.parametrize("t,f16", [(GGML_Q4_0, False), (GGML_Q4_K, False), (GGML_Q6_K, False), (GGML_Q6_K, True)])
def test_prefill_one_launch_merge(t, f16):
    """The same with a residual: the decoder's o and down projections add into the rows they read."""
    cfg = LlamaConfig(2, 512, 8, 4, 1536, 512, max_seq=128)
    lib = _lib.load()
    m = HipLlama(cfg, kv_f16=f16)
    m.load(list(synthetic_weights(cfg, 41, ggml_type=t)), ggml_type=t)
    for n in (16, 32, 64):
        prompt = synthetic_prompt(cfg, 41, n)
        got = []
        prev = lib.tl_hip_debug_one_launch_merge(1)
        try:
            for on in (1, 1, 0):
                lib.tl_hip_debug_one_launch_merge(on)
                m.reset()
                got.append(m.forward(prompt, prefill_f16=f16))
        finally:
            lib.tl_hip_debug_one_launch_merge(prev)
        assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    m.close()


@pytest.mark.parametrize("t", [GGML_Q4_0, GGML_Q8_0, GGML_Q4_K, GGML_Q6_K])
def test_prefill_gemm_without_workspace(t):
    """Each of a layer's four f32 GEMMs in turn (RMSNorm rows, a residual, RMSNorm rows, SwiGLU rows
    with a residual) finds no memory for its workspace: rows formed in memory and the plain FMA
    form, within the f32 class of an undisturbed prefill."""
    cfg = LlamaConfig(1, 512, 8, 4, 768, 512, max_seq=64)
    lib = _lib.load()
    m = HipLlama(cfg)
    m.load(list(synthetic_weights(cfg, 43, ggml_type=t)), ggml_type=t)
    prompt = synthetic_prompt(cfg, 43, 21)
    want = m.forward(prompt)  # grows the activation buffers
    for i in range(4):
        m.reset()
        lib.tl_hip_debug_fail_alloc(i)
        try:
            got = m.forward(prompt)
        finally:
            lib.tl_hip_debug_fail_alloc(-1)
        assert 0 < float(np.max(np.abs(got - want)) / np.max(np.abs(want))) <= 1e-4, i
    m.reset()
    assert np.array_equal(m.forward(prompt), want)
    m.close()
