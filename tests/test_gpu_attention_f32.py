"""The matrix-instruction form of f32 attention at the edges of its row blocks, position tiles
and head sizes: the scaled-dot-product-attention operator against 64-bit arithmetic, and the
decoder's f32 prefill (causal, f32 and f16 caches, chunked prompts) against the oracle."""
import ctypes as C

import numpy as np
import pytest

import oracle
from tl_amd import _lib
from tl_amd.llama import SLOTS, HipLlama, LlamaConfig, synthetic_prompt, synthetic_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slices,sq,sk,dk,dv,mask", [
    (1, 1, 1, 4, 4, None), (3, 1, 129, 64, 64, None), (2, 16, 128, 64, 8, "random"), (5, 17, 63, 32, 64, "causal"),
    (2, 65, 257, 60, 36, "random"), (1, 15, 1000, 128, 128, None), (4, 33, 65, 128, 20, "random"),
    (40, 225, 90, 64, 64, "causal"), (64, 129, 66, 80, 128, "short"), (300, 64, 96, 128, 96, "causal"),
    # more slices than CUs over few rows: row blocks without rows
    (300, 1, 70, 64, 64, None), (270, 17, 130, 48, 64, "causal"), (300, 16, 65, 128, 128, "random"),
    (280, 33, 70, 96, 128, None), (600, 1, 130, 128, 128, "random"), (520, 17, 70, 100, 72, "causal"),
])
def test_sdpa_row_blocks_and_tiles(dev, slices, sq, sk, dk, dv, mask):
    rng = np.random.default_rng(0x715a0000 + slices + sq + sk + dk + dv)
    q, k, v = (rng.standard_normal((slices, a, b)).astype(np.float32) for a, b in ((sq, dk), (sk, dk), (sk, dv)))
    m, keep = None, np.ones((sq, sk), bool)
    if mask == "causal":
        keep = np.tril(keep, sk - sq) if sk >= sq else np.tril(keep)
        m = keep.astype(np.float32)
    elif mask == "random":
        keep = rng.random((sq, sk)) > 0.3
        m = np.where(keep, 2.0, 0.0).astype(np.float32)
    elif mask == "short":  # entries past the mask's end leave their scores alone
        m = (rng.random(sq * sk // 2 + 1) > 0.5).astype(np.float32)
        keep.reshape(-1)[:m.size] = m != 0
    t = dev.tensor_new
    got = dev.tensor_scaled_dot_product_attention(t(q), t(k), t(v), t(m) if m is not None else None).to_numpy()
    q, k, v = (a.astype(np.float64) for a in (q, k, v))
    s = np.where(keep, q @ k.transpose(0, 2, 1) / np.sqrt(dk), -1e9)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    # a score is off by at most dk + 2 roundings of its terms' magnitudes, a weight by twice that
    # relatively, and each sum over the keys by sk more
    es = (dk + 2) * 2.0 ** -24 * (np.abs(q) @ np.abs(k).transpose(0, 2, 1)).max(-1, keepdims=True) / np.sqrt(dk)
    assert np.all(np.abs(got - p @ v) <= (2 * es + (2 * sk + 16) * 2.0 ** -24) * (p @ np.abs(v)) + 1e-37)


def test_sdpa_as_many_slices_as_a_grid_takes(dev):
    """2^23 slices of one row: 512 threads each would be a grid of 2^32.  One key: the value itself."""
    v = np.arange(4 << 23, dtype=np.float32).reshape(1 << 23, 1, 4)
    q = dev.tensor_new(np.ones_like(v))
    assert np.array_equal(dev.tensor_scaled_dot_product_attention(q, q, dev.tensor_new(v)).to_numpy(), v)


def test_sdpa_special_values(dev):
    """Infinite and NaN scores, and NaN values under a zero weight, as the operator defines them."""
    rng = np.random.default_rng(0x715a0100)
    q, k, v = (rng.standard_normal((2, 70, 64)).astype(np.float32) for _ in range(3))
    k[0, 3] = np.inf          # slice 0: +-inf or NaN scores
    q[1, 5] = np.nan
    k[1, 66, 0] = -np.inf     # slice 1: one key at +-inf by the sign of q
    ref = oracle.sdpa(q, k, v, None)
    t = dev.tensor_new
    got = dev.tensor_scaled_dot_product_attention(t(q), t(k), t(v)).to_numpy()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert ok.any() and np.max(np.abs(got[ok] - ref[ok])) <= 1e-5


@pytest.mark.parametrize("heads,kv,hd", [(4, 2, 64), (8, 1, 64), (4, 4, 64), (2, 2, 128), (8, 2, 128)])
@pytest.mark.parametrize("kv_f16", [False, True])
def test_f32_prefill(heads, kv, hd, kv_f16):
    """Prompts from position 0 against the oracle (whose scale is the chatbot's 0.125, so at head
    size 64); chunks at later positions (row blocks of every size, ends inside tiles) against
    the same tokens one at a time, which take the decode attention."""
    cfg = LlamaConfig(2, heads * hd, heads, kv, 512, 500, max_seq=384)
    tensors = list(synthetic_weights(cfg, 23))
    gpu = HipLlama(cfg, kv_f16=kv_f16)
    gpu.load(tensors)
    prompt = synthetic_prompt(cfg, 23, 330)
    err = lambda a, b: float(np.max(np.abs(a - b)) / np.max(np.abs(b)))  # noqa: E731
    if hd == 64:
        cpu = oracle.Llama(cfg)
        cpu.load(tensors)
    for n in (5, 66, 330) if hd == 64 else ():
        gpu.reset()
        cpu.reset()
        assert err(gpu.forward(prompt[:n]), cpu.forward(prompt[:n])) <= (1e-2 if kv_f16 else 1e-4), n
    gpu.configure(kv_f16, rope_per_token=True)
    one = [gpu.forward(prompt[i:i + 1]) for i in range(200)]
    gpu.reset()
    at = 0
    for n in (5, 61, 130):
        a = gpu.forward(prompt[at:at + n])
        at += n
        assert err(a, one[at - 1]) <= (1e-3 if kv_f16 else 1e-4), at
    gpu.close()


@pytest.mark.parametrize("d,ffn", [(256, 12544), (512, 256), (12544, 256)])
def test_f32_prefill_forms_rows_in_the_gemm(d, ffn):
    """RMSNorm and SwiGLU formed where the GEMM splits its input: rows held in registers and
    rows past 12288 elements, against one token at a time."""
    cfg = LlamaConfig(1, d, d // 64, d // 256, ffn, 256, max_seq=64)
    gpu = HipLlama(cfg, kv_f16=False)
    gpu.configure(False, rope_per_token=True)
    gpu.load(list(synthetic_weights(cfg, 29)))
    prompt = synthetic_prompt(cfg, 29, 37)
    want = [gpu.forward(prompt[i:i + 1]) for i in range(37)][-1]
    gpu.reset()
    got = gpu.forward(prompt)
    assert float(np.max(np.abs(got - want)) / np.max(np.abs(want))) <= 1e-4
    gpu.close()


@pytest.mark.parametrize("which,value", [("embedding", np.inf), ("embedding", 1e30), ("norm", 1e25)])
def test_f32_prefill_special_rows(which, value):
    """A row that is or becomes infinite or NaN (an infinite embedding; a SwiGLU past f32's range),
    or whose sum of squares overflows, goes through as it does one token at a time."""
    cfg = LlamaConfig(2, 512, 8, 4, 512, 256, max_seq=64)
    prompt = synthetic_prompt(cfg, 31, 9)
    tensors = [list(t) for t in synthetic_weights(cfg, 31)]
    for t in tensors:
        if which == t[0] == "embedding":
            i = next(i for i, a in enumerate(t) if isinstance(a, np.ndarray))
            t[i] = t[i].copy()
            t[i].reshape(-1, 512)[prompt[-1], :3 if np.isinf(value) else 512] = value
        elif which == "norm" and t[:3] == ["norm", 0, 1]:
            i = next(i for i, a in enumerate(t) if isinstance(a, np.ndarray))
            t[i] = t[i] * np.float32(value)
    gpu = HipLlama(cfg, kv_f16=False)
    gpu.configure(False, rope_per_token=True)
    gpu.load([tuple(t) for t in tensors])
    want = [gpu.forward(prompt[i:i + 1]) for i in range(9)][-1]
    gpu.reset()
    got = gpu.forward(prompt)
    assert np.isnan(want).all() if value != 1e30 else np.isfinite(want).all()
    assert np.array_equal(got, want, equal_nan=True) if value == 1e30 else np.isnan(got).all()
    gpu.close()


def test_f32_prefill_wide_rows():
    """RMSNorm and SwiGLU rows with one entry 1e12 above the rest, whose weights are zero:
    nothing of the others is lost."""
    cfg = LlamaConfig(1, 512, 8, 4, 768, 256, max_seq=64)
    gate, up, down = 4, 5, 6
    tensors = [list(t) for t in synthetic_weights(cfg, 37)]
    for t in tensors:
        if t[0] == "norm" and t[1] == 0:
            t[3] = t[3].copy()
            t[3][0] *= np.float32(1e12)
        elif t[0] == "linear" and t[1] == 0:
            b = t[3].copy().reshape(cfg.linear_shape(SLOTS[t[2]])[0], -1, 18)  # Q4_0 blocks of each row
            b[:, 0, 2] = (b[:, 0, 2] & 0xF0) | 8  # column 0: zero
            if t[2] in (gate, up):  # SwiGLU's entry 0: scales of 30000 against about 0.01
                b[0, :, :2] = np.float16(30000).reshape(1).view(np.uint8)
            t[3] = b.reshape(-1)
    assert SLOTS[gate] == "ffn_gate" and SLOTS[up] == "ffn_up" and SLOTS[down] == "ffn_down"
    prompt = synthetic_prompt(cfg, 37, 21)
    cpu = oracle.Llama(cfg)
    cpu.load([tuple(t) for t in tensors])
    want = cpu.forward(prompt)
    gpu = HipLlama(cfg, kv_f16=False)
    gpu.load([tuple(t) for t in tensors])
    got = gpu.forward(prompt)
    gpu.close()
    assert np.isfinite(want).all()
    assert float(np.max(np.abs(got - want)) / np.max(np.abs(want))) <= 1e-4


# tlhip::launch_attention_prefill_f32: the public entries show the last row only, which attends all
PREFILL_F32 = "_ZN5tlhip28launch_attention_prefill_f32EPKfPKvS3_iPfiiiilPKifP12ihipStream_t"


@pytest.mark.parametrize("n,pos,hq,hkv,d", [(37, 0, 4, 2, 64), (5, 70, 4, 4, 64), (200, 33, 64, 8, 64),
                                            (70, 0, 4, 1, 128), (130, 9, 32, 32, 128)])
@pytest.mark.parametrize("kv_f16", [False, True])
def test_f32_prefill_stops_at_a_rows_own_position(dev, n, pos, hq, hkv, d, kv_f16):
    """Values (and keys) of later tokens that are infinite or NaN reach no earlier row."""
    rng = np.random.default_rng(0x715a0300 + n + pos + d)
    lmax, kt = pos + n + 3, np.float16 if kv_f16 else np.float32
    q = rng.standard_normal((n, hq, d)).astype(np.float32)
    k, v = (rng.standard_normal((hkv, lmax, d)).astype(kt) for _ in range(2))
    k[:, pos + n:] = v[:, pos + n:] = np.nan          # not written yet
    v[0, pos + n - 2, 3], v[-1, pos + n - 1] = np.inf, np.nan
    k[0, pos + n - 1, 0] = np.nan
    v[0, pos + n // 2, d - 1] = -np.inf
    new = dev.tensor_new_f16 if kv_f16 else dev.tensor_new
    qt, kd, vd, out = dev.tensor_new(q), new(k), new(v), dev.tensor_new(np.zeros((n, hq, d), np.float32))
    at = dev.tensor_new(np.array([pos], np.int32).view(np.float32))
    lib = _lib.load()
    f = lib[PREFILL_F32]
    f.restype, p = C.c_int, C.c_void_p
    f.argtypes = [p, p, p, C.c_int, p, C.c_int, C.c_int, C.c_int, C.c_int, C.c_int64, p, C.c_float, p]
    assert f(qt.data_ptr, kd.data_ptr, vd.data_ptr, 1 if kv_f16 else 0, out.data_ptr, n, hq, hkv, d, lmax, at.data_ptr,
             1 / np.sqrt(d), lib.tl_hip_stream()) == 0
    got = out.to_numpy()
    q, k, v = (a.astype(np.float64) for a in (q, k, v))
    with np.errstate(invalid="ignore"):
        for i in range(n):
            for h in range(hq):
                kh, vh = k[h * hkv // hq, :pos + i + 1], v[h * hkv // hq, :pos + i + 1]
                s = kh @ q[i, h] / np.sqrt(d)
                w = np.exp(s - s.max())
                w /= w.sum()
                want, mag = w @ vh, w @ np.abs(vh)
                assert np.array_equal(np.isnan(got[i, h]), np.isnan(want)), (i, h)
                ok = np.isfinite(want)
                assert np.array_equal(got[i, h][~ok & ~np.isnan(want)], want[~ok & ~np.isnan(want)].astype(np.float32))
                es = (d + 2) * 2.0 ** -24 * (np.abs(kh) @ np.abs(q[i, h])).max() / np.sqrt(d)
                assert np.all(np.abs(got[i, h] - want)[ok] <= (2 * es + (2 * len(s) + 16) * 2.0 ** -24) * mag[ok] + 1e-37)
