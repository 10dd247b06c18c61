"""The block-wise fetch and fp16 append (kv_cache.hip) at the edges of their 8-key blocks: windows
that start and end anywhere in a block, appends that fill, start in and end in one, sources whose
rows are off 16 bytes, outputs off 16 bytes. Bytes are exact: against the whole fetch, the snapshot
tensors (codes dequantized by the oracle) and the appended rows themselves."""
import ctypes

import numpy as np
import pytest

import oracle
from conftest import rng
from test_gpu_kv import _gpu, _np

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("mode", ["affine4", "affine8", "int8", "fp16"])
def test_windows_of_a_fetch(mode, D):
    import qw_amd

    r = rng(D + len(mode))
    k, v = (r.standard_normal((3, 101, D)).astype(np.float16) for _ in range(2))
    c = qw_amd.KVCache(mode, 3, D)
    c.update(_gpu(k), _gpu(v))
    K, V = (_np(x)[0] for x in c.dequantize())
    if mode == "fp16":
        np.testing.assert_array_equal(K, k)
        np.testing.assert_array_equal(V, v)
    elif mode == "int8":
        for got, x in ((K, k), (V, v)):
            np.testing.assert_array_equal(got, oracle.int8_dequantize(*oracle.int8_quantize(x)))
    else:
        bits = int(mode[-1])
        for got, x in ((K, k), (V, v)):
            np.testing.assert_array_equal(got, oracle.affine_dequantize(*oracle.affine_quantize(x, bits), bits))
    for start, n in ((0, 1), (7, 1), (8, 8), (3, 5), (5, 11), (95, 6), (100, 1), (1, 100), (64, 33)):
        a, b = (_np(x)[0] for x in c.dequantize(start, n))
        np.testing.assert_array_equal(a, K[:, start:start + n])
        np.testing.assert_array_equal(b, V[:, start:start + n])


@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("mode", ["affine4", "affine8", "int8", "fp16"])
def test_long_windows_of_a_fetch(mode, D):
    """Windows of 3 n D halves about 1 << 19, the line between a key and a block a thread."""
    import qw_amd

    r, n = rng(D + len(mode)), (1 << 19) // (3 * D)
    k, v = (r.standard_normal((3, n + 30, D)).astype(np.float16) for _ in range(2))
    c = qw_amd.KVCache(mode, 3, D)
    c.update(_gpu(k), _gpu(v))
    K, V = (np.concatenate([_np(c.dequantize(s, min(400, n + 30 - s))[i])[0] for s in range(0, n + 30, 400)], axis=1)
            for i in (0, 1))
    for start, m in ((0, n), (0, n + 1), (3, n + 1), (5, n + 9), (7, n), (29, n + 1), (0, n + 30)):
        a, b = (_np(x)[0] for x in c.dequantize(start, m))
        np.testing.assert_array_equal(a, K[:, start:start + m])
        np.testing.assert_array_equal(b, V[:, start:start + m])


@pytest.mark.parametrize("D", [128, 256])
def test_fp16_appends_around_blocks(D):
    import qw_amd

    r = rng(D)
    k, v = (r.standard_normal((2, 300, D)).astype(np.float16) for _ in range(2))
    c, at = qw_amd.KVCache("fp16", 2, D), 0
    for n in (1, 7, 8, 9, 3, 13, 16, 60, 5, 100, 78):
        c.update(_gpu(k[:, at:at + n]), _gpu(v[:, at:at + n]))
        at += n
    assert at == 300 == c.offset
    K, V = (_np(x)[0] for x in c.dequantize())
    np.testing.assert_array_equal(K, k)
    np.testing.assert_array_equal(V, v)


@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("at,extra,skew", [(0, -1, 0), (0, 0, 0), (8, 5, 0), (3, -1, 0), (3, 0, 0),
                                           (5, 6, 0), (7, 1, 3), (0, 2, 3)])
def test_long_fp16_appends(D, at, extra, skew):
    """About the line to the block-wise form (2 n D halves: 3 << 17 from a block's start, 3 << 18
    from inside one), from and to the middle of blocks; skew: the rows off 16 bytes."""
    import qw_amd

    r, H = rng(D + at + extra), 2
    n = (3 << (18 if at % 8 else 17)) // (H * D) + extra
    k, v = (r.standard_normal((H, at + n, D)).astype(np.float16) for _ in range(2))
    c, L = qw_amd.KVCache("fp16", H, D), qw_amd.lib()
    if at:
        c.update(_gpu(k[:, :at]), _gpu(v[:, :at]))
    src = torch.zeros(2 * H * n * D + skew, dtype=torch.float16, device="cuda:0")
    src[skew:] = _gpu(np.concatenate([k[:, at:].reshape(-1), v[:, at:].reshape(-1)]))
    p = src.data_ptr() + 2 * skew
    assert L.qw_kv_update(c._h, p, p + 2 * H * n * D, n, torch.cuda.current_stream().cuda_stream) == 0
    K, V = (_np(x)[0] for x in c.dequantize())
    np.testing.assert_array_equal(K, k)
    np.testing.assert_array_equal(V, v)


def test_fp16_pointers_off_16_bytes():
    import qw_amd

    r = rng(9)
    H, n, D = 2, 37, 128
    k, v = (r.standard_normal((H, n, D)).astype(np.float16) for _ in range(2))
    src = torch.zeros(2 * H * n * D + 3, dtype=torch.float16, device="cuda:0")
    src[3:3 + H * n * D] = _gpu(k).reshape(-1)
    src[3 + H * n * D:] = _gpu(v).reshape(-1)
    c, L = qw_amd.KVCache("fp16", H, D), qw_amd.lib()
    st = torch.cuda.current_stream().cuda_stream
    p = src.data_ptr()
    assert L.qw_kv_update(c._h, p + 6, p + 6 + 2 * H * n * D, n, st) == 0
    out = torch.zeros(2 * H * n * D + 1, dtype=torch.float16, device="cuda:0")
    p = out.data_ptr()
    assert L.qw_kv_dequantize(c._h, 0, n, p + 2, p + 2 + 2 * H * n * D, ctypes.c_void_p(st)) == 0
    got = out[1:].cpu().numpy().reshape(2, H, n, D)
    np.testing.assert_array_equal(got[0], k)
    np.testing.assert_array_equal(got[1], v)


@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("mode", ["affine4", "affine8"])
@pytest.mark.parametrize("odd", [False, True])
def test_long_affine_append_stores_the_bytes_of_short_ones(mode, D, odd):
    """One append past the block-wise form's line (4 * n * D >= 5 << 18) from the middle of a block
    to the middle of one, against the same rows in short appends: ties, constant, zero, tiny and
    the largest groups; with rows that are not finite as well."""
    import qw_amd

    r, H, n = rng(D + odd), 4, (5 << 18) // (4 * D) + 11
    k, v = (r.standard_normal((H, n, D)).astype(np.float16) for _ in range(2))
    bins = (1 << int(mode[-1])) - 1
    for x in (k, v):
        x[0, 20:60] = (r.integers(0, 2 * bins + 1, (40, D)) / 2 - bins / 2).astype(np.float16)
        x[1, 30:40] = np.float16(0.37)
        x[1, 50:60] = 0
        x[2, 70:90] = (x[2, 70:90].astype(np.float32) * 1e-6).astype(np.float16)
        x[2, 100:120] = np.where(r.random((20, D)) < 0.5, np.float16(65504), np.float16(-65504))
        x[3, n - 20:] *= np.float16(300)
    if odd:
        k[0, 33, 7], k[3, n - 1, D - 1], k[1, 3, 64] = np.inf, np.nan, -np.inf
        v[0, 35, 9], v[2, n - 2, 0], v[1, 0, 1] = np.nan, -np.inf, np.inf
    one, many = (qw_amd.KVCache(mode, H, D, capacity=n + 64) for _ in range(2))
    for c in (one, many):
        c.update(_gpu(k[:, :5]), _gpu(v[:, :5]))
    one.update(_gpu(k[:, 5:]), _gpu(v[:, 5:]))
    for at in range(5, n, 200):
        many.update(_gpu(k[:, at:at + 200]), _gpu(v[:, at:at + 200]))
    a, b = one.snapshot_tensors(), many.snapshot_tensors()
    assert a.keys() == b.keys()
    for name in a:
        x, y = (np.asarray(t.cpu() if hasattr(t, "cpu") else t) for t in (a[name], b[name]))
        np.testing.assert_array_equal(x.view(np.uint8), y.view(np.uint8), err_msg=name)
