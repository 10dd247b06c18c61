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
