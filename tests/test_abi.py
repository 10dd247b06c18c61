"""The C ABI library loads and exports every entry point include/qwattn.h
declares; argument checks that run before any device call return the
documented status codes. CPU only: nothing here launches a kernel."""
import ctypes
import os
import re

import pytest

from conftest import ROOT

HEADER = os.path.join(ROOT, "include", "qwattn.h")


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(qw_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def qwlib():
    import qw_amd

    if not os.path.exists(qw_amd.LIB_PATH):
        from qw_amd import build

        build.build()
    return qw_amd.lib()


def test_header_declares_the_path():
    names = _declared()
    for n in ("qw_kv_create", "qw_kv_update", "qw_kv_update_and_attention", "qw_kv_trim",
              "qw_kv_export", "qw_kv_import", "qw_dlsa_sparse_attention"):
        assert n in names


def test_every_declared_symbol_is_exported(qwlib):
    missing = [n for n in _declared() if not hasattr(qwlib, n)]
    assert not missing, missing


def test_abi_version_matches_header(qwlib):
    m = re.search(r"#define QWATTN_ABI_VERSION (\d+)", open(HEADER).read())
    assert qwlib.qw_abi_version() == int(m.group(1))


def test_invalid_arguments_fail_before_device_work(qwlib):
    h = ctypes.c_void_p()
    assert qwlib.qw_kv_create(7, 64, 4, 256, 1024, 0, ctypes.byref(h)) == 1
    assert b"mode" in qwlib.qw_last_error()
    assert qwlib.qw_kv_create(2, 32, 4, 256, 1024, 0, ctypes.byref(h)) == 2  # group != 64
    assert qwlib.qw_kv_create(2, 64, 4, 96, 1024, 0, ctypes.byref(h)) == 2   # head_dim
    assert qwlib.qw_kv_create(2, 64, 0, 256, 1024, 0, ctypes.byref(h)) == 1
    assert qwlib.qw_kv_create(2, 64, 4, 256, 1024, 0, None) == 1
    assert not h.value
    # null handle
    off = ctypes.c_int()
    assert qwlib.qw_kv_offset(None, ctypes.byref(off)) == 1
    assert qwlib.qw_kv_trim(None, 1, None) == 1
    assert qwlib.qw_kv_destroy(None) == 0
    # D-LSA geometry checks
    f = qwlib.qw_dlsa_sparse_attention
    assert f(None, None, None, 0, 0, 0, 0, None, None, 1, 1, 24, 4, 256, 10, 0.1, None, None) == 1
    one = ctypes.c_void_p(16)
    args = [one, one, one, 0, 256, 0, 256, one, one, 1, 8, 24, 4, 256, 10, 0.1, one, None]
    args_bad_dim = list(args)
    args_bad_dim[13] = 96
    assert f(*args_bad_dim) == 1
    args_bad_g = list(args)
    args_bad_g[11], args_bad_g[12] = 68, 4  # 17 heads per KV head
    assert f(*args_bad_g) == 1
    args_bad_w = list(args)
    args_bad_w[10] = 0
    assert f(*args_bad_w) == 1


def test_fused_rope_contract_fails_before_device_work(qwlib):
    """fused_rope_append.cpp:394-418: the argument contract, checked before
    any launch (status 1, QW_ERR_INVALID_ARGUMENT)."""
    f = qwlib.qw_fused_rope_qk_append
    one = ctypes.c_void_p(16)

    def call(**kw):
        a = dict(batch=1, seq=4, hq=8, hkv=2, D=128, R=64, base=10000.0, scale=1.0, trad=0,
                 pos=0, layout=0)
        a.update(kw)
        return f(one, a["batch"], a["seq"], a["hq"], a["hkv"], a["D"], a["R"], a["base"],
                 a["scale"], a["trad"], a["pos"], a["layout"], one, one, one, None)

    assert call(R=0) == 1
    assert b"rope_dims" in qwlib.qw_last_error()
    assert call(R=63) == 1
    assert call(R=130) == 1
    assert call(D=127, R=64) == 1
    assert b"head_dim must be even" in qwlib.qw_last_error()
    assert call(hq=0) == 1
    assert call(hkv=-1) == 1
    assert call(layout=2) == 1
    assert b"dest_layout" in qwlib.qw_last_error()
    assert call(seq=-1) == 1
    assert call(seq=0) == 0  # nothing to do: no launch
    assert f(None, 1, 4, 8, 2, 128, 64, 10000.0, 1.0, 0, 0, 0, None, None, None, None) == 1
    assert qwlib.qw_kv_rope_update(None, one, 8, 4, 64, 0, 10000.0, 1.0, 0, one, None) == 1


def test_general_attention_contract_fails_before_device_work(qwlib):
    """qw_sdpa's argument contract (mask, softcap and window as the reference's
    layers::attention / causal_attention take them), checked before any HIP
    call."""
    f = qwlib.qw_sdpa
    one = ctypes.c_void_p(16)

    def call(**kw):
        a = dict(hq=8, L=4, hkv=2, T=100, D=128, causal=1, window=0, softcap=0.0, mask=None,
                 md=0, mhs=0, mrs=100)
        a.update(kw)
        return f(one, a["hq"], a["L"], one, one, a["hkv"], a["T"], a["D"], a["T"] * a["D"],
                 a["D"], a["T"] * a["D"], a["D"], 0.1, a["causal"], a["window"], a["softcap"],
                 a["mask"], a["md"], a["mhs"], a["mrs"], one, None)

    assert call(D=96) == 1
    assert call(hq=9) == 1                     # not a multiple of the KV heads
    assert call(T=3) == 1                      # causal with fewer keys than rows
    assert call(causal=0, window=8) == 1       # a window is the windowed causal mask
    assert b"window" in qwlib.qw_last_error()
    assert call(softcap=-1.0) == 1
    assert call(mask=one, md=7) == 1           # unknown mask dtype
    assert call(mask=one, md=3, softcap=5.0) == 2  # bool mask with softcap
    assert b"bool mask" in qwlib.qw_last_error()
    assert call(mask=one, md=0, mrs=-1) == 1
    assert f(None, 8, 4, one, one, 2, 100, 128, 0, 128, 0, 128, 0.1, 1, 0, 0.0, None, 0, 0, 0,
             one, None) == 1


@pytest.mark.parametrize("hq,hkv,D,L,T,kind,generic_us,rows_us", [
    # calls that both kernels were timed on, near the line
    (24, 4, 256, 85, 4000, "causal", 51, 37),
    (24, 4, 256, 42, 4000, "causal", 33, 37),
    (24, 4, 256, 42, 16000, "causal", 85, 64),
    (24, 4, 256, 256, 300, "causal", 28, 32),
    (8, 8, 128, 384, 4000, "causal", 46, 33),
    (8, 8, 128, 192, 1000, "causal", 16, 21),
    (32, 8, 128, 64, 16000, "causal", 102, 58),
    (16, 1, 64, 96, 4000, "causal", 24, 21),
    (16, 1, 64, 96, 1000, "causal", 12, 20),
    (16, 2, 64, 24, 16000, "causal", 23, 25),
    (16, 1, 128, 12, 4000, "causal", 16, 20),
    (24, 4, 256, 42, 4000, "bool", 43, 36),
    (16, 2, 64, 32, 1000, "bool", 15, 25),
    (8, 8, 128, 192, 4000, "bool", 47, 29),
    (8, 8, 64, 96, 4000, "f16", 28, 34),
    (8, 8, 64, 425, 4000, "window 64", 11, 23),
    (24, 4, 256, 170, 16000, "softcap", 350, 147),
    (8, 8, 64, 96, 4000, "softcap", 20, 27),
])
def test_sdpa_row_kernel_line(qwlib, hq, hkv, D, L, T, kind, generic_us, rows_us):
    """The kernel of a qw_sdpa call: the one that measured faster."""
    window = 64 if kind == "window 64" else 0
    mask = {"bool": 3, "f16": 0}.get(kind, -1)
    takes = qwlib.qw_sdpa_takes_rows(hq, L, hkv, T, D, int(mask < 0), window,
                                     30.0 if kind == "softcap" else 0.0, mask)
    assert takes == (rows_us < generic_us)


def test_sdpa_row_kernel_line_limits(qwlib):
    f = qwlib.qw_sdpa_takes_rows
    assert f(24, 3072, 4, 524288, 256, 1, 0, 0.0, -1) == 1
    assert f(24, 3072, 4, 2097153, 256, 1, 0, 0.0, -1) == 0  # images past 4 GiB
    assert f(16, 1, 1, 1 << 20, 256, 1, 0, 0.0, 3) == 0      # 16 rows a KV head
    assert f(24, 1536, 4, 9728, 256, 1, (1 << 31) - 1, 0.0, -1) == 1  # a window past any position
    assert f(24, 4, 5, 100, 256, 1, 0, 0.0, -1) == 0 and f(24, 0, 4, 100, 256, 1, 0, 0.0, -1) == 0
    assert f(24, 1 << 20, 4, 1 << 20, 256, 1, 0, 0.0, -1) == 1  # (no overflow on the way)


@pytest.mark.parametrize("dt,hq,hkv,D,L,T,W,kind,rows_us,here_us", [
    # calls timed row by row and by the unions of neighbouring rows, near the line
    ("f16", 24, 4, 256, 1536, 33280, 4612, "sliding", 1312, 345),
    ("f16", 16, 2, 64, 1100, 4000, 1024, "single draws", 72, 110),
    ("f16", 32, 8, 128, 97, 8000, 1100, "shared", 39, 44),
    ("f16", 16, 2, 64, 194, 8000, 2200, "shared", 39, 42),
    ("bf16", 24, 4, 256, 512, 16000, 4612, "sliding", 7572, 175),
    ("bf16", 24, 4, 256, 48, 1000, 128, "sliding", 79, 38),
    ("bf16", 8, 8, 128, 96, 1000, 64, "shared", 16, 24),
    ("f32", 8, 8, 128, 96, 1000, 64, "single draws", 21, 47),
    ("f32", 4, 2, 256, 192, 1000, 64, "shared", 22, 36),
    ("f32", 24, 4, 256, 512, 16000, 4612, "sliding", 7530, 744),
])
def test_dlsa_union_line(qwlib, dt, hq, hkv, D, L, T, W, kind, rows_us, here_us):
    """Whether a sparse read's rows share their gathers: where that measured faster."""
    c = {"f16": 0, "bf16": 1, "f32": 2}[dt]
    n = qwlib.qw_dlsa_union_keys(c, c, L, W, hq, hkv, D, T)
    assert (n > 0) == (here_us < rows_us) and n <= T


def test_dlsa_union_line_limits(qwlib):
    f = qwlib.qw_dlsa_union_keys
    assert f(1, 1, 47, 4612, 24, 4, 256, 100000) == 0                 # split lists
    assert 0 < f(1, 1, 1 << 20, 1 << 16, 24, 4, 256, 1 << 30) < 1 << 30  # (no overflow on the way)
    assert f(0, 0, 1 << 20, 1 << 20, 16, 1, 64, (1 << 31) - 1) >= 0
    assert f(0, 0, 0, 64, 16, 1, 64, 100) == 0 and f(0, 0, 9999, 64, 17, 1, 64, 100) == 0
