"""GPU parity of the row kernel behind qw_sdpa (attend_rows.hip: many query rows over fp16 K/V
views, laid out once as tile images) against oracle.sdpa_general, at the sizes where it can go
wrong: key counts around a tile (64 / 128 / 256 keys at D 256 / 128 / 64), rows around a wave and
a workgroup, split and unsplit plans, every mask type at odd strides, windows below a tile.

Bar: the attention tolerance (2e-3 max-abs, 1e-3 relative L2); the masks' rows that see nothing
are exact zeros."""
import numpy as np
import pytest

import oracle
from conftest import rng
from test_gpu_kv import _gpu, _np, assert_close

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _views(r, hkv, T, D, pad):
    """fp16 K, V [hkv, T, D] and the same rows as views of a larger allocation whose other rows
    are NaN (nothing past the view may be read into a result)."""
    k = r.standard_normal((hkv, T, D)).astype(np.float16)
    v = r.standard_normal((hkv, T, D)).astype(np.float16)
    kb = torch.full((hkv, T + pad, D + 8), float("nan"), dtype=torch.float16, device="cuda:0")
    vb = torch.full_like(kb, float("nan"))
    kb[:, :T, :D] = _gpu(k)
    vb[:, :T, :D] = _gpu(v)
    return k, v, kb[:, :T, :D], vb[:, :T, :D]


def takes_rows(hq, hkv, D, L, T, causal=True, window=0, softcap=0.0, mask=-1):
    """Whether the call runs the row kernel (mask: its ABI dtype)."""
    import qw_amd

    return bool(qw_amd.lib().qw_sdpa_takes_rows(hq, L, hkv, T, D, int(causal), window, softcap, mask))


CASES = [
    # hq, hkv, D, L, T, causal, window, softcap
    (24, 4, 256, 129, 2048, True, 0, 0.0),     # whole tiles; 774 rows a head, a ragged last tile
    (24, 4, 256, 257, 1985, True, 0, 0.0),     # one key into the last tile
    (24, 4, 256, 257, 1983, True, 0, 0.0),     # one key short of it
    (8, 8, 128, 700, 2305, True, 0, 0.0),      # G = 1
    (32, 8, 128, 200, 2047, True, 300, 0.0),   # a window of a few tiles
    (8, 8, 128, 151, 2047, True, 130, 0.0),    # and about one
    (24, 4, 256, 90, 1000, True, 64, 0.0),
    (16, 2, 64, 300, 1281, True, 0, 0.0),      # 256-key tiles in two halves
    (16, 2, 64, 300, 2500, True, 900, 20.0),   # capped, in a window
    (24, 4, 256, 130, 1400, True, 100, 30.0),
    (24, 4, 128, 220, 1400, False, 0, 30.0),   # capped, not causal
    (24, 4, 128, 220, 1400, True, 0, 128.0),   # caps far above the scores
    (24, 4, 128, 220, 1400, True, 0, 300.0),
    (12, 1, 256, 300, 1000, True, 0, 0.0),     # one KV head, G = 12
    (24, 4, 256, 1100, 1100, True, 0, 0.0),    # prefill into nothing: rows from one key on
]
# shapes that the generic kernel serves faster (it must agree there too)
GENERIC = [
    (32, 8, 128, 200, 2047, True, 130, 0.0),
    (16, 2, 64, 256, 1281, True, 0, 0.0),
    (16, 2, 64, 300, 1500, True, 33, 20.0),
    (12, 1, 256, 190, 1000, True, 0, 0.0),
]


@pytest.mark.parametrize("hq,hkv,D,L,T,causal,window,softcap", CASES + GENERIC)
def test_rows_match_oracle(hq, hkv, D, L, T, causal, window, softcap):
    import qw_amd

    print(f"case hq={hq} hkv={hkv} D={D} L={L} T={T} causal={causal} w={window} sc={softcap}",
          flush=True)
    shape = (hq, hkv, D, L, T, causal, window, softcap)
    assert takes_rows(*shape) == (shape in CASES), "the kernel of the call"
    r = rng(hq + D + L + T)
    q = r.standard_normal((hq, L, D)).astype(np.float16)
    k, v, kv, vv = _views(r, hkv, T, D, 9)
    out = _np(qw_amd.attention(_gpu(q), kv, vv, D ** -0.5, None, softcap, window, causal))[0]
    assert np.isfinite(out).all()
    assert_close(out, oracle.sdpa_general(q, k, v, D ** -0.5, causal, window, softcap),
                 f"rows D={D} L={L} T={T}")


@pytest.mark.parametrize("kind", ["bool", "f16", "bf16", "f32"])
@pytest.mark.parametrize("hq,hkv,D,L,T,causal,per_head", [
    (24, 4, 256, 13, 6500, False, False),
    (24, 4, 128, 60, 2051, True, True),
    (16, 2, 64, 100, 3333, False, True),
    (24, 4, 128, 41, 2051, True, True),       # (a bool mask alone; the others in the generic kernel)
    (16, 2, 64, 20, 3333, False, True),       # (the generic kernel)
])
def test_rows_masks_match_oracle(kind, hq, hkv, D, L, T, causal, per_head):
    import qw_amd

    print(f"case {kind} hq={hq} D={D} L={L} T={T} causal={causal}", flush=True)
    code = {"bool": 3, "f16": 0, "bf16": 1, "f32": 2}[kind]
    assert takes_rows(hq, hkv, D, L, T, causal, 0, 0.0, code) == \
        (L in (13, 60, 100) or (L == 41 and kind == "bool")), "the kernel of the call"
    r = rng(hq + D + L + T + len(kind))
    q = r.standard_normal((hq, L, D)).astype(np.float16)
    k, v, kv, vv = _views(r, hkv, T, D, 3)
    H = hq if per_head else 1
    hidden = r.random((H, L, T)) < 0.3
    hidden[:, 0, :] = True                       # a row that sees nothing
    hidden[:, 1:, 0] = False
    if kind == "bool":
        m = ~hidden
        full = torch.zeros((H, L, T + 5), dtype=torch.bool, device="cuda:0")
    else:
        m = (2 * r.standard_normal((H, L, T))).astype(np.float32)
        m[hidden] = -np.inf
        dt = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[kind]
        full = torch.zeros((H, L, T + 5), dtype=dt, device="cuda:0")
    view = full[:, :, 1:T + 1]                   # odd row stride, off any vector alignment
    view.copy_(torch.from_numpy(m))
    m = view.cpu().numpy() if kind == "bool" else view.float().cpu().numpy()
    sc = 0.0 if kind == "bool" else 25.0
    for cap in {0.0, sc}:
        out = _np(qw_amd.attention(_gpu(q), kv, vv, D ** -0.5, view, cap, 0, causal))[0]
        assert np.isfinite(out).all() and np.all(out[:, 0] == 0)
        ref = oracle.sdpa_general(q, k, v, D ** -0.5, causal, 0, cap, m)
        assert_close(out[:, 1:], ref[:, 1:], f"rows {kind} cap={cap}")


def test_rows_route_agrees_with_the_general_kernel():
    """The same rows in one call (row kernel) and in calls of few rows (the general kernel)."""
    import qw_amd

    r = rng(5)
    hq, hkv, D, L, T = 24, 4, 256, 160, 1700
    assert takes_rows(hq, hkv, D, L, T) and not takes_rows(hq, hkv, D, 16, T)
    q = _gpu(r.standard_normal((hq, L, D)).astype(np.float16))
    _, _, kv, vv = _views(r, hkv, T, D, 0)
    whole = _np(qw_amd.causal_attention(q, kv, vv, 1 / 16))[0]
    step = 16
    parts = [_np(qw_amd.causal_attention(q[:, i:i + step].contiguous(), kv[:, :T - L + i + step],
                                         vv[:, :T - L + i + step], 1 / 16))[0]
             for i in range(0, L, step)]
    assert_close(whole, np.concatenate(parts, axis=1), "one call vs pieces")


@pytest.mark.parametrize("hkv,D", [(4, 256), (4, 128), (2, 64)])
def test_rows_largest_weight_is_not_rounded(hkv, D):
    """One key outweighs an earlier one by a score of 1 to 5, V is 1: P is taken against the running
    maximum, so that key's weight is exactly 1 in fp16. What is left is the other key's rounding
    (below e^-1 2^-12) and fp32 sums: the result is within 2^-12 of 1, which rounds to 1."""
    import qw_amd

    G, L, T = 6, 400, 1300
    s = np.linspace(1, 5.4, L).astype(np.float16)
    q = np.zeros((G * hkv, L, D), np.float16)
    q[:, :, 0] = s * np.float16(16)
    k = np.zeros((hkv, T, D), np.float16)
    k[:, :, 0] = -60
    k[:, 3, 0] = 0
    k[:, 66 if D == 256 else 130, 0] = 1  # the next 64- or 128-key step of the same key split
    assert takes_rows(G * hkv, hkv, D, L, T, False), "a shape of the row kernel"
    out = _np(qw_amd.attention(_gpu(q), _gpu(k), _gpu(np.ones_like(k)), 1 / 16))[0]
    assert np.all(out == 1), np.unique(out)


@pytest.mark.parametrize("hq,hkv,D,L,T,window,softcap,masked", [
    (24, 4, 256, 230, 1400, 0, 0.0, False),
    (24, 4, 256, 130, 1400, 100, 30.0, False),
    (8, 8, 128, 700, 2305, 0, 0.0, False),
    (8, 8, 128, 701, 2305, 300, 0.0, False),
    (8, 8, 128, 151, 2047, 130, 0.0, False),
    (24, 4, 256, 90, 1000, 64, 0.0, False),
    (16, 2, 64, 300, 1281, 0, 0.0, False),
    (16, 2, 64, 301, 2500, 900, 25.0, False),
    (24, 4, 256, 100, 1290, 0, 0.0, True),
])
def test_rows_keep_keys_outside_their_limits_out(hq, hkv, D, L, T, window, softcap, masked):
    """Infinite and NaN keys that none of a wave's 16 rows sees (later than the last one's position,
    earlier than the first one's window) change none of its outputs."""
    import qw_amd

    G = hq // hkv
    assert takes_rows(hq, hkv, D, L, T, True, window, softcap, 3 if masked else -1), "a shape of the row kernel"
    r = rng(hq + D + L + window)
    q = _gpu(r.standard_normal((hq, L, D)).astype(np.float16))
    k, v, kv, vv = _views(r, hkv, T, D, 0)
    mask = torch.ones((1, 1, L, T), dtype=torch.bool, device="cuda:0") if masked else None
    call = lambda: _np(qw_amd.attention(q, kv, vv, D ** -0.5, mask, softcap, window, True))[0]  # noqa: E731
    clean = call()
    ref = oracle.sdpa_general(_np(q), k, v, D ** -0.5, True, window, softcap)
    assert_close(clean, ref, f"D={D} L={L} T={T} w={window}")
    wave = (np.arange(G * L) // 16).reshape(L, G).T                     # of (head in group, row)
    first, last = T - L + wave * 16 // G, T - L + np.minimum(wave * 16 + 15, G * L - 1) // G
    for t in (T - L + 20, T - L // 2, T - L // 2 + 5, T - 7):
        keep = kv[:, t].clone(), vv[:, t].clone()
        kv[:, t], vv[:, t] = float("nan"), float("inf")
        blind = (t > last) | ((t < first - window + 1) if window else False)
        out, blind = call(), np.tile(blind, (hkv, 1))
        assert blind.any() and np.isfinite(out[blind]).all(), f"key {t}"
        np.testing.assert_array_equal(out[blind], clean[blind], f"key {t}")
        kv[:, t], vv[:, t] = keep
