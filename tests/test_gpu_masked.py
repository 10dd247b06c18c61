"""GPU parity of masked attention over a cache (the block kernel on the codes, qw_kv_attention_general)
against oracle.sdpa_general on the cache's own dequantized rows (Turbo4: on the oracle's rotated
expansion of its snapshot): every mode and mask type, rows below and above one 16-row tile, one
query tile and several, key counts around a 64 / 128-key tile, split and unsplit, causal or not,
masks with odd strides, rows that see nothing.

Bar: the attention tolerance (2e-3 max-abs, 1e-3 relative L2); rows that see nothing are zeros."""
import numpy as np
import pytest

import oracle
from conftest import rng
from test_gpu_kv import _gpu, _np, assert_close

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _mask(r, kind, H, L, T):
    """(what the oracle takes, a device view off any vector alignment), row 1 sees nothing."""
    hidden = r.random((H, L, T)) < 0.3
    hidden[:, :, 0] = False
    hidden[:, 1] = True
    if kind == "bool":
        view = torch.zeros((H, L, T + 3), dtype=torch.bool, device="cuda:0")[:, :, 1:T + 1]
        view.copy_(torch.from_numpy(~hidden))
        return ~hidden, view
    m = (2 * r.standard_normal((H, L, T))).astype(np.float32)
    m[hidden] = -np.inf
    view = torch.zeros((H, L, T + 3), dtype=DT[kind], device="cuda:0")[:, :, 1:T + 1]
    view.copy_(torch.from_numpy(m))
    return view.float().cpu().numpy(), view


def _reference(cache, mode, q, D, scale, causal, m):
    if mode != "turbo4":
        kd, vd = (_np(x)[0] for x in cache.dequantize())
        return oracle.sdpa_general(q, kd, vd, scale, causal, mask=m)
    snap = {n: _np(x) for n, x in cache.snapshot_tensors().items()}
    tab = oracle.turbo4_tables(D)
    q_rot = oracle.turbo4_rotate(q.astype(np.float64), tab["k_s1"], tab["k_s2"]).astype(np.float16)
    k_rot = oracle.turbo4_expand_rotated(snap["k_packed"], snap["k_rescale"][..., 0], tab)
    v_rot = oracle.turbo4_expand_rotated(snap["v_packed"], snap["v_rescale"][..., 0], tab)
    o = oracle.sdpa_general(q_rot, k_rot, v_rot, scale, causal, mask=m)
    return oracle.turbo4_rotate(o.astype(np.float64), tab["v_s2"], tab["v_s1"]).astype(np.float16)


CASES = [
    # hq, hkv, D, L, T, causal, kind, a mask for each head
    (24, 4, 256, 2, 63, False, "bool", False),      # 12 rows a head, under one tile of keys
    (24, 4, 256, 3, 65, True, "f16", False),        # 18 rows, one key into the second tile
    (24, 4, 256, 13, 1500, False, "bool", False),   # five 16-row tiles, key split
    (24, 4, 256, 23, 640, True, "f32", True),       # 138 rows: two query tiles
    (16, 2, 128, 40, 385, False, "bf16", False),    # 320 rows, one key into a tile
    (32, 8, 128, 2, 3000, True, "f32", False),
]


@pytest.mark.parametrize("mode", ["affine4", "affine8", "int8", "turbo4", "fp16"])
@pytest.mark.parametrize("hq,hkv,D,L,T,causal,kind,per_head", CASES)
def test_masked_cache_matches_oracle(mode, hq, hkv, D, L, T, causal, kind, per_head):
    import qw_amd

    print(f"case {mode} hq={hq} hkv={hkv} D={D} L={L} T={T} causal={causal} {kind}", flush=True)
    r = rng(hq + D + L + T)
    k, v = (r.standard_normal((hkv, T, D)).astype(np.float16) for _ in range(2))
    q = r.standard_normal((hq, L, D)).astype(np.float16)
    m, view = _mask(r, kind, hq if per_head else 1, L, T)
    cache = qw_amd.KVCache(mode, hkv, D)
    cache.update(_gpu(k[:, :T - L]), _gpu(v[:, :T - L])) if T > L else None
    if causal:
        cache.update(_gpu(k[:, T - L:]), _gpu(v[:, T - L:]))
        out = _np(cache.attention_general(_gpu(q), D ** -0.5, causal=True, mask=view))[0]
    else:
        out = _np(cache.update_and_attention(_gpu(q), _gpu(k[:, T - L:]), _gpu(v[:, T - L:]),
                                             D ** -0.5, mask=view))[0]
    assert cache.offset == T and np.isfinite(out).all() and np.all(out[:, 1] == 0)
    ref = _reference(cache, mode, q, D, D ** -0.5, causal, m)
    keep = [i for i in range(L) if i != 1]
    assert_close(out[:, keep], ref[:, keep], f"{mode} {kind} L={L} T={T}")


@pytest.mark.parametrize("mode", ["affine4", "affine8"])
def test_masked_cache_with_extreme_scales(mode):
    """A scale outside the exact two-step dequant's range: the separately rounded pass."""
    import qw_amd

    r = rng(17)
    hq, hkv, D, L, T = 12, 2, 256, 5, 300
    k, v = (r.standard_normal((hkv, T, D)).astype(np.float16) for _ in range(2))
    k[:, 7, :64] *= np.float16(1e-4)
    v[:, 9, 64:128] *= np.float16(1e-4)
    v[:, 11, :64] *= np.float16(2000)
    q = r.standard_normal((hq, L, D)).astype(np.float16)
    m, view = _mask(r, "bool", 1, L, T)
    m[..., 11] = False
    view[..., 11] = False
    cache = qw_amd.KVCache(mode, hkv, D)
    cache.update(_gpu(k), _gpu(v))
    out = _np(cache.attention_general(_gpu(q), 1 / 16, mask=view))[0]
    ref = _reference(cache, mode, q, D, 1 / 16, False, m)
    keep = [0, 2, 3, 4]
    assert_close(out[:, keep], ref[:, keep], f"{mode} extreme scales")


@pytest.mark.parametrize("D,L", [(256, 13), (128, 40)])
def test_masked_largest_weight_is_not_rounded(D, L):
    """As test_gpu_rows.py's: a key that outweighs an earlier one has a weight of exactly 1 in fp16,
    and rows of ones come back as ones."""
    import qw_amd

    hq, hkv, T = 24, 4, 1500
    s = np.linspace(1, 5.4, L).astype(np.float16)
    q = np.zeros((hq, L, D), np.float16)
    q[:, :, 0] = s * np.float16(16)
    k = np.zeros((hkv, T, D), np.float16)
    k[:, :, 0] = -60
    k[:, 1, 0] = 0                      # in one 64 / 128-key tile's first half, the winner in
    k[:, 200, 0] = 1                    # a later tile of the same split
    mask = torch.ones((1, 1, L, T), dtype=torch.bool, device="cuda:0")
    cache = qw_amd.KVCache("fp16", hkv, D)
    cache.update(_gpu(k), _gpu(np.ones_like(k)))
    out = _np(cache.attention_general(_gpu(q), 1 / 16, mask=mask))[0]
    assert np.all(out == 1), np.unique(out)


@pytest.mark.parametrize("mode", ["affine4", "affine8", "int8", "turbo4", "fp16"])
@pytest.mark.parametrize("D,L,causal", [(256, 13, False), (128, 40, False), (256, 3, True)])
def test_masked_cache_after_a_trim(mode, D, L, causal):
    """Rows that a trim left behind the offset take no part, whatever they hold: the call returns
    what a cache that never held them does, bit for bit."""
    import qw_amd

    r = rng(D + L)
    hq, hkv, T = 24, 4, 700
    k, v = (r.standard_normal((hkv, T, D)).astype(np.float16) for _ in range(2))
    q = r.standard_normal((hq, L, D)).astype(np.float16)
    bad = np.zeros((hkv, L + 50, D), np.float16)
    bad[:, ::2] = np.inf
    bad[:, 1::2] = np.nan
    _, view = _mask(r, "bool", 1, L, T)
    outs = []
    for poisoned in (False, True):
        cache = qw_amd.KVCache(mode, hkv, D, capacity=1024)
        cache.update(_gpu(k[:, :T - L]), _gpu(v[:, :T - L]))
        if poisoned:
            cache.update(_gpu(bad), _gpu(bad))
            cache.trim(L + 50)
        cache.update(_gpu(k[:, T - L:]), _gpu(v[:, T - L:]))
        outs.append(_np(cache.attention_general(_gpu(q), D ** -0.5, causal=causal, mask=view))[0])
    assert np.isfinite(outs[1]).all()
    # (an affine cache that ever held a scale outside the two-step dequant's exact range rounds in
    # two steps from then on; both are the same values)
    np.testing.assert_array_equal(outs[0], outs[1])


@pytest.mark.parametrize("mode", ["affine4", "affine8", "int8", "turbo4", "fp16"])
@pytest.mark.parametrize("hq,hkv,D,L,T", [
    (32, 8, 128, 1020, 1155),   # 4080 rows a head: whole rounds of unsplit query tiles
    (32, 16, 128, 1050, 1155),  # 2100: a round of them and a split tail in one launch
    (24, 12, 256, 1500, 1601),  # 3000, a head count that does not divide the CUs
    (32, 8, 128, 1030, 1155),   # 4120: dequantized once, the row kernel
])
def test_masked_cache_of_many_rows(mode, hq, hkv, D, L, T):
    """Both sides of the line at 4096 rows a KV head, and the plans below it: every 97th row and the
    last against the oracle, the causal cut put into its mask."""
    import qw_amd

    print(f"case {mode} hq={hq} hkv={hkv} D={D} L={L} T={T}", flush=True)
    r = rng(hkv + D + L)
    k, v = (r.standard_normal((hkv, T, D)).astype(np.float16) for _ in range(2))
    q = r.standard_normal((hq, L, D)).astype(np.float16)
    m, view = _mask(r, "bool", 1, L, T)
    cache = qw_amd.KVCache(mode, hkv, D)
    cache.update(_gpu(k), _gpu(v))
    out = _np(cache.attention_general(_gpu(q), D ** -0.5, causal=True, mask=view))[0]
    assert np.isfinite(out).all() and np.all(out[:, 1] == 0)
    rows = np.unique(np.append(np.arange(0, L, 97), L - 1))
    seen = m[:, rows] & (np.arange(T) <= (T - L + rows)[:, None])
    ref = _reference(cache, mode, q[:, rows], D, D ** -0.5, False, seen)
    assert_close(out[:, rows], ref, f"{mode} L={L} T={T}")
