"""GPU parity of the D-LSA read for prefill row counts (dlsa_rows.hip: groups of neighbouring rows
read the union of their keys once) against the float64 restatement, where it can go wrong: lists
that share all, some or none of their keys, entries that are -1 or out of range, a key listed
twice, ragged and zero lengths, a last group that is not full, unions around a tile, keys past one
bitmap pass, infinite values that only some rows list.

fp16: the attention tolerance (2e-3 max-abs, 1e-3 relative L2). bf16: the output's rounding, half
a unit of 2^-8 relative to each value, plus 1e-5 of the row for the 32-bit sums."""
import numpy as np
import pytest

import oracle
from conftest import rng
from test_gpu_kv import _gpu, _np, assert_close

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _lists(r, kind, L, W, T):
    if kind == "shared":     # one set for all rows, each row in its own order
        base = r.choice(T, W, replace=False)
        return np.stack([r.permutation(base) for _ in range(L)]).astype(np.int32)
    if kind == "sliding":    # a shared half and a window that moves by one
        base = np.sort(r.choice(T - W - L, W - W // 2, replace=False))
        return np.stack([np.concatenate([base, T - L - W // 2 + i + np.arange(W // 2)])
                         for i in range(L)]).astype(np.int32)
    if kind == "own":        # nothing in common but chance
        return np.stack([r.choice(T, W, replace=False) for _ in range(L)]).astype(np.int32)
    if kind == "mixed":      # the groups of the first half share, the others do not
        a = _lists(r, "sliding", L // 2, W, T)
        return np.concatenate([a, _lists(r, "own", L - L // 2, W, T)])
    raise ValueError(kind)


def _check(out, q, k, v, lists, lengths, scale, bf16, what):
    ref = oracle.dlsa_attention_f64(q, k, v, lists, lengths, scale)
    assert np.isfinite(out).all(), what
    if not bf16:
        assert_close(out, ref.astype(np.float32), what)
        return
    bound = np.abs(ref) * 2.0 ** -8 + 1e-5 * np.linalg.norm(ref, axis=-1, keepdims=True)
    assert np.all(np.abs(out.astype(np.float64) - ref) <= bound), what


def _run(q, k, v, lists, lengths, scale, bf16):
    import qw_amd

    if not bf16:
        return _np(qw_amd.sparse_attention(_gpu(q), _gpu(k), _gpu(v), _gpu(lists), _gpu(lengths),
                                           scale))[0]
    t = [_gpu(x).to(torch.bfloat16) for x in (q, k, v)]
    return qw_amd.sparse_attention_typed(*t, _gpu(lists), _gpu(lengths), scale)[0].float().cpu().numpy()


TYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
# half a unit in the last place of the output's type, relative to the value
ROUND = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8, "f32": 0.0}


def _takes_it(hq, hkv, D, L, T, W, dt="f16"):
    """Whether the call's rows share their keys' gathers."""
    import qw_amd

    c = {"f16": 0, "bf16": 1, "f32": 2}[dt]
    return qw_amd.lib().qw_dlsa_union_keys(c, c, L, W, hq, hkv, D, T) > 0


CASES = [
    # hq, hkv, D, L, T, W, kind, whether an fp16 call takes the kernel too
    (24, 4, 256, 101, 8000, 2200, "sliding", True),   # the last group one row
    (24, 4, 256, 700, 2000, 320, "shared", False),    # the union exactly five tiles
    (24, 4, 256, 700, 2000, 321, "shared", False),    # one key past them
    (24, 4, 256, 112, 40000, 2000, "own", False),
    (24, 4, 256, 160, 40000, 1400, "mixed", False),
    (8, 8, 128, 130, 4000, 900, "sliding", True),     # G = 1: 32 rows a group
    (24, 3, 128, 96, 6000, 3000, "sliding", True),    # KV heads that do not divide 256
    (16, 2, 64, 300, 9000, 1500, "sliding", False),   # 256-key tiles in two halves
    (16, 1, 128, 600, 4000, 1500, "shared", False),   # G = 16: 8 rows a group
    (24, 4, 256, 96, 90000, 2300, "sliding", False),  # three bitmap passes
    (24, 4, 256, 1300, 2600, 400, "sliding", False),  # whole rounds and a split rest
    (24, 4, 256, 440, 2000, 512, "shared", False),    # the union exactly eight tiles
    (24, 4, 256, 440, 2000, 513, "shared", False),
    (16, 2, 64, 300, 6000, 1500, "sliding", False),
    (16, 1, 128, 600, 2500, 1500, "shared", False),
    (24, 4, 256, 700, 700, 321, "shared", True),      # (fp16's of the kinds above)
    (24, 4, 256, 900, 2000, 512, "shared", True),
    (24, 4, 256, 900, 2000, 513, "shared", True),
    (16, 2, 64, 300, 6000, 3000, "sliding", True),
    (16, 1, 128, 600, 3000, 2500, "shared", True),
    (24, 4, 256, 1300, 2600, 800, "sliding", True),
]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("hq,hkv,D,L,T,W,kind,fp16", CASES)
def test_rows_match_oracle(hq, hkv, D, L, T, W, kind, fp16, bf16):
    print(f"case hq={hq} hkv={hkv} D={D} L={L} T={T} W={W} {kind} bf16={bf16}", flush=True)
    assert fp16 == _takes_it(hq, hkv, D, L, T, W), "the route of the fp16 call"
    assert _takes_it(hq, hkv, D, L, T, W, "bf16"), "a shape of the bf16 call's kernel"
    if bf16 and hq // hkv > 8:
        pytest.skip("the typed read takes at most 8 heads a KV head")
    r = rng(hq + D + L + T + W)
    f = (lambda x: torch.from_numpy(x).to(torch.bfloat16).float().numpy()) if bf16 else (
        lambda x: x.astype(np.float16))
    q, k, v = (f(r.standard_normal(s).astype(np.float32))
               for s in ((hq, L, D), (hkv, T, D), (hkv, T, D)))
    lists = _lists(r, kind, L, W, T)
    lists[::5, 3::11] = -1
    lists[::7, 5::13] = T + 4
    lengths = np.where(np.arange(L) % 9 == 4, r.integers(0, W, L), W).astype(np.int32)
    lengths[2] = 0
    out = _run(q, k, v, lists, lengths, D ** -0.5, bf16)
    assert np.all(out[:, 2] == 0)
    _check(out, q, k, v, lists, lengths, D ** -0.5, bf16, f"{kind} D={D} L={L}")


@pytest.mark.parametrize("bf16", [False, True])
def test_a_key_listed_twice_counts_twice(bf16):
    r = rng(3)
    hq, hkv, D, L, T, W = 24, 4, 128, 100, 5000, 2200
    f = (lambda x: torch.from_numpy(x).to(torch.bfloat16).float().numpy()) if bf16 else (
        lambda x: x.astype(np.float16))
    q, k, v = (f(r.standard_normal(s).astype(np.float32))
               for s in ((hq, L, D), (hkv, T, D), (hkv, T, D)))
    lists = _lists(r, "shared", L, W, T)
    lists[50, 7] = lists[50, 2080]
    lengths = np.full(L, W, np.int32)
    out = _run(q, k, v, lists, lengths, 0.1, bf16)
    _check(out, q, k, v, lists, lengths, 0.1, bf16, "a key twice")


@pytest.mark.parametrize("dt,hq,hkv,D,L,T,W,served", [
    ("f32", 24, 3, 128, 1100, 16000, 256, False),   # every union but the last, short group's too large
    ("bf16", 8, 8, 128, 384, 30000, 256, False),
    ("f32", 4, 2, 256, 200, 4000, 256, False),      # (no whole group served)
    ("bf16", 8, 8, 128, 600, 30000, 512, True),     # an eighth of the groups left, the others served
    ("f32", 24, 4, 256, 300, 30000, 700, True),
])
def test_typed_rows_left_in_part_or_together(dt, hq, hkv, D, L, T, W, served):
    """Unions past the limit: more than a quarter of the groups takes the others along."""
    import qw_amd

    c = {"bf16": 1, "f32": 2}[dt]
    NR, limit = min(32, 128 // (hq // hkv)) & ~1, qw_amd.lib().qw_dlsa_union_keys(c, c, L, W, hq, hkv, D, T)
    r = rng(D + L + T)
    own = L // 8 if served else L
    lists = np.stack([np.sort(r.permutation(T)[:W]) for _ in range(own)] +
                     [np.sort(r.permutation(T)[:W])] * (L - own)).astype(np.int32)
    unions = [len(np.unique(lists[g:g + NR])) for g in range(0, L, NR)]
    left = sum(n > limit for n in unions)
    assert 0 < limit < max(unions) and (0 < 4 * left <= len(unions) if served else 4 * left > len(unions))
    dev = [torch.from_numpy(r.standard_normal(s).astype(np.float32)).to(TYPES[dt]).cuda()
           for s in ((hq, L, D), (hkv, T, D), (hkv, T, D))]
    q, k, v = (x.float().cpu().numpy() for x in dev)
    lengths = np.full(L, W, np.int32)
    out = qw_amd.sparse_attention_typed(*dev, _gpu(lists), _gpu(lengths), D ** -0.5)[0].float().cpu().numpy()
    rows = np.unique(np.append(np.arange(0, L, 7), L - 1))
    ref = oracle.dlsa_attention_f64(q[:, rows], k, v, lists[rows], lengths[rows], D ** -0.5)
    bound = np.abs(ref) * ROUND[dt] + 1e-5 * np.linalg.norm(ref, axis=-1, keepdims=True) + 1e-7
    assert np.isfinite(out).all() and np.all(np.abs(out[:, rows].astype(np.float64) - ref) <= bound)


def _fp16_inputs(r, hq, hkv, D, L, T):
    return (r.standard_normal(s).astype(np.float16) for s in ((hq, L, D), (hkv, T, D), (hkv, T, D)))


def _check_some(out, q, k, v, lists, lengths, scale, what):
    """Every 23rd row and the last (the float64 restatement of a whole call would take minutes)."""
    rows = np.unique(np.append(np.arange(0, len(lists), 23), len(lists) - 1))
    assert np.isfinite(out).all(), what
    _check(out[:, rows], q[:, rows], k, v, lists[rows], lengths[rows], scale, False, what)


@pytest.mark.parametrize("hq,hkv,D,L,T,W,left", [
    (24, 4, 256, 1400, 40000, 2200, "all"),     # every union too large: all groups handed over
    (24, 4, 256, 1400, 40000, 2200, "half"),    # more than a quarter: the others with them
    (24, 4, 256, 1400, 40000, 2200, "eighth"),  # served in part; a split tail of six groups
    (24, 4, 256, 1400, 90000, 2200, "none"),    # three bitmap passes
    (24, 4, 128, 2000, 30000, 3100, "eighth"),
])
def test_fp16_rows_over_many_keys(hq, hkv, D, L, T, W, left):
    assert _takes_it(hq, hkv, D, L, T, W), "a shape of the kernel"
    r = rng(L + T + D)
    q, k, v = _fp16_inputs(r, hq, hkv, D, L, T)
    n = {"all": L, "half": L // 2, "eighth": L // 8, "none": 0}[left]
    lists = np.concatenate([_lists(r, "own", n, W, T).reshape(n, W) if n else np.zeros((0, W), np.int32),
                            _lists(r, "sliding", L - n, W, T)] if n < L else [_lists(r, "own", L, W, T)])
    lists = np.ascontiguousarray(np.roll(lists, L // 3, axis=0))  # away from the groups' start
    lengths = np.full(L, W, np.int32)
    out = _run(q, k, v, lists, lengths, D ** -0.5, False)
    _check_some(out, q, k, v, lists, lengths, D ** -0.5, f"{left} left, T={T}")


def test_duplicates_in_a_third_of_the_groups():
    """More than a quarter of the groups list a key twice, in an fp16 call whose tail is split."""
    hq, hkv, D, L, T, W = 24, 4, 256, 700, 4000, 1600
    assert _takes_it(hq, hkv, D, L, T, W), "a shape of the kernel"
    r = rng(12)
    q, k, v = _fp16_inputs(r, hq, hkv, D, L, T)
    lists = _lists(r, "sliding", L, W, T)
    lists[::60, 5] = lists[::60, 4]  # one row of every third group of 20
    lengths = np.full(L, W, np.int32)
    _check_some(_run(q, k, v, lists, lengths, 1 / 16, False), q, k, v, lists, lengths, 1 / 16, "duplicates")


def test_non_finite_groups_do_not_move_the_others():
    """Infinite values in the first 30 of 70 groups (their outputs are left to the row kernel): the
    other groups, later workgroups and a split tail among them, give the clean call's bits."""
    hq, hkv, D, L, T, W = 24, 4, 256, 1400, 13000, 2200
    assert _takes_it(hq, hkv, D, L, T, W), "a shape of the kernel"
    r = rng(13)
    q, k, v = _fp16_inputs(r, hq, hkv, D, L, T)
    lists = _lists(r, "sliding", L, W, T - 1)
    lists[:600, 0] = T - 1
    lengths = np.full(L, W, np.int32)
    clean = _run(q, k, v, lists, lengths, 1 / 16, False)
    _check_some(clean, q, k, v, lists, lengths, 1 / 16, "clean")
    v[:, T - 1] = np.inf
    for _ in range(3):
        out = _run(q, k, v, lists, lengths, 1 / 16, False)
        assert not np.isfinite(out[:, :600]).any()
        np.testing.assert_array_equal(out[:, 600:], clean[:, 600:])


@pytest.mark.parametrize("bf16", [False, True])
def test_infinite_values_stay_with_the_rows_that_list_them(bf16):
    r = rng(4)
    hq, hkv, D, L, T, W = 24, 4, 128, 100, 5000, 2200
    f = (lambda x: torch.from_numpy(x).to(torch.bfloat16).float().numpy()) if bf16 else (
        lambda x: x.astype(np.float16))
    q, k, v = (f(r.standard_normal(s).astype(np.float32))
               for s in ((hq, L, D), (hkv, T, D), (hkv, T, D)))
    lists = np.stack([r.permutation(T - 1)[:W] for _ in range(2)])[np.zeros(L, int)].astype(np.int32)
    lists[41, 3] = T - 1
    v[:, T - 1, 5] = np.inf
    lengths = np.full(L, W, np.int32)
    out = _run(q, k, v, lists, lengths, 0.1, bf16)
    rows = np.setdiff1d(np.arange(L), [40, 41])  # (row 40 is row 41's pair in the row kernel)
    _check(out[:, rows], q[:, rows], k, np.where(np.isinf(v), 0, v), lists[rows], lengths[rows], 0.1,
           bf16, "rows without the infinite key")
    assert not np.isfinite(out[:, 41, 5]).any()


@pytest.mark.parametrize("qt,kt", [("f32", "f32"), ("bf16", "f16"), ("f16", "f32"), ("f32", "bf16"),
                                   ("f16", "bf16"), ("f16", "f16")])
@pytest.mark.parametrize("hq,hkv,D,L,T,W,kind", [
    (24, 4, 256, 101, 3000, 300, "sliding"),   # 32-key tiles; the last group one row
    (16, 2, 128, 96, 900, 128, "shared"),      # the union exactly two tiles
    (16, 2, 128, 96, 900, 129, "own"),
    (16, 2, 128, 70, 900, 129, "own"),         # (row by row: split lists)
    (8, 8, 64, 99, 2000, 333, "mixed"),        # G = 1
    (6, 1, 32, 200, 2000, 500, "sliding"),     # 256-key tiles
])
def test_typed_rows_match_float64(qt, kt, hq, hkv, D, L, T, W, kind):
    """fp32 arithmetic: 1e-5 of the row, as the reference holds its f32 read (dlsa_attention.rs:
    213-255), and the output's rounding."""
    import qw_amd

    print(f"case q={qt} kv={kt} hq={hq} hkv={hkv} D={D} L={L} W={W} {kind}", flush=True)
    c = {"f16": 0, "bf16": 1, "f32": 2}
    here = qw_amd.lib().qw_dlsa_union_keys(c[qt], c[kt], L, W, hq, hkv, D, T) > 0
    assert here == (L != 70 and (qt != kt or qt != "f16" or D == 32)), "the kernel of the call"
    r = rng(hq + D + L + T + W)
    dev = [torch.from_numpy(r.standard_normal(s).astype(np.float32)).to(TYPES[t]).cuda()
           for s, t in (((hq, L, D), qt), ((hkv, T, D), kt), ((hkv, T, D), kt))]
    q, k, v = (x.float().cpu().numpy() for x in dev)
    lists = _lists(r, kind, L, W, T)
    lists[::5, 3::11] = -1
    lists[::7, 5::13] = T + 4
    lengths = np.where(np.arange(L) % 9 == 4, r.integers(0, W, L), W).astype(np.int32)
    lengths[2] = 0
    out = qw_amd.sparse_attention_typed(*dev, _gpu(lists), _gpu(lengths), D ** -0.5)[0]
    assert out.dtype == TYPES[qt]
    out = out.float().cpu().numpy()
    assert np.all(out[:, 2] == 0)
    ref = oracle.dlsa_attention_f64(q, k, v, lists, lengths, D ** -0.5)
    bound = np.abs(ref) * ROUND[qt] + 1e-5 * np.linalg.norm(ref, axis=-1, keepdims=True) + 1e-7
    assert np.isfinite(out).all() and np.all(np.abs(out.astype(np.float64) - ref) <= bound)


@pytest.mark.parametrize("D", [64, 128, 256])
def test_bf16_weights_keep_32_bits(D):
    """Two keys whose scores differ by 2^-13, of opposite values, and a third of value 0 above them:
    what is left is the difference of two weights of about 0.7, some 3e-5, and weights held in 16
    bits (2^-18 of them each) are up to 2e-6 off. Bound: the output's rounding, half a unit of 2^-8
    relative, and 3e-7 for 32-bit scores, exponentials and sums (five roundings of 2^-24)."""
    import qw_amd

    hq, hkv, L, T, W = 24, 4, 64, 2000, 400
    assert _takes_it(hq, hkv, D, L, T, W, "bf16"), "a shape of the kernel"
    f = lambda x: torch.from_numpy(x).to(torch.bfloat16)  # noqa: E731
    q = np.zeros((hq, L, D), np.float32)
    q[:, :, 0], q[:, :, 1] = np.linspace(0.25, 1.0, L), 2.0 ** -6
    k, v = np.zeros((2, hkv, T, D), np.float32)
    k[:, :, 0] = -16384
    k[:, 2, 0], k[:, 5, 0], k[:, 9, 0], k[:, 9, 1] = 3, 1, 1, -2.0 ** -5
    v[:, 5], v[:, 9] = 1, -1
    q, k, v = f(q), f(k), f(v)
    lists = np.tile(np.arange(W, dtype=np.int32), (L, 1))
    lengths = np.full(L, W, np.int32)
    out = qw_amd.sparse_attention_typed(q.cuda(), k.cuda(), v.cuda(), _gpu(lists), _gpu(lengths), 0.25)[0]
    s = 0.25 * (q[:, :, 0].double().numpy()[..., None] * np.array([3, 1, 1]) - np.array([0, 0, 2.0 ** -11]))
    w = np.exp(s - s[..., :1])
    ref = ((w[..., 1] - w[..., 2]) / w.sum(axis=-1))[..., None]
    assert np.all(np.abs(out.double().cpu().numpy() - ref) <= np.abs(ref) * 2.0 ** -8 + 3e-7)
