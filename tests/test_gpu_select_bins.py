"""The K1 select's score bins (dlsa_select.hip) at the edges of what they take: score shapes that
fill one bin just within and just past its limit, ranges that are infinite, vanish or overflow, a
wanted bin that reaches past the picks, rows as long as the threads' registers hold and one
longer. Exact against the oracle, for workgroups of 64 to 1024 threads."""
import numpy as np
import pytest

from conftest import rng
from test_gpu_dlsa_select import QWEN, _check, _members

pytestmark = pytest.mark.gpu


def _shapes(r, n):
    base = r.standard_normal(n).astype(np.float32)
    top = np.sort(base)[::-1]
    yield "normal", base
    for same in (63, 64, 65, 255, 256, 257, 500):               # equal scores in a wanted bin
        s = base.copy()
        s[r.choice(n, min(n, same), replace=False)] = top[3]
        yield f"{same} equal", s
        s = base.copy()
        s[r.choice(n, min(n, same), replace=False)] = top[min(n - 1, 1023)]
        yield f"{same} equal at the threshold", s
    s = base.copy()
    s[r.random(n) < 0.4] = -np.inf
    yield "-inf", s
    s = base.copy()
    s[5] = np.inf
    yield "+inf", s
    yield "all -inf", np.full(n, -np.inf, np.float32)
    yield "one value", np.full(n, 0.25, np.float32)
    yield "signed zeros", np.where(r.random(n) < 0.5, 0.0, -0.0).astype(np.float32)
    yield "tiny range", (base * 1e-38).astype(np.float32)
    yield "overflowing range", (base * 1e38).astype(np.float32)
    yield "an outlier", np.where(np.arange(n) == n // 2, 1e20, base).astype(np.float32)
    s = base.copy()
    s[7] = np.nan
    yield "nan", s
    yield "descending", top.copy()
    s = base.copy()
    s[::3] = np.finfo(np.float32).min
    yield "a third masked", s
    s = base.copy()
    s[:n // 2] = -1e4
    yield "the first half masked", s
    s[n // 2:] = np.where(r.random(n - n // 2) < 0.9, -np.inf, s[n // 2:])
    yield "few finite", s
    for k in (3, 4, 70, 300):                        # fewer than the groups of lanes, as many, more than a bin
        s = base.copy()
        s[r.choice(n, min(n, k), replace=False)] = np.inf if k == 3 else 1e3
        yield f"{k} outliers", s
    yield "heavy tail", np.exp(3 * base)


@pytest.mark.parametrize("t,threads", [(1024, 64), (8704, 64), (8704, 256), (8704, 1024),
                                       (8192, 64), (9216, 64), (131072, 1024), (131584, 1024)])
def test_bins_match_oracle(oracle_lib, t, threads):
    r = rng(t + threads)
    n = t // 512 * 64
    members = _members(r, QWEN, n)
    rows = list(_shapes(r, n))
    print(f"case t={t} threads={threads} shapes={len(rows)}", flush=True)
    scores = np.stack([s for _, s in rows])
    positions = np.full(len(rows), t + 7, np.int32)
    _check(oracle_lib, scores, members, positions, n, QWEN, threads, f"t={t} threads={threads}")
    p = dict(QWEN, top_p=2048, top_k=9000)
    _check(oracle_lib, scores, members, positions, n, p, threads, f"t={t} top_p 2048")
