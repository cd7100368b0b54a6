"""The fused op's groups of sixteen rows on the matrix cores: windows of every alignment, and what sends a group back to the
row-by-row path."""
import numpy as np
import pytest

import dlspm_hip as dl
import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def window(M, K, band, seed, holes=0.0):
    rng = np.random.default_rng(seed)
    first = np.clip(np.arange(M) * K // M - band // 2, 0, K)
    end = np.clip(np.arange(M) * K // M - band // 2 + band, 0, K)
    rows = [np.arange(a, b) for a, b in zip(first, end)]
    if holes:
        rows = [r[rng.random(r.size) >= holes] for r in rows]
    ro = np.concatenate(([0], np.cumsum([r.size for r in rows]))).astype(np.int32)
    return ro, np.concatenate(rows).astype(np.int32), rng


def run(ro, ci, Q, Km, V, scale):
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    args = (d(ro), d(ci), d(Q), d(Km), d(V), scale)
    got = dl.fused(*args).cpu().numpy()
    dl.set_tuning(rules_off=dl.RULES["dense_groups"])
    try:
        other = dl.fused(*args).cpu().numpy()
    finally:
        dl.set_tuning()
    return got, other


@pytest.mark.parametrize("M,K,band,D,holes", [(16385, 16384, 128, 64, 0.0), (9001, 9007, 250, 80, 0.1), (20000, 18000, 97, 128, 0.4),
                                              (24581, 24581, 289, 36, 0.0), (24581, 24581, 290, 36, 0.0), (40000, 9000, 65, 48, 0.2),
                                              (13000, 13000, 100, 96, 0.6), (5000, 3000, 260, 96, 0.0), (70000, 5000, 40, 44, 0.0)])
def test_windows(M, K, band, D, holes):
    ro, ci, rng = window(M, K, band, M + D, holes)
    ro[-1] = ci.size
    Q, Km, V = (rng.normal(size=(n, D)).astype(np.float32) for n in (M, K, K))
    got, other = run(ro, ci, Q, Km, V, 0.125)
    assert oracle.rel_frobenius(got, oracle.fused(ro, ci, Q, Km, V, 0.125)) <= 1e-5
    on = not np.array_equal(got, other)
    assert on == (ci.size * D >= 1.2e8 and 12 * ci.size <= M * K)
    if on:  # rows past the last whole group of sixteen are left to the row-by-row path
        assert np.array_equal(got[M // 16 * 16:], other[M // 16 * 16:])


@pytest.mark.parametrize("what", ["unordered", "twice", "inf", "far", "empty"])
def test_what_is_left_to_the_row_by_row_path(what):
    M = K = 16384
    D, band = 64, 128
    ro, ci, rng = window(M, K, band, 7)
    Q, Km, V = (rng.normal(size=(n, D)).astype(np.float32) for n in (M, K, K))
    rows = np.arange(100, M, 160)  # one row in every tenth group
    groups = np.unique(rows // 16)
    for r in rows:
        lo, hi = ro[r], ro[r + 1]
        if what == "unordered":
            rng.shuffle(ci[lo + 1:hi - 1])  # inside the span: still taken
        elif what == "twice":
            ci[lo + 5] = ci[lo + 6]
        elif what == "far":
            ci[hi - 2] = (r + K // 2) % K  # not at the end of the row: outside the span that its ends say
    if what == "inf":
        V[rows[:5]] = np.inf
    if what == "empty":
        keep = np.ones(ci.size, bool)
        for r in rows:
            keep[ro[r]:ro[r + 1]] = False
        counts = np.diff(ro)
        counts[rows] = 0
        ro, ci = np.concatenate(([0], np.cumsum(counts))).astype(np.int32), ci[keep]
    got, other = run(ro, ci, Q, Km, V, 0.5)
    if what == "inf":
        fine = np.isfinite(other)
        assert np.array_equal(fine, np.isfinite(got)) and np.array_equal(np.isnan(got), np.isnan(other))
        got, other = np.where(fine, got, 0.0), np.where(fine, other, 0.0)
    else:
        assert oracle.rel_frobenius(got, oracle.fused(ro, ci, Q, Km, V, 0.5)) <= 1e-5
    assert np.linalg.norm(got - other) <= 1e-5 * np.linalg.norm(other)
    if what in ("twice", "far"):
        assert np.linalg.norm(got[groups[3] * 16:groups[3] * 16 + 16] - other[groups[3] * 16:groups[3] * 16 + 16]) <= 1e-6 * np.linalg.norm(other[groups[3] * 16:groups[3] * 16 + 16])
