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


# Error against 64 bits, of the matrix cores and of the row-by-row path: chains of D / 8 for the scores on both; for the
# rows four chains of sixteen per block of 64 columns, against two to eight chains over the whole row.
@pytest.mark.parametrize("M,band,D", [(16384, 128, 128), (16384, 256, 64), (9000, 260, 112), (24000, 220, 44)])
def test_no_less_precise_than_row_by_row(M, band, D):
    ro, ci, rng = window(M, M, band, M + D)
    Q, Km, V = (rng.normal(size=(M, D)).astype(np.float32) for _ in range(3))
    got, other = run(ro, ci, Q, Km, V, 0.125)
    rows = slice(M // 2, M // 2 + 512)
    scores = np.zeros((512, M))
    for i, r in enumerate(range(rows.start, rows.stop)):
        c = ci[ro[r]:ro[r + 1]]
        scores[i, c] = 0.125 * (Km[c].astype(np.float64) @ Q[r].astype(np.float64))
    want = scores @ V.astype(np.float64)
    here, there = (np.linalg.norm(x[rows] - want) / np.linalg.norm(want) for x in (got, other))
    assert not np.array_equal(got, other)
    assert here <= 1.6e-7 and here <= 1.02 * there, (here, there)


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("M,band,D", [(16385, 128, 64), (9001, 260, 112)])
def test_operands_on_any_float(M, band, D, off):
    """every operand one, two or three floats behind a 16-byte boundary: the same bits, and nothing written outside O"""
    ro, ci, rng = window(M, M, band, 3)
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    args = [d(ro), d(ci)] + [d(rng.normal(size=(M, D)).astype(np.float32)) for _ in range(3)]
    assert dl.describe_schedule(dl.OP_FUSED, M, M, D, ci.size)["schedule"] == "dense_groups"
    want = dl.fused(*args, 0.125)

    def shifted(t):
        room = torch.full((t.numel() + 8,), 7, dtype=t.dtype, device="cuda")
        view = room[off:off + t.numel()].view(t.shape)
        view.copy_(t)
        return room, view

    room, out = shifted(torch.zeros_like(want))
    dl.fused(*(shifted(t)[1] for t in args), 0.125, out=out)
    assert torch.equal(out, want)
    assert bool((room[:off] == 7).all()) and bool((room[off + want.numel():] == 7).all())


@pytest.mark.parametrize("where", ["Q", "K", "V", "scale inf", "scale nan", "overflow", "tiny scores", "tiny V"])
def test_values_that_are_not_finite_or_tiny(where):
    """what is not finite lies where it lies row by row, in the same kind; subnormal scores and results are kept"""
    M, band, D = 16384, 128, 64
    ro, ci, rng = window(M, M, band, 7)
    Q, Km, V = (rng.normal(size=(M, D)).astype(np.float32) for _ in range(3))
    scale, bad = 0.5, np.arange(100, M, 3000)
    if where in ("Q", "K", "V"):
        x = {"Q": Q, "K": Km, "V": V}[where]
        x[bad[::2], 3], x[bad[1::2], 5] = np.inf, np.nan
    elif where.startswith("scale"):
        scale = float(where.split()[1])
    elif where == "overflow":
        Q[bad], V[bad] = 1e30, 1e30
    elif where == "tiny scores":
        Q *= np.float32(1e-25)
        Km *= np.float32(1e-15)
        V *= np.float32(1e10)
    else:
        V *= np.float32(1e-39)
    got, other = run(ro, ci, Q, Km, V, scale)
    fine = np.isfinite(other)
    assert np.array_equal(fine, np.isfinite(got)) and np.array_equal(np.isnan(other), np.isnan(got))
    if where.startswith("tiny"):  # (half a unit of 1.4e-45 in each of 128 terms)
        assert np.abs(other).max() > 0 and np.linalg.norm(got - other) <= 1e-3 * np.linalg.norm(other)
    elif fine.any():
        assert np.linalg.norm(got[fine].astype(np.float64) - other[fine]) <= 1e-5 * np.linalg.norm(other[fine].astype(np.float64))


@pytest.mark.parametrize("M,D", [(20000, 64), (16395, 112)])
def test_groups_led_by_workgroups_of_other_rows(M, D):
    """Runs of window rows between rows with scattered columns, rows longer than a group's columns (all of them twice) and rows without
    any: who leads a group is not who owns its row blocks, and what a group is must come out the same for both."""
    K, band = M, 200
    ro, ci, rng = window(M, K, band, M)
    rows = np.split(ci, ro[1:-1])
    kind = rng.integers(0, 5, M // 48 + 1)
    for r in range(M):
        if kind[r // 48] == 1:
            rows[r] = np.sort(rng.choice(K, rows[r].size, replace=False)).astype(np.int32)
        elif kind[r // 48] == 2 and r % 16 == 5:
            rows[r] = np.repeat(rows[r], 2)
        elif kind[r // 48] == 3 and r % 7 == 0:
            rows[r] = rows[r][:0]
    ro = np.concatenate(([0], np.cumsum([r.size for r in rows]))).astype(np.int32)
    ci = np.concatenate(rows)
    Q, Km, V = (rng.normal(size=(n, D)).astype(np.float32) for n in (M, K, K))
    got, other = run(ro, ci, Q, Km, V, 0.125)
    assert oracle.rel_frobenius(got, oracle.fused(ro, ci, Q, Km, V, 0.125)) <= 1e-5  # (as in test_windows)
    differ = (got != other).any(axis=1)[:M // 16 * 16].reshape(-1, 16)
    whole = np.array([[kind[(g * 16 + i) // 48] for i in range(16)] for g in range(M // 16)])
    assert differ[(whole == 0).all(axis=1)].any(axis=1).all()  # on the matrix cores
    assert not differ[(whole == 1).all(axis=1)].any()          # row by row


@pytest.mark.parametrize("D", [36, 64, 68, 96, 100, 128])
def test_widths_whole_and_ragged(D):
    """Q goes through LDS a whole number of times per thread, or once and a half (D = 65 ... 96): every row of a group is there"""
    ro, ci, rng = window(20003, 20003, 200, D, 0.02)
    Q, Km, V = (rng.normal(size=(20003, D)).astype(np.float32) for _ in range(3))
    got, other = run(ro, ci, Q, Km, V, 0.125)
    differ = (got != other).any(axis=1)[:20000]
    assert differ.mean() > 0.99
    # row by row: each row's own error is that of its chains (as in test_no_less_precise_than_row_by_row, of one row: three times the mean)
    off = np.linalg.norm(got - other, axis=1) / np.linalg.norm(other, axis=1)
    assert off.max() <= 2e-6, off.max()
