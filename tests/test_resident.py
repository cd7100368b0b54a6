"""The resident schedule of SpMM (slices of B in LDS) at the edges of its tiles: rows and columns that do not fill a workgroup,
a slice or a tile, rows longer than what is loaded ahead, columns that do not ascend, duplicates, empty rows."""
import numpy as np
import pytest

import dlspm_hip as dl
import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def pattern(kind, M, K, density, seed):
    rng = np.random.default_rng(seed)
    share = np.full(M, density)
    if kind == "uneven":
        share = np.clip(density * np.exp(rng.normal(0.0, 0.8, M)), 0.0, 1.0)
        share[::17] = 0.0
        share[5::64] = 1.0  # full rows: more in a slice than is loaded ahead
    keep = rng.random((M, K), dtype=np.float32) < share[:, None]
    ro = np.concatenate(([0], np.cumsum(keep.sum(1)))).astype(np.int32)
    ci = np.nonzero(keep)[1].astype(np.int32)
    if kind == "unordered":  # whole rows shuffled, and a column that comes twice
        for r in range(0, M, 3):
            rng.shuffle(ci[ro[r]:ro[r + 1]])
        for r in range(1, M, 5):
            if ro[r + 1] - ro[r] > 1:
                ci[ro[r + 1] - 1] = ci[ro[r]]
    return ro, ci


def sequential_row(ro, ci, va, B, r):
    """fma by fma in CSR order (80-bit products and sums rounded to 32 bits at every step)"""
    acc = np.zeros(B.shape[1], np.float32)
    for j in range(ro[r], ro[r + 1]):
        acc = (np.longdouble(va[j]) * B[ci[j]].astype(np.longdouble) + acc.astype(np.longdouble)).astype(np.float32)
    return acc


CASES = [(4001, 1023, 197), (2048, 512, 392), (2017, 610, 510), (1025, 1024, 784), (8129, 2049, 100), (12289, 609, 130), (65, 304, 9001)]


@pytest.mark.parametrize("M,K,N", CASES)
@pytest.mark.parametrize("kind,density", [("even", 0.3), ("uneven", 0.4), ("unordered", 0.35), ("even", 0.9)])
def test_against_oracle_and_order(M, K, N, kind, density):
    ro, ci = pattern(kind, M, K, density, M + N)
    rng = np.random.default_rng(1)
    va, B = rng.normal(size=ci.size).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    guard = torch.full((M * N + 64,), 7.0, device="cuda")
    out = guard[:M * N].view(M, N)
    args = (d(ro), d(ci), d(va), d(B))
    dl.spmm(*args, out=out)
    got = out.cpu().numpy()
    assert bool((guard[M * N:] == 7.0).all())
    assert oracle.rel_frobenius(got, oracle.spmm(ro, ci, va, B)) <= 1e-5
    again = dl.spmm(*args).cpu().numpy()
    assert np.array_equal(got, again)
    dl.set_tuning(rules_off=dl.RULES["resident_slices"])
    try:
        other = dl.spmm(*args).cpu().numpy()
    finally:
        dl.set_tuning()
    resident = not np.array_equal(got, other)
    if kind != "uneven" and (M, K, N) != (65, 304, 9001):
        assert resident  # these sizes are in the schedule's range
    if resident:
        for r in (0, 1, 5, 17, 63, 64, M // 2, M - 1):
            if r < M:
                assert np.array_equal(got[r], sequential_row(ro, ci, va, B, r)), r


@pytest.mark.parametrize("how", ["even", "row_plan", "cut_plan", "memory"])
def test_every_way_of_calling(how):
    M, K, N = 4096, 1024, 256
    ro, ci = pattern("even", M, K, 0.4, 3)
    rng = np.random.default_rng(2)
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    args = (d(ro), d(ci), d(rng.normal(size=ci.size).astype(np.float32)), d(rng.normal(size=(K, N)).astype(np.float32)))
    want = dl.spmm(*args)
    kwargs = {"even": {"workspace": dl.ROWS_EVEN}, "row_plan": {"plan": dl.row_plan(args[0])},
              "cut_plan": {"plan": dl.cut_plan(args[0], dl.OP_SPMM, N)},
              "memory": {"workspace": torch.empty(max(16, dl.workspace_bytes(dl.OP_SPMM, M, K, N, ci.size)), dtype=torch.uint8, device="cuda")}}[how]
    assert torch.equal(dl.spmm(*args, **kwargs), want)


def test_rows_of_b_that_nothing_refers_to():
    """An infinity in a row of B counts only where a nonzero refers to it."""
    M, K, N = 4096, 1000, 200
    ro, ci = pattern("even", M, K, 0.3, 4)
    ci = np.where(ci == 17, 18, ci).astype(np.int32)
    rng = np.random.default_rng(5)
    va, B = rng.normal(size=ci.size).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)
    B[17] = np.inf
    B[17, ::3] = np.nan
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    got = dl.spmm(d(ro), d(ci), d(va), d(B)).cpu().numpy()
    B[17] = 0.0
    assert oracle.rel_frobenius(got, oracle.spmm(ro, ci, va, B)) <= 1e-5
