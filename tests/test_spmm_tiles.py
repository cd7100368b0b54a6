"""SpMM on dense tiles: edges of the tiles, and what sends a row back to its floats."""
import numpy as np
import pytest

import dlspm_hip as dl


def tiles(M, K, N, nnz, size=1 << 40):
    return dl.describe_schedule(dl.OP_SPMM, M, K, N, nnz, workspace_bytes=size | dl.HINT_ROWS_EVEN)["schedule"] == "dense_tiles"


def test_who_runs_on_tiles():
    M, K, N = 16384, 8192, 128
    nnz = M * 2457
    need = K * N * 6 + K // 16 * N // 32 * 8
    cp = dl.advise(dl.OP_SPMM, N, dl.MatrixInfo(M, K, nnz, 2600, 0, K, 8000, 1000))
    assert (cp.build, cp.bytes, cp.hints) == (dl.BUILD_NOTHING, need, dl.HINT_ROWS_EVEN)
    shape = dl.describe_schedule(dl.OP_SPMM, M, K, N, nnz, workspace_bytes=need | dl.HINT_ROWS_EVEN)
    assert shape == {"schedule": "dense_tiles", "rows": 64, "slice_rows": 0, "chunks": 0, "tile_columns": 128}
    # less memory, none, no word about the rows, a band, or few nonzeros: as before
    for size in ((need - 1) | dl.HINT_ROWS_EVEN, dl.HINT_ROWS_EVEN, 1 << 40, 1 << 40 | dl.HINT_ROWS_EVEN | dl.HINT_BANDED):
        assert dl.describe_schedule(dl.OP_SPMM, M, K, N, nnz, workspace_bytes=size)["schedule"] == "resident"
    assert not tiles(M, K, N, M * 819) and not tiles(2048, 512, 256, 2048 * 102)
    uneven = dl.advise(dl.OP_SPMM, N, dl.MatrixInfo(M, K, nnz, 6000, 0, K, 8000, 1000))
    assert not uneven.hints & dl.HINT_ROWS_EVEN
    for rule in ("dense_groups", "resident_slices"):
        dl.set_tuning(rules_off=dl.RULES[rule])
        assert not tiles(M, K, N, nnz)
    dl.set_tuning()


def matrix(M, K, N, density, seed):
    rng = np.random.default_rng(seed)
    keep = rng.random((M, K)) < density
    ro = np.concatenate(([0], np.cumsum(keep.sum(1)))).astype(np.int32)
    ci = np.nonzero(keep)[1].astype(np.int32)
    return ro, ci, rng.normal(size=ci.size).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32), rng


def run(ro, ci, va, B):
    """on tiles, and from slices of B"""
    import torch

    M, (K, N), guard = ro.size - 1, B.shape, 256
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    need = -(-N // 32) * -(-K // 128) * 8 * (3072 + 8)
    assert tiles(M, K, N, ci.size, need)
    memory = torch.full((need + guard,), 77, dtype=torch.uint8, device="cuda")
    args = tuple(d(a) for a in (ro, ci, va, B))
    got = dl.spmm(*args, plan=dl.Prepared(memory, need | dl.HINT_ROWS_EVEN, None))
    assert bool((memory[need:] == 77).all())
    return got.cpu().numpy(), dl.spmm(*args, workspace=dl.ROWS_EVEN).cpu().numpy()


SIZES = [(1000, 511, 2100, 0.95), (16321, 1000, 128, 0.3), (3000, 770, 1030, 0.6), (16384, 513, 96, 0.95), (16384, 640, 127, 0.8),
         (20000, 1024, 101, 0.45), (1000, 640, 4100, 0.7), (4096, 1024, 512, 0.4)]


# Error against 64 bits: sums of four products of sixteen each in 32 bits, the rest in 64 bits, against chains of sixteen products in 32 bits
# from slices of B. Both are rounded once at the end (2^-25 of a result in the mean of squares and more: 2.5e-8).
@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,density", SIZES)
def test_edges_of_the_tiles(M, K, N, density):
    ro, ci, va, B, rng = matrix(M, K, N, density, M + N)
    got, other = run(ro, ci, va, B)
    assert not np.array_equal(got, other)
    for rows in (slice(0, 66), slice(M - 130, M), slice(M // 2, M // 2 + 64)):
        dense = np.zeros((rows.stop - rows.start, K))
        for i, r in enumerate(range(rows.start, rows.stop)):
            dense[i, ci[ro[r]:ro[r + 1]]] = va[ro[r]:ro[r + 1]]
        want = dense @ B.astype(np.float64)
        here, there = (np.linalg.norm(x[rows] - want) / np.linalg.norm(want) for x in (got, other))
        assert here <= 5e-8 and here <= 1.02 * there, (here, there)
        assert np.abs(got[rows] - want).max() <= 1e-6 * np.abs(want).max()
    assert np.linalg.norm(got - other) <= 2e-7 * np.linalg.norm(other)


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["unordered", "twice", "empty", "full", "unused inf", "inf", "nan", "overflow", "tiny values", "tiny B", "subnormal results"])
def test_what_is_computed_from_the_floats(what):
    M, K, N = 3000, 770, 1030
    ro, ci, va, B, rng = matrix(M, K, N, 0.6, 5)
    rows = np.arange(3, M, 77)
    for r in rows:
        a, b = ro[r], ro[r + 1]
        if what == "unordered":
            order = rng.permutation(b - a)
            ci[a:b], va[a:b] = ci[a:b][order], va[a:b][order]
        elif what == "twice":
            ci[a + 9], ci[b - 1] = ci[a + 10], ci[b - 2]
    if what in ("empty", "full"):
        keep = rng.random((M, K)) < 0.6
        keep[rows] = what == "full"
        ro, ci = np.concatenate(([0], np.cumsum(keep.sum(1)))).astype(np.int32), np.nonzero(keep)[1].astype(np.int32)
        va = rng.normal(size=ci.size).astype(np.float32)
    elif what == "unused inf":
        ci = np.where(ci == 17, 18, ci).astype(np.int32)  # (and column 18 twice in some rows)
        B[17] = np.inf
        B[17, ::3] = np.nan
    elif what in ("inf", "nan"):
        va[::100003], B[40, 7] = (np.inf, -np.inf) if what == "inf" else (np.nan, np.nan)
    elif what == "overflow":
        va[ro[rows]], B[:, 5] = 3e38, 3.4e38
    elif what == "tiny values":
        va[ro[rows]] = 1e-35
        va[ro[rows] + 1] = 1e-45
    elif what == "tiny B":
        B[:] *= np.float32(1e-36)
        B[5], B[:, 3] = 1e-40, 1e-44
        va *= np.float32(1e30)
    elif what == "subnormal results":
        B *= np.float32(1e-20)
        va *= np.float32(1e-20)
    with np.errstate(all="ignore"):
        got, other = run(ro, ci, va, B)
    dense = np.zeros((M, K))
    np.add.at(dense, (np.repeat(np.arange(M), np.diff(ro)), ci), va.astype(np.float64))
    if what == "unused inf":
        B[17] = 0.0
    if what in ("inf", "nan"):
        fine = np.isfinite(other)
        assert np.array_equal(fine, np.isfinite(got)) and np.array_equal(np.isnan(other), np.isnan(got))
        assert np.array_equal(got[~fine & ~np.isnan(other)], other[~fine & ~np.isnan(other)])
        got, want = np.where(fine, got, 0.0), np.where(fine, other, 0.0).astype(np.float64)
    else:
        want = dense @ B.astype(np.float64)
    if what == "empty":
        assert not got[rows].any()
    if what == "overflow":  # a sum that overflows on the way and not in the end is what it is in the end
        fine = np.abs(want) <= 3.4e38
        assert np.isfinite(got[fine]).all() and np.isfinite(other).sum() < fine.sum() < want.size
        got, want = np.where(fine, got / 1e30, 0.0), np.where(fine, want / 1e30, 0.0)
    # column by column, so that a column of small numbers counts like the others
    off, norm = np.linalg.norm(got - want, axis=0), np.linalg.norm(want, axis=0)
    if what == "subnormal results":
        # every product of sixteen is rounded to a multiple of 2^-149, six for each of the 49 steps and two ways: half a unit each
        # at most, a third in the mean of squares; from slices of B every one of the 462 products is
        assert norm.min() > 0 and np.abs(got - want).max() <= 6 * 49 * 2.0 ** -150
        assert (off <= 1.1 * np.linalg.norm(other - want, axis=0)).all()
    else:
        assert (off <= 3e-7 * norm).all()


@pytest.mark.gpu
@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("M,K,N,density", SIZES[2:5])
def test_operands_on_any_float(M, K, N, density, off):
    """every operand one, two or three floats behind a 16-byte boundary: the same bits, and nothing written outside C"""
    import torch

    ro, ci, va, B, _ = matrix(M, K, N, density, 9)
    args = [torch.from_numpy(a).cuda() for a in (ro, ci, va, B)]
    plan = dl.prepare(*args[:2], K, dl.OP_SPMM, N)
    assert dl.describe_schedule(dl.OP_SPMM, M, K, N, ci.size, plan=plan)["schedule"] == "dense_tiles"
    want = dl.spmm(*args, plan=plan)

    def shifted(t):
        room = torch.full((t.numel() + 8,), 7, dtype=t.dtype, device="cuda")
        view = room[off:off + t.numel()].view(t.shape)
        view.copy_(t)
        return room, view

    room, out = shifted(torch.zeros_like(want))
    dl.spmm(*(shifted(t)[1] for t in args), out=out, plan=plan)
    assert torch.equal(out, want)
    assert bool((room[:off] == 7).all()) and bool((room[off + want.numel():] == 7).all())


@pytest.mark.gpu
def test_one_plan_on_two_streams_and_in_a_graph():
    """Each call has memory of its own: calls that overlap in time do not meet in it."""
    import torch

    M, K, N, density = SIZES[7]
    ro, ci, va, B, rng = matrix(M, K, N, density, 2)
    args = [torch.from_numpy(a).cuda() for a in (ro, ci, va)]
    dense = [torch.from_numpy(rng.normal(size=(K, N)).astype(np.float32)).cuda() for _ in range(2)]
    plan = dl.prepare(*args[:2], K, dl.OP_SPMM, N)
    assert plan.memory is None and dl.describe_schedule(dl.OP_SPMM, M, K, N, ci.size, plan=plan)["schedule"] == "dense_tiles"
    want = [dl.spmm(*args, b, plan=plan) for b in dense]
    assert torch.equal(dl._spmm(*args, dense[0], plan=plan), want[0])  # (the calls through ctypes)
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(8):
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                got[i].append(dl.spmm(*args, dense[i], plan=plan))
    torch.cuda.synchronize()
    assert all(torch.equal(x, want[i]) for i in range(2) for x in got[i])
    b, out, graph = dense[0].clone(), torch.empty_like(want[0]), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        dl.spmm(*args, b, out=out, plan=plan)
    for i in (0, 1, 0, 1):
        b.copy_(dense[i])
        graph.replay()
        other = dl.spmm(*args, dense[1 - i], plan=plan)
        torch.cuda.synchronize()
        assert torch.equal(out, want[i]) and torch.equal(other, want[1 - i])


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["a row", "scattered", "everything", "one column", "explicit zeros", "large"])
@pytest.mark.parametrize("M,K,N,density", [SIZES[0], SIZES[2], SIZES[5]])
def test_values_of_B_that_have_no_parts(what, M, K, N, density):
    """Infinities, NaN and values that bf16 rounds to infinity reach the rows that use them, in the columns that hold them, as from
    slices of B; all other results are what they are with zeros in their place."""
    ro, ci, va, B, rng = matrix(M, K, N, density, 21)
    bad = np.zeros(B.shape, bool)
    if what in ("a row", "explicit zeros"):
        bad[K - 2] = True
    elif what == "scattered":
        bad[rng.integers(0, K, 40), rng.integers(0, N, 40)] = True
    elif what == "everything":
        bad[:] = True
    elif what == "one column":
        bad[:, N - 1] = True
    else:
        bad[rng.integers(0, K, 5), rng.integers(0, N, 5)] = True
    B[bad] = np.float32(3.4e38) if what == "large" else rng.choice(np.array([np.inf, -np.inf, np.nan, 3.4e38], np.float32), bad.sum(), p=[0.4, 0.3, 0.2, 0.1])
    if what == "explicit zeros":
        va[::3] = 0.0
    elif what == "large":
        va *= np.float32(0.1)  # (finite results)
    with np.errstate(all="ignore"):
        got, other = run(ro, ci, va, B)
    fine = np.isfinite(other)
    assert fine.any() == (what != "everything") and (what == "large" or not fine.all())
    if what == "large":
        assert fine.all() and np.isfinite(got).all()
        off, norm = np.linalg.norm((got - other) / 1e38, axis=0), np.linalg.norm(other / 1e38, axis=0)
        assert (off <= 3e-7 * norm + 1e-38).all()
        return
    # (a sum that overflows on the way only, from slices of B in 32 bits, is what it is in 64 bits here)
    sums = ~fine & np.isfinite(got)
    assert sums.sum() <= 1e-3 * got.size and np.array_equal(np.isfinite(got) & ~sums, fine)
    assert np.array_equal(np.isnan(got[~sums]), np.isnan(other[~sums]))
    infinite = np.isinf(other) & ~sums
    assert np.array_equal(got[infinite], other[infinite])
    small = fine & (np.abs(other) < 1e30)
    assert np.linalg.norm(np.where(small, got - other, 0)) <= 3e-7 * np.linalg.norm(np.where(small, other, 0)) + 1e-38


@pytest.mark.gpu
@pytest.mark.parametrize("small", [1e-33, 1e-36, 1e-44])
@pytest.mark.parametrize("where", ["A", "B", "both", "A, results of few terms"])
def test_values_too_small_for_their_parts(where, small):
    """Values below 2^-109 lose up to 2^-134 in their parts, which no result may show: the large ones because they are large, the small
    ones because they are computed from the floats."""
    M, K, N, density = SIZES[2]
    ro, ci, va, B, rng = matrix(M, K, N, density, 33)
    if where != "B":
        va[rng.random(ci.size) < 0.02] = small
    if where in ("B", "both"):
        B[rng.random(B.shape) < 0.02] = small
    if where == "A, results of few terms":  # whole columns of results that only such values make
        B[:, 7:40] = 0.0
        B[3, 7:40] = rng.normal(size=33)
        va[ci == 3] = np.where(rng.random((ci == 3).sum()) < 0.5, small, va[ci == 3])
    got, other = run(ro, ci, va, B)
    dense = np.zeros((M, K))
    dense[np.repeat(np.arange(M), np.diff(ro)), ci] = va
    want = dense @ B.astype(np.float64)
    # every result by itself: rounded once, or 2^-22 of what its terms come to together, or half of the smallest float
    terms = np.abs(dense) @ np.abs(B).astype(np.float64)
    assert (np.abs(got - want) <= 2.0 ** -22 * terms + 2.0 ** -149).all()
    few = (terms > 0) & (terms < 1e-30)
    assert few.any() == (where == "A, results of few terms")
    # (down to the smallest ones, which one term makes: exact but for the rounding of the product)
    assert (np.abs(got - want)[few] <= 2.0 ** -23 * terms[few] + 2.0 ** -149).all()


@pytest.mark.gpu
def test_memory_for_a_call_of_the_c_entry_point():
    """Prepared.for_call(): what a caller of the entry point passes, as the benchmark's host leg does, runs the schedule that
    dlspm_describe_schedule names for the plan; a plan of another op is given memory by both kinds of Python call."""
    import ctypes

    import torch

    M, K, N, density = SIZES[7]
    ro, ci, va, B, rng = matrix(M, K, N, density, 2)
    args = [torch.from_numpy(a).cuda() for a in (ro, ci, va, B)]
    plan = dl.prepare(*args[:2], K, dl.OP_SPMM, N)
    pointer, size = plan.for_call()
    assert pointer.value and size == plan.size_and_hints
    out, address = torch.empty((M, N), device="cuda"), lambda t: ctypes.c_void_p(t.data_ptr())
    st = dl.lib().spmm_csr_f32(M, K, N, ci.size, *(address(t) for t in args), address(out), pointer, size, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == dl.OK and torch.equal(out, dl.spmm(*args, plan=plan)) and not torch.equal(out, dl.spmm(*args, workspace=dl.ROWS_EVEN))
    lhs, rhs = torch.randn((M, 256), device="cuda"), torch.randn((K, 256), device="cuda")
    assert torch.equal(dl.sddmm(*args[:2], lhs, rhs, plan=plan), dl._sddmm(*args[:2], lhs, rhs, plan=plan))
    held = dl.prepare(*args[:2], K, dl.OP_SDDMM, 256)
    assert held.memory is None or held.for_call()[0].value == held.memory.data_ptr()


# one slice and two: nothing is left to place behind the first fill, and every load of B ahead is of the same slice
ONE_SLICE = [(16384, 100, 1024, 0.9), (16384, 128, 256, 0.9), (16384, 200, 1024, 0.5)]


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["ascending", "unordered", "one sign"])
@pytest.mark.parametrize("M,K,N,density", ONE_SLICE + SIZES[2:4])
def test_the_smallest_matrices_and_operands_of_one_sign(M, K, N, density, what):
    """As test_edges_of_the_tiles. Operands of one sign: a bias in the rounding of the matrix cores' sums would add up."""
    ro, ci, va, B, rng = matrix(M, K, N, density, 3 * M + N)
    if what == "one sign":
        va, B = np.abs(va), np.abs(B)
    elif what == "unordered":
        for r in range(5, M, 301):
            order = rng.permutation(ro[r + 1] - ro[r])
            ci[ro[r]:ro[r + 1]], va[ro[r]:ro[r + 1]] = ci[ro[r]:ro[r + 1]][order], va[ro[r]:ro[r + 1]][order]
    got, other = run(ro, ci, va, B)
    for rows in (slice(0, 70), slice(M // 2, M // 2 + 64), slice(M - 320, M)):
        dense = np.zeros((rows.stop - rows.start, K))
        for i, r in enumerate(range(rows.start, rows.stop)):
            dense[i, ci[ro[r]:ro[r + 1]]] = va[ro[r]:ro[r + 1]]
        want = dense @ B.astype(np.float64)
        here, there = (np.linalg.norm(x[rows] - want) / np.linalg.norm(want) for x in (got, other))
        assert here <= 1.02 * there and here <= 5e-8, (here, there)
        if what == "one sign":  # (rounded once at the end, to nearest: no mean error to speak of)
            assert abs(((got[rows] - want) / want).mean()) <= 5e-9
