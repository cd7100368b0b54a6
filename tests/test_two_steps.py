"""The fused op on dense masks as SDDMM on dense tiles and then SpMM, the scores in the caller's memory in between."""
import numpy as np
import pytest

import dlspm_hip as dl

EVEN = dl.HINT_ROWS_EVEN


def schedule(M, K, D, nnz, size):
    return dl.describe_schedule(dl.OP_FUSED, M, K, D, nnz, workspace_bytes=size)


def test_who_runs_in_two_steps():
    M = K = 8192
    D, nnz = 128, 8192 * 2457
    scores = nnz * 4
    cp = dl.advise(dl.OP_FUSED, D, dl.MatrixInfo(M, K, nnz, 2700, 0, K, 8000, 1000))
    assert (cp.build, cp.bytes, cp.hints) == (dl.BUILD_NOTHING, scores, EVEN)
    run = schedule(M, K, D, nnz, scores | EVEN)
    assert run == {"schedule": "two_steps", "rows": 64, "slice_rows": 0, "chunks": 0, "tile_columns": 256, "second": "resident"}
    assert schedule(M, K, D, nnz, scores)["schedule"] == "two_steps"
    # the second step on dense tiles, with memory for V's parts behind the scores
    cp = dl.advise(dl.OP_FUSED, D, dl.MatrixInfo(2 * M, K, 2 * nnz, 2700, 0, K, 8000, 1000))
    assert cp.bytes == 2 * scores + K * D * 6 + K // 16 * D // 32 * 8
    assert [schedule(2 * M, K, D, 2 * nnz, n | EVEN)["second"] for n in (cp.bytes, cp.bytes - 1, 2 * scores)] == ["dense_tiles", "resident", "resident"]
    # less memory, none, a band, wide or sparse masks: as before; too little memory for the slices is refused as before
    other = schedule(M, K, D, nnz, EVEN)
    assert schedule(M, K, D, nnz, (scores - 4) | EVEN) == other and other["schedule"] != "two_steps"
    for size in (0, scores | EVEN | dl.HINT_BANDED, dl.row_plan_bytes(M) | dl.HINT_ROW_PLAN):
        assert schedule(M, K, D, nnz, size)["schedule"] != "two_steps"
    assert schedule(M, K, 132, nnz, 1 << 40)["schedule"] != "two_steps" and schedule(M, K, D, M * 300, 1 << 40)["schedule"] != "two_steps"
    need = dl.workspace_bytes(dl.OP_FUSED, M, K, D, nnz)
    assert schedule(M, K, D, nnz, need)["schedule"] == "sliced"
    with pytest.raises(dl.DlspmError):
        schedule(M, K, D, nnz, need - 256)
    for rule in ("dense_groups", "resident_slices"):
        dl.set_tuning(rules_off=dl.RULES[rule])
        assert schedule(M, K, D, nnz, 1 << 40)["schedule"] != "two_steps"
    dl.set_tuning()


def operands(M, K, D, density, seed):
    rng = np.random.default_rng(seed)
    keep = rng.random((M, K)) < density
    ro = np.concatenate(([0], np.cumsum(keep.sum(1)))).astype(np.int32)
    return (ro, np.nonzero(keep)[1].astype(np.int32), *(rng.normal(size=(n, D)).astype(np.float32) for n in (M, K, K))), rng


def run(args, scale, second, even=True):
    """in two steps, and by the fused kernels"""
    import torch

    ro, ci, Q, Km, V = args
    M, (K, D) = ro.size - 1, Km.shape
    parts = -(-D // 32) * -(-K // 128) * 8 * (3072 + 8) if second == "dense_tiles" else 0
    need = -(-ci.size * 4 // 256) * 256 + parts
    hint = EVEN if even else 0
    if not even:
        need = max(need, dl.workspace_bytes(dl.OP_FUSED, M, K, D, ci.size))
    assert schedule(M, K, D, ci.size, need | hint).get("second") == second
    memory = torch.full((need + 256,), 77, dtype=torch.uint8, device="cuda")
    on_gpu = [torch.from_numpy(a).cuda() for a in args]
    got = dl.fused(*on_gpu, scale, plan=dl.Prepared(memory, need | hint, None))
    assert bool((memory[need:] == 77).all())
    return got.cpu().numpy(), dl.fused(*on_gpu, scale, workspace=dl.ROWS_EVEN).cpu().numpy()


def exact(args, scale, rows):
    ro, ci, Q, Km, V = args
    scores = np.zeros((len(rows), Km.shape[0]))
    for i, r in enumerate(rows):
        c = ci[ro[r]:ro[r + 1]]
        np.add.at(scores[i], c, scale * (Km[c].astype(np.float64) @ Q[r].astype(np.float64)))
    return scores @ V.astype(np.float64)


CASES = [(6145, 1027, 100, 0.35, "resident", True), (12290, 2045, 128, 0.25, "resident", False), (12290, 2045, 128, 0.25, "dense_tiles", True),
         (8200, 1500, 65, 0.5, "dense_tiles", True), (3001, 1030, 128, 0.6, "row_blocks", True)]


# Error against 64 bits: of the scores (six products of parts for one, sums of 16 ... 128) and of the sums over a row, each no larger than
# in the fused kernels (chains of D / 8 and of a quarter of a row in 32 bits; a second step of row blocks has the latter too, the others
# add up in 64 bits, so that what is left of 1e-7 or so is the scores' and one rounding at the end)
@pytest.mark.gpu
@pytest.mark.parametrize("M,K,D,density,second,even", CASES)
def test_no_less_precise_than_the_fused_kernels(M, K, D, density, second, even):
    args, rng = operands(M, K, D, density, M + D)
    got, other = run(args, 0.125, second, even)
    assert not np.array_equal(got, other)
    rows = np.concatenate((np.arange(70), np.arange(M // 2, M // 2 + 60), np.arange(M - 70, M)))
    want = exact(args, 0.125, rows)
    here, there = (np.linalg.norm(x[rows] - want) / np.linalg.norm(want) for x in (got, other))
    assert here <= 1.02 * there and (second == "row_blocks" or here <= 1.6e-7), (here, there)
    assert np.linalg.norm(got - other) <= 5e-7 * np.linalg.norm(other)


@pytest.mark.gpu
@pytest.mark.parametrize("second,case", [("resident", 0), ("dense_tiles", 3)])
@pytest.mark.parametrize("what", ["unordered", "twice", "empty", "unused inf", "inf", "nan", "scale 0", "scale inf", "scale nan", "scale tiny"])
def test_special_values_and_structures(what, second, case):
    M, K, D, density = CASES[case][:4]
    (ro, ci, Q, Km, V), rng = operands(M, K, D, density, 11)
    rows, scale = np.arange(5, M, 97), 0.25
    for r in rows:
        a, b = ro[r], ro[r + 1]
        if what == "unordered":
            rng.shuffle(ci[a:b])
        elif what == "twice":
            ci[a + 3] = ci[a + 4]
    if what == "empty":
        keep = np.ones(ci.size, bool)
        counts = np.diff(ro)
        for r in rows:
            keep[ro[r]:ro[r + 1]] = False
        counts[rows] = 0
        ro, ci = np.concatenate(([0], np.cumsum(counts))).astype(np.int32), ci[keep]
    elif what == "unused inf":
        ci = np.where(ci == 17, 18, ci).astype(np.int32)
        Km[17], V[17] = np.inf, np.nan
    elif what == "inf":
        Q[7, 3], V[9, 1] = np.inf, -np.inf
    elif what == "nan":
        Q[7, 3], Km[40, 2] = np.nan, np.nan
    elif what.startswith("scale"):
        scale = {"0": 0.0, "inf": np.inf, "nan": np.nan, "tiny": 1e-38}[what.split()[1]]
    args = (ro, ci, Q, Km, V)
    got, other = run(args, scale, second)
    fine = np.isfinite(other)
    assert np.array_equal(fine, np.isfinite(got)) and np.array_equal(np.isnan(other), np.isnan(got))
    got, other = np.where(fine, got, 0.0).astype(np.float64), np.where(fine, other, 0.0).astype(np.float64)
    if what == "scale tiny":
        # scores are rounded to multiples of 2^-149 once on both paths: K of them, half a unit each, times V
        assert np.linalg.norm(other) > 0 and np.abs(got - other).max() <= K * 2.0 ** -149 * np.abs(V).max() + 1e-6 * np.abs(other).max()
    else:
        assert np.linalg.norm(got - other) <= 5e-7 * np.linalg.norm(other)
    if what == "empty":
        assert not got[rows].any()


@pytest.mark.gpu
def test_one_plan_on_two_streams_and_in_a_graph():
    """Each call has memory of its own: calls that overlap in time do not meet in it."""
    import torch

    M, K, D, density, second, _ = CASES[3]
    (ro, ci, Q, Km, V), rng = operands(M, K, D, density, 2)
    args = [torch.from_numpy(a).cuda() for a in (ro, ci)]
    sets = [[torch.from_numpy(rng.normal(size=a.shape).astype(np.float32)).cuda() for a in (Q, Km, V)] for _ in range(2)]
    plan = dl.prepare(*args, K, dl.OP_FUSED, D)
    assert plan.memory is None and dl.describe_schedule(dl.OP_FUSED, M, K, D, ci.size, plan=plan)["second"] == second
    want = [dl.fused(*args, *s, 0.5, plan=plan) for s in sets]
    assert torch.equal(dl._fused(*args, *sets[0], 0.5, plan=plan), want[0])  # (the calls through ctypes)
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(8):
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                got[i].append(dl.fused(*args, *sets[i], 0.5, plan=plan))
    torch.cuda.synchronize()
    assert all(torch.equal(x, want[i]) for i in range(2) for x in got[i])
    inputs, out, graph = [t.clone() for t in sets[0]], torch.empty_like(want[0]), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        dl.fused(*args, *inputs, 0.5, out=out, plan=plan)
    for i in (0, 1, 0, 1):
        for t, s in zip(inputs, sets[i]):
            t.copy_(s)
        graph.replay()
        other = dl.fused(*args, *sets[1 - i], 0.5, plan=plan)
        torch.cuda.synchronize()
        assert torch.equal(out, want[i]) and torch.equal(other, want[1 - i])


def test_the_rule_holds_beside_powers_of_two():
    """At density 0.1, D = 128 up to 8192 rows (as many row blocks, in two ranges of columns, as there are compute units), and not where
    the next row block begins a second round."""
    def runs(M, K, D, density, even=True):
        info = dl.MatrixInfo(M, K, int(M * K * density), int(K * density * 1.2) if even else K, 0, K, 8000, 1000)
        cp = dl.advise(dl.OP_FUSED, D, info)
        return dl.describe_schedule(dl.OP_FUSED, M, K, D, info.nnz, workspace_bytes=cp.bytes | cp.hints)["schedule"] == "two_steps"

    rng = np.random.default_rng(3)
    assert all(runs(8192 - int(a), 8192 - int(b), 128, d) for a, b, d in zip(rng.integers(0, 64, 200), rng.integers(0, 64, 200), rng.uniform(0.0985, 0.1015, 200)))
    assert not runs(8321, 8180, 128, 0.113) and not runs(8578, 8015, 120, 0.098)
    # one size each of a second step from slices of B, on tiles and of row blocks, and those that measured slower
    assert runs(17343, 3729, 128, 0.132) and runs(16075, 7628, 128, 0.305) and runs(4822, 6818, 96, 0.241) and runs(4676, 7785, 128, 0.212)
    assert not runs(2096, 7374, 128, 0.44) and not runs(7808, 7995, 96, 0.087) and not runs(23879, 3669, 64, 0.113) and not runs(17071, 7498, 32, 0.251)
    assert not runs(12772, 3715, 96, 0.135, even=False) and runs(28641, 1244, 64, 0.254, even=False)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,D,density,second,even", CASES)
def test_operands_of_one_sign(M, K, D, density, second, even):
    (ro, ci, Q, Km, V), rng = operands(M, K, D, density, M - D)
    args = ro, ci, np.abs(Q), np.abs(Km), np.abs(V)
    got, other = run(args, 0.125, second, even)
    rows = np.concatenate((np.arange(70), np.arange(M - 70, M)))
    want = exact(args, 0.125, rows)
    here, there = (np.linalg.norm(x[rows] - want) / np.linalg.norm(want) for x in (got, other))
    assert here <= 1.02 * there, (here, there)
