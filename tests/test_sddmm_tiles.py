"""SDDMM on dense tiles (dlspm-esimd_amd/csrc/sddmm_tiles.hip) at the edges of tiles, steps and ranges, against 64 bits and
against the gathering kernels."""
import pytest

import dlspm_hip as dl

TILES = dl.RULES["dense_groups"]


@pytest.fixture(scope="module")
def torch_cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch


def mask(torch, M, K, density, seed, rows="even"):
    """CSR on the GPU, columns ascending; rows "some_empty": every third one is"""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    keep = torch.rand((M, K), device="cuda", generator=g) < density
    if rows == "some_empty":
        keep[::3] = False
    offsets = torch.zeros(M + 1, dtype=torch.int32, device="cuda")
    offsets[1:] = keep.sum(1).cumsum(0)
    row, col = keep.nonzero(as_tuple=True)
    return offsets, col.to(torch.int32), row


def operands(torch, M, K, D, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn((M, D), device="cuda", generator=g), torch.randn((K, D), device="cuda", generator=g)


def exact(torch, lhs, rhs, row, col):
    out = []
    for i in range(0, row.numel(), 1 << 20):
        r, c = row[i:i + (1 << 20)], col[i:i + (1 << 20)].long()
        out.append((lhs[r].double() * rhs[c].double()).sum(1))
    return torch.cat(out)


def both(torch, ro, ci, lhs, rhs):
    """the call's result and the gathering kernels', each into memory that shows what was not written"""
    on = torch.full((ci.numel(),), float("nan"), device="cuda")
    off = on.clone()
    assert "tile_columns" in dl.describe_schedule(dl.OP_SDDMM, lhs.shape[0], rhs.shape[0], lhs.shape[1], ci.numel())
    dl.sddmm(ro, ci, lhs, rhs, out=on)
    dl.set_tuning(rules_off=TILES)
    dl.sddmm(ro, ci, lhs, rhs, out=off)
    dl.set_tuning()
    return on, off


def error(got, want):
    return float((got.double() - want).norm() / want.norm())


def test_where_tiles_are_chosen():
    case = lambda M, K, D, density, **kw: dl.describe_schedule(dl.OP_SDDMM, M, K, D, int(M * K * density), **kw)  # noqa: E731
    assert case(24576, 8192, 32, 0.2) == {"schedule": "flat", "rows": 64, "slice_rows": 0, "chunks": 0, "tile_columns": 256}
    assert "tile_columns" in case(8192, 8192, 128, 0.3, workspace_bytes=dl.HINT_ROWS_EVEN)
    for M, K, D, density in ((2048, 2048, 128, 0.05), (24576, 8192, 32, 0.05), (8192, 8192, 129, 0.3), (8192, 8192, 16, 0.3), (512, 512, 64, 0.5)):
        assert "tile_columns" not in case(M, K, D, density)
    dl.set_tuning(rules_off=TILES)
    assert "tile_columns" not in case(24576, 8192, 32, 0.2)


@pytest.mark.parametrize("named,runs,size", [({"flat": 0}, "row_blocks", 0), ({"flat": 1}, "flat", 0), ({"slices": 4}, "sliced", 1 << 40), ({"split": (4, 2)}, "flat", 0),
                                             ({"split": (4, 2), "flat": 0}, "row_blocks", 0), ({"xcd_contiguous": 1}, "flat", 0), ({"flat_chunk": 512}, "flat", 0)])
def test_a_schedule_asked_for_by_name_runs(named, runs, size):
    """Tuning overrides that name a schedule of the gathering kernels get it, as for SpMM; the fused op's two steps need tiles."""
    M, K, D, nnz = 24576, 8192, 32, int(24576 * 8192 * 0.2)
    tiles = lambda: "tile_columns" in dl.describe_schedule(dl.OP_SDDMM, M, K, D, nnz, workspace_bytes=size)  # noqa: E731
    assert tiles()
    dl.set_tuning(**named)
    run, fused = dl.describe_schedule(dl.OP_SDDMM, M, K, D, nnz, workspace_bytes=size), dl.describe_schedule(dl.OP_FUSED, 16384, 8192, 128, 16384 * 2457, workspace_bytes=1 << 40)
    dl.set_tuning()
    assert run["schedule"] == runs and "tile_columns" not in run and fused["schedule"] != "two_steps"
    dl.set_tuning(stream_results=1)  # (not a schedule)
    assert tiles()
    dl.set_tuning()


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,D,density", [(4097, 4095, 17, 0.9), (4100, 4097, 32, 0.9), (4095, 3841, 31, 0.95), (24576, 2048, 32, 0.25), (1983, 4097, 33, 0.9),
                                           (1985, 4095, 63, 0.6), (2111, 2303, 64, 0.9), (2049, 2305, 65, 0.5), (1023, 2048, 96, 0.9), (1025, 2304, 97, 0.6),
                                           (1000, 2000, 127, 0.9), (1087, 2817, 128, 0.7), (40000, 300, 128, 0.5), (300, 30000, 100, 0.4), (33000, 1025, 50, 0.7)])
def test_tiles_against_64_bits(torch_cuda, M, K, D, density):
    torch = torch_cuda
    ro, ci, row = mask(torch, M, K, density, M + D, "some_empty" if M % 2 else "even")
    if M % 2:  # (dense enough all the same)
        assert ci.numel() > 0.3 * density * M * K
    lhs, rhs = operands(torch, M, K, D, K)
    if "tile_columns" not in dl.describe_schedule(dl.OP_SDDMM, M, K, D, ci.numel()):
        ro, ci, row = mask(torch, M, K, density, M + D)
    on, off = both(torch, ro, ci, lhs, rhs)
    want = exact(torch, lhs, rhs, row, ci)
    # every result is one dot product: no worse than 2^-22 of the sum of its terms' magnitudes, and together no worse than the
    # gathering kernels' results
    terms = exact(torch, lhs.abs(), rhs.abs(), row, ci)
    assert bool(((on.double() - want).abs() <= 2.0 ** -22 * terms).all())
    assert error(on, want) <= error(off, want)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,D", [(4096, 4096, 32), (1500, 2300, 64), (1000, 2300, 128)])
@pytest.mark.parametrize("kind", ["descending", "shuffled", "duplicates"])
def test_columns_that_do_not_ascend(torch_cuda, M, K, D, kind):
    torch = torch_cuda
    ro, ci, row = mask(torch, M, K, 0.9, 3)
    lhs, rhs = operands(torch, M, K, D, 4)
    at = torch.arange(ci.numel(), device="cuda")
    first, end = ro[:-1].long()[row], ro[1:].long()[row]
    some = row % 5 != 0  # (the others stay as they are)
    if kind == "descending":
        ci = torch.where(some, ci[first + end - 1 - at], ci)
    elif kind == "shuffled":
        key = row.double() + torch.rand(ci.numel(), device="cuda") * 0.5
        ci = torch.where(some, ci[key.argsort()], ci)
    else:
        ci = torch.where(some & (at % 7 == 3) & (at > first), ci[(at - 1).clamp(min=0)], ci)
    on, off = both(torch, ro, ci.contiguous(), lhs, rhs)
    want = exact(torch, lhs, rhs, row, ci)
    assert error(on, want) <= 1e-6 and error(off, want) <= 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("D", [32, 64, 128])
def test_values_that_the_parts_do_not_hold(torch_cuda, D):
    torch = torch_cuda
    M, K = 4096, 4096
    ro, ci, row = mask(torch, M, K, 0.6, 5)
    lhs, rhs = operands(torch, M, K, D, 6)
    lhs[7, 3], lhs[900, 1], lhs[3000, D - 1] = float("inf"), float("nan"), 3.4e38
    rhs[11, 5], rhs[2222, 0], rhs[4000, 2] = float("-inf"), float("nan"), -3.4e38
    lhs[40] *= 1e-36  # (below what three bf16 hold; the products are ordinary numbers)
    rhs[77] *= 1e-38
    rhs[500] *= 1e30
    lhs[60, 4] = 1e-40
    on, off = both(torch, ro, ci, lhs, rhs)
    assert bool((on.isnan() == off.isnan()).all()) and bool((on.isinf() == off.isinf()).all())
    assert bool((on[on.isinf()] == off[off.isinf()]).all())
    for rows in (row == 40, row == 60, ci == 77, ci == 500):
        few = rows & on.isfinite()
        want = exact(torch, lhs, rhs, row[few], ci[few])
        assert error(on[few], want) <= max(2.0 * error(off[few], want), 2.0 ** -22)
    ordinary = on.isfinite() & (ci != 77) & (ci != 500) & (row != 40)
    assert error(on[ordinary], exact(torch, lhs, rhs, row[ordinary], ci[ordinary])) <= 1e-6


@pytest.mark.gpu
def test_the_same_bits_whatever_comes_with_the_call(torch_cuda):
    torch = torch_cuda
    M, K, D = 6000, 3000, 64
    ro, ci, row = mask(torch, M, K, 0.4, 8)
    lhs, rhs = operands(torch, M, K, D, 9)
    first = dl.sddmm(ro, ci, lhs, rhs)
    ways = [dict(), dict(workspace=dl.ROWS_EVEN), dict(banded=True), dict(plan=dl.row_plan(ro)), dict(plan=dl.cut_plan(ro, dl.OP_SDDMM, D)),
            dict(plan=dl.prepare(ro, ci, K, dl.OP_SDDMM, D))]
    for way in ways:
        assert torch.equal(dl.sddmm(ro, ci, lhs, rhs, **way), first)
    graph, out = torch.cuda.CUDAGraph(), torch.empty_like(first)
    with torch.cuda.graph(graph):
        dl.sddmm(ro, ci, lhs, rhs, out=out)
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, first)
    # operands on any float
    shifted = torch.empty(lhs.numel() + 1, device="cuda")[1:].view(M, D).copy_(lhs), torch.empty(rhs.numel() + 3, device="cuda")[3:].view(K, D).copy_(rhs)
    assert torch.equal(dl.sddmm(ro, ci, *shifted), first)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,D,density", [(4096, 4096, 32, 0.9), (1500, 2300, 64, 0.9), (1000, 2000, 127, 0.9), (300, 30000, 100, 0.4), (40000, 300, 128, 0.5)])
@pytest.mark.parametrize("kind", ["a tenth of the rows", "every row", "behind the first 64", "one row in four, descending"])
def test_how_many_rows_ascend(torch_cuda, M, K, D, density, kind):
    """Few rows that do not ascend are shared by the waves behind the tiles, more than half of a tile's are gathered in its place, and
    rows found out on the way are finished by their wave: every nonzero once, with several ranges of columns too."""
    torch = torch_cuda
    ro, ci, row = mask(torch, M, K, density, 13)
    lhs, rhs = operands(torch, M, K, D, 14)
    at = torch.arange(ci.numel(), device="cuda")
    first, end = ro[:-1].long()[row], ro[1:].long()[row]
    if kind == "one row in four, descending":
        ci = torch.where(row % 4 == 1, ci[first + end - 1 - at], ci)
    else:
        some = row % 10 == 3 if kind == "a tenth of the rows" else at - first >= 64 if kind == "behind the first 64" else row >= 0
        key = torch.where(some, torch.rand(ci.numel(), device="cuda", dtype=torch.float64) * 0.4 + 0.1, (at - first).double() * 1e-9)
        ci = ci[(row.double() + key).argsort()]
    on, off = both(torch, ro, ci.contiguous(), lhs, rhs)
    want = exact(torch, lhs, rhs, row, ci)
    terms = exact(torch, lhs.abs(), rhs.abs(), row, ci)
    assert bool(((on.double() - want).abs() <= 2.0 ** -22 * terms).all())
    # (a row's last nonzeros and its neighbour's first ones are written by different waves: none into the other's)
    assert bool(((on - off).abs() <= 2.0 ** -21 * terms).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,D,density", [(4096, 4096, 32, 0.9), (16448, 9000, 32, 0.3), (1500, 2300, 64, 0.9), (1000, 2000, 127, 0.9), (300, 30000, 100, 0.4)])
@pytest.mark.parametrize("small", [1e-33, 1e-36, 1e-44])
@pytest.mark.parametrize("where", ["rhs", "lhs", "both", "rhs, results of few terms"])
def test_values_too_small_for_their_parts(torch_cuda, M, K, D, density, small, where):
    """Values below 2^-109: rows of lhs with one are gathered, results of a row of rhs with one unless they are large against what its
    parts may have lost. Every result by itself, the smallest ones too."""
    torch = torch_cuda
    ro, ci, row = mask(torch, M, K, density, 23)
    lhs, rhs = operands(torch, M, K, D, 24)
    g = torch.Generator(device="cuda")
    g.manual_seed(25)
    few = lambda n: torch.rand((n, D), device="cuda", generator=g) < 0.004  # noqa: E731
    if where != "rhs" and not where.endswith("terms"):
        lhs[few(M)] = small
    if where != "lhs":
        rhs[few(K)] = small
    if where.endswith("terms"):  # columns whose results are made by such a value alone, in one row of lhs out of three by nothing
        rhs[5::19] = 0.0
        rhs[5::19, 3] = small
        lhs[::3, 3] = 0.0
    on, off = both(torch, ro, ci, lhs, rhs)
    want, terms = exact(torch, lhs, rhs, row, ci), exact(torch, lhs.abs(), rhs.abs(), row, ci)
    # (the gathering kernels round to multiples of 2^-149 as often as there are products)
    assert bool(((on.double() - want).abs() <= 2.0 ** -22 * terms + D * 2.0 ** -149).all())
    alone = (terms > 0) & (terms < 1e-30)
    assert bool(alone.any()) == where.endswith("terms")
    assert bool(((on.double() - want).abs()[alone] <= 2.0 ** -23 * terms[alone] + 2.0 ** -149).all())
    assert error(on, want) <= 1.02 * error(off, want)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,D,density", [(4096, 4096, 32, 0.9), (1500, 2300, 64, 0.9)])
def test_results_that_are_not_finite_run_by_run(torch_cuda, M, K, D, density):
    """What is gathered again is the run of 64s between the first and the last result that asks for it, of 256: at the ends of rows, of
    ranges and of such runs."""
    torch = torch_cuda
    ro, ci, row = mask(torch, M, K, density, 33)
    lhs, rhs = operands(torch, M, K, D, 34)
    columns = torch.tensor([0, 63, 64, 255, 256, 700, K - 1], device="cuda")
    rhs[columns] = torch.tensor([1.0, float("inf"), float("nan"), 3.4e38, 1.0, float("-inf"), float("nan")], device="cuda")[:, None]
    rhs[columns, 1:] = rhs[columns, 1:] * torch.sign(operands(torch, 7, 7, D - 1, 35)[0])
    lhs[::7] = float("nan")
    on, off = both(torch, ro, ci, lhs, rhs)
    assert bool((on.isnan() == off.isnan()).all())
    assert bool((on[on.isinf()] == off[on.isinf()]).all()) and bool((on.isinf() == off.isinf()).all())
    fine = on.isfinite()
    assert float((on - off)[fine].norm() / off[fine].norm()) <= 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,D,density", [(4100, 4097, 32, 0.9), (4097, 4095, 17, 0.9), (2111, 2303, 64, 0.9), (1985, 4095, 63, 0.6), (1023, 2048, 96, 0.9), (1087, 2817, 128, 0.7),
                                           (1000, 2000, 127, 0.9)])
def test_hinted_stores_change_no_bit(torch_cuda, M, K, D, density):
    """Results that go past the caches and those that do not, of kernels of their own for both, at every number of segments and for
    whole and ragged widths; columns that do not ascend and a NaN among them (whose results are stored by the row)."""
    torch = torch_cuda
    ro, ci, row = mask(torch, M, K, density, 43)
    lhs, rhs = operands(torch, M, K, D, 44)
    rhs[K // 2] = float("nan")
    at = torch.arange(ci.numel(), device="cuda")
    first, end = ro[:-1].long()[row], ro[1:].long()[row]
    ci = torch.where(row % 11 == 2, ci[first + end - 1 - at], ci)
    got = []
    for stream in (0, 1):
        dl.set_tuning(stream_results=stream)
        assert "tile_columns" in dl.describe_schedule(dl.OP_SDDMM, M, K, D, ci.numel())
        out = torch.full((ci.numel() + 64,), 7.0, device="cuda")
        dl.sddmm(ro, ci, lhs, rhs, out=out[:ci.numel()])
        assert bool((out[ci.numel():] == 7.0).all())
        got.append(out[:ci.numel()].view(torch.int32))
    dl.set_tuning()
    assert torch.equal(*got) and bool((got[0].view(torch.float32).isnan() == (ci == K // 2)).all())


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["both signs", "one sign", "unordered"])
@pytest.mark.parametrize("M,K,D,density", [(16384, 64, 128, 0.9), (16384, 200, 64, 0.9), (4100, 4097, 32, 0.9), (2111, 2303, 64, 0.9), (1087, 2817, 128, 0.7),
                                           (1983, 4097, 33, 0.9), (2049, 2305, 65, 0.5), (1025, 2304, 97, 0.6), (1000, 2000, 127, 0.9)])
def test_a_single_tile_and_operands_of_one_sign(torch_cuda, M, K, D, density, what):
    """Masks narrower than a tile, where waves lie beyond the last column; operands of one sign, where a bias in the rounding of the
    matrix cores' sums would add up."""
    torch = torch_cuda
    ro, ci, row = mask(torch, M, K, density, 53)
    lhs, rhs = operands(torch, M, K, D, 54)
    if what == "one sign":
        lhs, rhs = lhs.abs(), rhs.abs()
    elif what == "unordered":
        at = torch.arange(ci.numel(), device="cuda")
        ci = torch.where(row % 3 == 0, ci[ro[:-1].long()[row] + ro[1:].long()[row] - 1 - at], ci).contiguous()
    on, off = both(torch, ro, ci, lhs, rhs)
    want, terms = exact(torch, lhs, rhs, row, ci), exact(torch, lhs.abs(), rhs.abs(), row, ci)
    assert bool(((on.double() - want).abs() <= 2.0 ** -22 * terms).all())
    assert error(on, want) <= error(off, want)
    if what == "one sign":
        # (were the sums not rounded to nearest, the mean would not be far below the errors)
        assert 10 * abs(float(((on.double() - want) / want).mean())) <= error(off, want)
