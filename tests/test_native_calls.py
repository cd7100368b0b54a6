"""spmm, sddmm and fused as native functions against the Python implementations they hand unusual calls to: the same bits
for every way of passing the arguments, the same exceptions for what they refuse."""
import importlib.util
import inspect
import os
import subprocess
import sys
import warnings

import numpy as np
import pytest

import dlspm_hip as dl

torch = pytest.importorskip("torch")

OPS = ("spmm", "sddmm", "fused")


@pytest.mark.parametrize("name", OPS)
def test_signature_is_the_python_one(name):
    python = inspect.signature(getattr(dl, "_" + name))
    assert str(inspect.signature(getattr(dl, name))) == str(python)


def fresh_module():
    """dlspm_hip.py imported once more, before any of its native functions was used"""
    spec = importlib.util.spec_from_file_location("dlspm_hip_again", dl.__file__)
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def test_names_of_the_module():
    here = os.path.dirname(dl.__file__)
    for code in ("from dlspm_hip import *; spmm, sddmm, fused, prepare, OP_SPMM", "import dlspm_hip as d; assert {'spmm', 'sddmm', 'fused', 'prepare'} <= set(dir(d))",
                 "import dlspm_hip as d, sys; assert 'torch' not in sys.modules; dir(d); assert 'torch' not in sys.modules"):
        subprocess.run([sys.executable, "-c", code], check=True, cwd=here)
    assert set(dl.__all__) >= {*OPS, "prepare", "analyze", "DlspmError"} and not any(n.startswith("_") for n in dl.__all__)
    with pytest.raises(AttributeError):
        dl.nonsense  # noqa: B018


@pytest.mark.parametrize("what", ["missing", "broken"])
def test_without_the_native_module(tmp_path, what):
    """the ctypes implementations stand in, with a warning where a module is there that cannot be loaded"""
    m = fresh_module()
    m.CALLS_PATH = str(tmp_path / "_dlspm_torch.so")
    if what == "broken":
        open(m.CALLS_PATH, "w").write("no module")
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        assert m.spmm is m._spmm and m.sddmm is m._sddmm and m.fused is m._fused
    assert [w.category for w in seen] == ([RuntimeWarning] if what == "broken" else [])


def test_make_without_pytorch():
    here = os.path.dirname(dl.__file__)
    plan = lambda python: subprocess.run(["make", "-n", "-B", "all", f"PYTHON={python}"], check=True, cwd=here, capture_output=True, text=True).stdout  # noqa: E731
    assert "_dlspm_torch.so" in plan(sys.executable) and "libdlspm_hip.so" in plan(sys.executable)
    assert "_dlspm_torch.so" not in plan("/bin/false") and "libdlspm_hip.so" in plan("/bin/false")


def operands(name, M=37, K=29, N=12, device="cpu", kind=dl.PATTERN_BERNOULLI):
    ro, ci = dl.make_pattern(kind, 5, M, K, 0.3)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    dense = {"spmm": [(ci.size,), (K, N)], "sddmm": [(M, N), (K, N)], "fused": [(M, N), (K, N), (K, N)]}[name]
    return [t(ro), t(ci)] + [t(dl.fill("normal", 7 + i, s)) for i, s in enumerate(dense)]


@pytest.mark.parametrize("name", OPS)
@pytest.mark.parametrize("wrong", ["host", "missing", "unknown", "twice", "none"])
def test_refusals_are_the_python_ones(name, wrong):
    args, kwargs = operands(name), {}
    if wrong == "missing":
        args = args[:-1]
    elif wrong == "unknown":
        kwargs = {"nonsense": 1}
    elif wrong == "twice":
        kwargs = {"row_offsets": args[0]}
    elif wrong == "none":
        args[1] = None
    seen = []
    for call in (getattr(dl, name), getattr(dl, "_" + name)):
        with pytest.raises(Exception) as e:
            call(*args, **kwargs)
        seen.append((type(e.value), str(e.value)))
    assert seen[0] == seen[1]


@pytest.mark.gpu
@pytest.mark.parametrize("name", OPS)
@pytest.mark.parametrize("shape", [(37, 29, 12), (1, 1, 1), (300, 700, 65)])
def test_same_bits_as_the_python_calls(name, shape):
    args = operands(name, *shape, device="cuda")
    native, python = getattr(dl, name), getattr(dl, "_" + name)
    M, nnz = args[0].numel() - 1, args[1].numel()
    size = (nnz,) if name == "sddmm" else (M, shape[2])
    prepared = dl.prepare(args[0], args[1], shape[1], {"spmm": 0, "sddmm": 1, "fused": 2}[name], shape[2])
    names = list(inspect.signature(python).parameters)
    ways = [{}, {"plan": prepared}, {"out": torch.full(size, 7.0, device="cuda")}, {"plan": None, "workspace": None, "banded": False},
            {"workspace": dl.ROWS_EVEN}, {"banded": True}]
    ways += [{"K": shape[1]}, {"K": shape[1], "plan": prepared}] if name == "spmm" else []
    ways += [{"scale": 0.5}, {"scale": 2}] if name == "fused" else []
    for way in ways:
        want = python(*args, **dict(way, out=None))
        got = native(*args, **way)
        assert got.shape == size and torch.equal(got, want), way
        assert way.get("out") is None or got is way["out"]
        by_name = native(**dict(zip(names, args)), **dict(way, out=None))
        assert torch.equal(by_name, want), way


@pytest.mark.gpu
@pytest.mark.parametrize("name", OPS)
def test_wrong_operands_on_the_device(name):
    good = operands(name, device="cuda")
    native, python = getattr(dl, name), getattr(dl, "_" + name)
    bad = [good[:2] + [good[2].double()] + good[3:], good[:3] + [good[3].t()] + good[4:], good[:3] + [good[3][:, 0]] + good[4:],
           [good[0].long()] + good[1:], [good[0][:0]] + good[1:]]
    for args in bad:
        seen = []
        for call in (native, python):
            with pytest.raises(Exception) as e:
                call(*args)
            seen.append((type(e.value), str(e.value)))
        assert seen[0] == seen[1]
    with pytest.raises(ValueError):
        native(*good, out=torch.empty(1, device="cuda"))


@pytest.mark.gpu
@pytest.mark.parametrize("name", OPS)
def test_a_result_that_does_not_fit_is_out_of_memory(name):
    """the exception of torch.empty (a caller that frees its caches and tries again relies on it), and the call works afterwards"""
    z = lambda *shape: torch.zeros(shape, device="cuda")  # noqa: E731
    M, N = 4096, 1 << 16  # results of 1 GiB
    if name == "sddmm":  # every column of every row
        args = [torch.arange(M + 1, dtype=torch.int32, device="cuda") * N, torch.zeros(M * N, dtype=torch.int32, device="cuda"), z(M, 4), z(N, 4)]
    else:
        empty = [torch.zeros(M + 1, dtype=torch.int32, device="cuda"), torch.zeros(0, dtype=torch.int32, device="cuda")]
        args = empty + ([z(0), z(1, N)] if name == "spmm" else [z(M, N), z(1, N), z(1, N)])
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)
        for call in (getattr(dl, "_" + name), getattr(dl, name)):
            with pytest.raises(torch.OutOfMemoryError):
                call(*args)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert not getattr(dl, name)(*args).any()


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["spmm", "fused"])
def test_without_room_for_the_memory_of_a_call_it_runs_on_the_hints_alone(name):
    """The memory that prepare() leaves to each call is for speed: a call whose own result has room runs without it, by both kinds of
    call, with the bits of the call that passes the hints alone."""
    import torch

    M, K, N = (4096, 8192, 512) if name == "spmm" else (12288, 2048, 128)
    keep = torch.rand((M, K), device="cuda") < 0.4
    ro = torch.zeros(M + 1, dtype=torch.int32, device="cuda")
    ro[1:] = keep.sum(1).cumsum(0)
    ci = keep.nonzero()[:, 1].to(torch.int32)
    del keep
    r = lambda *s: torch.randn(s, device="cuda")  # noqa: E731
    args = (ro, ci, r(ci.numel()), r(K, N)) if name == "spmm" else (ro, ci, r(M, N), r(K, N), r(K, N), 0.5)
    plan = dl.prepare(ro, ci, K, dl.OP_SPMM if name == "spmm" else dl.OP_FUSED, N)
    size = plan.size_and_hints & ~dl.HINT_MASK
    assert plan.memory is None and size > 24 << 20 and plan.size_and_hints & dl.HINT_MASK == dl.HINT_ROWS_EVEN
    calls = (getattr(dl, "_" + name), getattr(dl, name))
    with_memory, hints_alone = calls[1](*args, plan=plan), calls[1](*args, workspace=dl.ROWS_EVEN)
    assert not torch.equal(with_memory, hints_alone)
    out = torch.empty_like(hints_alone)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (2 << 20)) / total)
        taken = []
        with pytest.raises(torch.OutOfMemoryError):
            while True:  # (what is free among the blocks in use)
                taken.append(torch.empty((size,), dtype=torch.uint8, device="cuda"))
        for call in calls:
            out.zero_()
            call(*args, out=out, plan=plan)
            assert torch.equal(out, hints_alone), call
        del taken
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    for call in calls:
        assert torch.equal(call(*args, plan=plan), with_memory)
