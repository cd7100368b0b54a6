"""spmm, sddmm and fused as native functions against the Python implementations they hand unusual calls to: the same bits
for every way of passing the arguments, the same exceptions for what they refuse."""
import inspect

import numpy as np
import pytest

import dlspm_hip as dl

torch = pytest.importorskip("torch")

OPS = ("spmm", "sddmm", "fused")


@pytest.mark.parametrize("name", OPS)
def test_signature_is_the_python_one(name):
    python = inspect.signature(getattr(dl, "_" + name))
    assert str(inspect.signature(getattr(dl, name))) == str(python)


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
