"""dlspm_describe_schedule: the schedule of a call, by the function that the call itself decides by."""
import json
import os
import sys
import types

import numpy as np
import pytest

import dlspm_hip as dl

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def schedule(op, M, K, N, nnz, workspace_bytes=0):
    return dl.describe_schedule(op, M, K, N, nnz, workspace_bytes=workspace_bytes)["schedule"]


def test_schedules():
    even, dense = dl.HINT_ROWS_EVEN, 8192 * 819
    assert dl.describe_schedule(dl.OP_SPMM, 8192, 8192, 128, dense, workspace_bytes=even) == {"schedule": "resident", "rows": 64, "slice_rows": 304, "chunks": 1}
    assert schedule(dl.OP_SPMM, 8192, 8192, 128, dense, even | dl.HINT_BANDED) == "resident"
    big = dl.describe_schedule(dl.OP_SPMM, 32768, 8192, 128, 32768 * 2457)
    assert big["schedule"] == "resident" and big["rows"] == 128 and big["chunks"] == 2
    assert schedule(dl.OP_SPMM, 8192, 8192, 128, dense) == "row_blocks"
    assert schedule(dl.OP_SPMM, 2048, 512, 256, 2048 * 50, dl.row_plan_bytes(2048) | dl.HINT_ROW_PLAN) == "row_plan"
    need = dl.row_plan_bytes_for(dl.OP_SPMM, 2048, 256)
    assert schedule(dl.OP_SPMM, 2048, 512, 256, 2048 * 50, need | dl.HINT_CUT_PLAN) == "cut_plan"
    assert schedule(dl.OP_SPMM, 8192, 32768, 256, 8192 * 300, dl.workspace_bytes(dl.OP_SPMM, 8192, 32768, 256, 8192 * 300)) == "sliced"
    assert schedule(dl.OP_SDDMM, 24576, 8192, 32, 24576 * 1638) == "flat"
    assert schedule(dl.OP_SDDMM, 24576, 8192, 32, 24576 * 1638, even) == "row_blocks"
    window = (dl.OP_FUSED, 16384, 16384, 128, 16384 * 128)
    assert schedule(*window) == schedule(*window, even) == "dense_groups"
    assert schedule(dl.OP_FUSED, 4096, 4096, 64, 4096 * 80) == "row_blocks"      # below the size that pays for the look
    assert schedule(dl.OP_FUSED, 16384, 16384, 256, 16384 * 128) == "row_blocks"  # wider than the groups are built for
    dl.set_tuning(rules_off=dl.RULES["resident_slices"] | dl.RULES["dense_groups"])
    assert schedule(dl.OP_SPMM, 8192, 8192, 128, dense, even) == schedule(*window) == "row_blocks"
    dl.set_tuning()
    for bad in (dict(workspace_bytes=1 << 57), dict(workspace_bytes=(need - 4) | dl.HINT_CUT_PLAN)):
        with pytest.raises(dl.DlspmError):
            dl.describe_schedule(dl.OP_SPMM, 2048, 512, 256, 2048 * 50, **bad)
    assert schedule(dl.OP_SPMM, 0, 5, 5, 0) == "row_blocks"


def test_a_recorded_traffic_figure_names_the_kernel_that_runs():
    """bench.py reports a figure of profiles/pmc_traffic.json for the launch it was recorded for only"""
    sys.path.insert(0, ROOT)
    import bench

    prep = types.SimpleNamespace(size_and_hints=dl.HINT_ROWS_EVEN, call_plan=types.SimpleNamespace(hints=dl.HINT_ROWS_EVEN, build=0))
    cfg4 = {"op": dl.OP_SPMM, "M": 2048, "K": 512, "N": 392, "nnz": 2048 * 102}
    signature = bench.launch_signature(dl, cfg4, prep)
    assert signature == "spmm:resident:rows64:slice-rows256:chunks1:DLSPM_HINT_ROWS_EVEN"
    assert bench.workgroups_of(dl, cfg4, prep) == 32 * 7
    dl.set_tuning(rules_off=dl.RULES["resident_slices"])
    assert bench.launch_signature(dl, cfg4, prep) == "spmm:vec4:row-lanes64x2:dot-lanes0x0:W4:R4:DLSPM_HINT_ROWS_EVEN"
    dl.set_tuning()
    record = json.load(open(os.path.join(ROOT, "profiles", "pmc_traffic.json")))["cfg4_spmm_2048x512x392_s80_topk_relu"]
    assert (record["launch"] == signature) == ("spmm_resident_kernel" in record["kernel"])


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,density", [(8192, 8192, 128, 0.1), (4096, 1024, 256, 0.4), (2048, 512, 256, 0.1), (4099, 700, 320, 0.2), (256, 2304, 784, 0.5)])
@pytest.mark.parametrize("way", ["null", "even", "banded", "row_plan", "cut_plan", "memory"])
def test_what_is_described_is_what_runs(M, K, N, density, way):
    torch = pytest.importorskip("torch")
    ro, ci = dl.make_pattern(dl.PATTERN_BERNOULLI, 5, M, K, density)
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    args = (d(ro), d(ci), torch.randn(ci.size, device="cuda"), torch.randn(K, N, device="cuda"))
    need = {"row_plan": dl.row_plan_bytes(M), "cut_plan": dl.row_plan_bytes_for(dl.OP_SPMM, M, N), "memory": dl.workspace_bytes(dl.OP_SPMM, M, K, N, ci.size)}
    size, kwargs = {"null": (0, {}), "even": (dl.HINT_ROWS_EVEN, {"workspace": dl.ROWS_EVEN}), "banded": (dl.HINT_BANDED, {"banded": True}),
                    "row_plan": (need["row_plan"] | dl.HINT_ROW_PLAN, {}), "cut_plan": (need["cut_plan"] | dl.HINT_CUT_PLAN, {}),
                    "memory": (need["memory"], {})}[way]
    if way == "row_plan":
        kwargs = {"plan": dl.row_plan(args[0])}
    elif way == "cut_plan":
        kwargs = {"plan": dl.cut_plan(args[0], dl.OP_SPMM, N)}
    elif way == "memory":
        if need["memory"] == 0:
            pytest.skip("no schedule memory at these sizes")
        kwargs = {"workspace": torch.empty(need["memory"], dtype=torch.uint8, device="cuda")}
    named = schedule(dl.OP_SPMM, M, K, N, int(ci.size), size)
    here = dl.spmm(*args, **kwargs)
    dl.set_tuning(rules_off=dl.RULES["resident_slices"])
    there = dl.spmm(*args, **kwargs)
    assert (named == "resident") == (not torch.equal(here, there))


def test_what_runs_on_the_matrix_cores_has_a_switch_each():
    M, K, nnz, size = 16384, 8192, 16384 * 2457, 1 << 40
    memory = size | dl.HINT_ROWS_EVEN

    def run(off):
        dl.set_tuning(rules_off=sum(dl.RULES[name] for name in off))
        sddmm = dl.describe_schedule(dl.OP_SDDMM, M, K, 128, nnz)
        spmm = dl.describe_schedule(dl.OP_SPMM, M, K, 128, nnz, workspace_bytes=memory)
        fused = dl.describe_schedule(dl.OP_FUSED, M, K, 128, nnz, workspace_bytes=memory)
        groups = dl.describe_schedule(dl.OP_FUSED, M, M, 128, M * 128)
        dl.set_tuning()
        return "tile_columns" in sddmm, spmm["schedule"], fused.get("second"), groups["schedule"]

    assert run([]) == (True, "dense_tiles", "dense_tiles", "dense_groups")
    assert run(["sddmm_tiles"]) == (False, "dense_tiles", "dense_tiles", "dense_groups")
    assert run(["spmm_tiles"]) == (True, "resident", "resident", "dense_groups")
    assert run(["two_steps"]) == (True, "dense_tiles", None, "dense_groups")
    assert run(["dense_groups"]) == (False, "resident", None, "row_blocks")
