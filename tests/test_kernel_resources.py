"""What the kernels of the built library take of a compute unit, from the metadata of its code objects: no scratch memory where
speed rests on registers, and no LDS of one path in a kernel that does not have it."""
import re
import struct
import subprocess

import pytest

import dlspm_hip as dl

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: {"lds", "scratch", "vgpr_spills"}}"""
    dl.lib()
    data, found, at = open(dl.LIB_PATH, "rb").read(), {}, 0
    folder = tmp_path_factory.mktemp("code_objects")
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target, entry = data[entry + 24:entry + 24 + length], entry + 24 + length
            if target.endswith(b"gfx950"):
                path = folder / str(at)
                path.write_bytes(data[at + offset:at + offset + size])
                notes = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True, text=True).stdout
                for part in notes.split("- .agpr_count:")[1:]:
                    number = lambda key: int(re.search(rf"\.{key}:\s+(\d+)", part).group(1))  # noqa: B023, E731
                    found[re.search(r"\.name:\s+(\S+)", part).group(1)] = {
                        "lds": number("group_segment_fixed_size"), "scratch": number("private_segment_fixed_size"),
                        "vgpr_spills": number("vgpr_spill_count")}
        at += 24
    return found


def of(kernels, name):
    return {k: v for k, v in kernels.items() if re.match(rf"_ZN5dlspm\d+{name}I", k)}


def test_resident_kernels_spill_nothing(kernels):
    used = of(kernels, "spmm_resident_kernel")
    assert len(used) == 7
    assert all(v["scratch"] == 0 and v["vgpr_spills"] == 0 for v in used.values()), used


def test_lds_of_the_dense_groups_is_in_their_kernels_only(kernels):
    groups, plain = of(kernels, "fused_groups_kernel"), of(kernels, "fused_kernel")
    assert len(groups) == 30 and all(v["lds"] > 20000 for v in groups.values())
    # per-wave partial rows, four waves: 4 x 4 KB at most for a tile of 1024 columns, sixteen waves of a tile of 512
    assert len(plain) > 100 and max(v["lds"] for v in plain.values()) <= 33000
    four_waves = {k: v for k, v in plain.items() if re.search(r"Li8ELi[234]ELi[01]ELi(16|32)ELi1ELi4ELi\d+EE", k)}
    assert len(four_waves) == 30 and max(v["lds"] for v in four_waves.values()) <= 4096, four_waves


def test_dense_tiles_spill_nothing(kernels):
    used = {k: v for k, v in kernels.items() if re.match(r"_ZN5dlspm\d+(spmm|sddmm)_tiles_kernel", k)}
    assert len(used) == 17
    assert all(v["scratch"] == 0 and v["vgpr_spills"] == 0 for v in used.values()), used
