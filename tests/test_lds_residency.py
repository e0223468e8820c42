"""LDS of the small-M int8 kernels in the built gfx950 code, read from the code
objects' metadata (no GPU needed): a CU's 160 KB are dealt in pieces of 1280
bytes, and at these widths a few hundred bytes decide how many workgroups fit."""
import os
import re
import subprocess

import pytest

from glypr_amd import _lib
from test_codegen_guard import MAGIC, TARGET, _tool


@pytest.fixture(scope="module")
def lds_bytes(tmp_path_factory):
    tools = [_tool(n) for n in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf")]
    if not os.path.exists(_lib.LIB_PATH) or not all(tools):
        pytest.skip("libglypr_hip.so not built or ROCm LLVM tools missing")
    objcopy, bundler, readelf = tools
    d = tmp_path_factory.mktemp("notes")
    fat = d / "fat.bin"
    subprocess.run([objcopy, f"--dump-section=.hip_fatbin={fat}", _lib.LIB_PATH, str(d / "x.so")],
                   check=True, capture_output=True)
    data = fat.read_bytes()
    starts = [m.start() for m in re.finditer(re.escape(MAGIC), data)] + [len(data)]
    out = {}
    for i, (a, b) in enumerate(zip(starts, starts[1:])):
        part, co = d / f"b{i}.bin", d / f"b{i}.co"
        part.write_bytes(data[a:b])
        subprocess.run([bundler, "--type=o", "--unbundle", f"--input={part}",
                        f"--targets={TARGET}", f"--output={co}"], check=True, capture_output=True)
        notes = subprocess.run([readelf, "--notes", str(co)], check=True, capture_output=True,
                               text=True).stdout
        for size, name in re.findall(r"\.group_segment_fixed_size:\s*(\d+).*?\n\s+\.name:\s*(\S+)",
                                     notes, re.S):
            out[name] = int(size)
    return out


@pytest.mark.parametrize("kernel,per_cu", [
    (r"gemm_i8_small_kernelILi1ELi2ELi1ELb0ELb[01]ELi3ELi64ELb0E", 5),
    (r"gemm_i8_small_kernelILi1ELi2ELi1ELb0ELb[01]ELi3ELi32ELb0E", 6),
    (r"gemm_i8_geglu8_kernelILb[01]ELi2ELi32E", 5)])
def test_workgroups_per_cu(lds_bytes, kernel, per_cu):
    sizes = [v for k, v in lds_bytes.items() if re.search(kernel, k)]
    assert len(sizes) == 2    # exact and two-op epilogue
    for v in sizes:
        assert 160 * 1024 // (-(-v // 1280) * 1280) == per_cu, v
