"""What the compiler made of this library's dense kernels, read from the
metadata of the code objects in libpet_attn.so: their accumulators stay in
registers. A wave's 64 x 128 tile is 512 bytes of accumulators a lane; indexed
by anything but constants they move to scratch, and every step of the K loop
then reads and writes them there."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from pet_kokkos_amd import _lib

LLVM = "/opt/rocm/llvm/bin"
TOOLS = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf")]


def kernels(tmp_path):
    """{mangled name: scratch bytes a lane} of every gfx950 kernel."""
    if not all(map(os.path.exists, TOOLS)):
        pytest.skip("the ROCm LLVM tools are not installed")
    objcopy, bundler, readelf = TOOLS
    fat = str(tmp_path / "fatbin")
    subprocess.run([objcopy, "--dump-section", f".hip_fatbin={fat}", _lib.LIB_PATH, str(tmp_path / "copy")], check=True)
    data = open(fat, "rb").read()
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)]
    out = {}
    for i, p in enumerate(starts):
        bundle, obj = str(tmp_path / f"b{i}"), str(tmp_path / f"o{i}")
        with open(bundle, "wb") as f:
            f.write(data[p:starts[i + 1] if i + 1 < len(starts) else None])
        subprocess.run([bundler, "--type=o", "--unbundle", f"--input={bundle}", f"--output={obj}",
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
        notes = subprocess.run([readelf, "--notes", obj], check=True, capture_output=True, text=True).stdout
        for k in re.split(r"\n  - \.a", notes)[1:]:
            name, size = re.search(r"\.name:\s+(\S+)", k), re.search(r"\.private_segment_fixed_size:\s+(\d+)", k)
            out[name[1]] = int(size[1])
    return out


def test_dense_kernels_keep_their_accumulators_in_registers(tmp_path):
    dense = {n: s for n, s in kernels(tmp_path).items() if re.search(r"gemm_(rows|ksplit|strip)_kernel", n)}
    assert len(dense) > 20
    assert {n: s for n, s in dense.items() if s > 256} == {}


def test_tiles_from_rows_and_pairs_use_no_scratch(tmp_path):
    """Three registers spilled in the K loop of the 256 x 256 tiles cost 11% of
    their time (62291 x 1024 x 512: 290 us against 259), so of the tile kernels only
    the one with block pairs out, whose epilogue spills, uses scratch."""
    tiles = {n: s for n, s in kernels(tmp_path).items() if "gemm_rows_kernel" in n}
    assert len(tiles) > 10
    assert [n for n, s in tiles.items() if s > 0 and "ILi4ELi8ELi4ELi2ELi2ELi2ELi2EE" not in n] == []
