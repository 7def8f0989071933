"""The workgroups of a grid barrier wait for each other, so all of them must be on the
device at once, also on its smallest partition (32 CUs) and beside three more launches of the
same kind on a whole chip (256 CUs).  Read off the built library: what the code object's notes
say that a workgroup of the kernel takes (LDS, vector registers, waves) against what a CU has
(160 KB, 512 registers for each of 4 SIMDs, 8 waves per SIMD)."""
import os
import re
import shutil
import struct
import subprocess

import pytest
import yaml

import nns_amd

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
LIB = os.path.join(os.path.dirname(nns_amd.__file__), "libnbx.so")
SOURCE = os.path.join(os.path.dirname(nns_amd.__file__), "csrc", "k_tree.hip")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(lib):
    data = open(lib, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            off, size, tlen = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + tlen].decode()
            p += 24 + tlen
            if "gfx950" in triple and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


def kernels(lib, tmp_path):
    found = {}
    for k, obj in enumerate(code_objects(lib)):
        path = tmp_path / f"{k}.o"
        path.write_bytes(obj)
        text = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        doc = text[text.index("---"):text.index("\n...")]
        for kernel in yaml.safe_load(doc)["amdhsa.kernels"]:
            found[kernel[".name"]] = kernel
    return found


def test_grid_barrier_workgroups_fit_the_smallest_partition(tmp_path):
    if not os.path.exists(LIB) or not os.path.exists(READELF):
        pytest.skip("no built library, or no tool to read its notes")
    source = open(SOURCE).read()
    blocks = int(re.search(r"\bkTopBlocks = (\d+)", source).group(1))
    # every kernel with the barrier: those whose body calls it
    names = {re.findall(r"__global__[^{;]*?\b(\w+_kernel)\(", source[:m.start()])[-1]
             for m in re.finditer(r"(?<!void )\btop_barrier\(", source)}
    assert names
    taken = {k: v for k, v in kernels(LIB, tmp_path).items() if any(n in k for n in names)}
    assert taken
    for name, k in taken.items():
        waves = -(-k[".max_flat_workgroup_size"] // 64)
        regs = -(-max(k[".vgpr_count"] + k.get(".agpr_count", 0), 1) // 8) * 8
        per_simd = min(8, 512 // regs)
        fit = min(4 * per_simd // waves, 160 * 1024 // max(k[".group_segment_fixed_size"], 1))
        assert 32 * fit >= blocks, (name, "smallest partition", fit, k)
        assert 256 * fit >= 4 * blocks + 256, (name, "four launches and as many other workgroups as CUs", fit)
