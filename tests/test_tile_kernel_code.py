"""CPU tests: properties of the built wavefront kernels that their speed rests on.

Read from the gfx950 code object inside the in-tree library (built from this
source by the Makefile) with the ROCm toolchain's readelf and objdump.
"""
import os
import re
import struct
import subprocess

import pytest

import cqmm

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(lib):
    data = open(lib, "rb").read()
    for m in re.finditer(re.escape(MAGIC), data):
        at = m.start() + len(MAGIC)
        (n,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, at)
            name = data[at + 24:at + 24 + idlen]
            at += 24 + idlen
            if b"gfx950" in name:
                yield data[m.start() + off:m.start() + off + size]


@pytest.fixture(scope="module")
def tile_code(tmp_path_factory):
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("no ROCm LLVM tools")
    for obj in _code_objects(cqmm.LIB_PATH):
        if b"k_wave_products" in obj:
            path = tmp_path_factory.mktemp("code") / "tile.co"
            path.write_bytes(obj)
            return str(path)
    raise AssertionError("no gfx950 code object with the wavefront kernels in the library")


def _wave_kernels(path):
    out = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "-sW", path], capture_output=True, text=True,
                         check=True).stdout
    names = sorted({w for w in out.split() if "k_wave_products" in w and "." not in w})
    assert names
    return names


def test_results_are_written_without_waiting_for_loads(tile_code):
    """A load between the stores of the results would wait for the stores before it."""
    names = _wave_kernels(tile_code)
    out = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn",
                          "--disassemble-symbols=" + ",".join(names), tile_code], capture_output=True, text=True,
                         check=True).stdout
    seen = 0
    for body in re.split(r"^[0-9a-f]+ <", out, flags=re.M)[1:]:
        name, code = body.split(">", 1)
        stores = code.index("global_store")
        assert not re.search(r"\b(global|flat|scratch)_load", code[stores:]), name
        seen += 1
    assert seen == len(names)


def test_registers_and_lds_fit_the_wavefronts(tile_code):
    """Two wavefronts per SIMD for FP64 blocks of 13 and 16, three for the others; no
    scratch memory but, in split BF16, for a few lane constants around the loop."""
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", tile_code], capture_output=True, text=True,
                           check=True).stdout
    names = set(_wave_kernels(tile_code))
    seen = 0
    for kernel in notes.split("  - .agpr_count")[1:]:
        field = dict(re.findall(r"^\s*\.(\w+):\s+(\S+)$", kernel, flags=re.M))
        if field["name"] not in names:
            continue
        mode, nsf = map(int, re.search(r"k_wave_productsILi(\d+)ELb[01]ELi(\d+)E", field["name"]).groups())
        waves = 2 if mode == 0 and nsf > 9 else 3
        assert int(field["vgpr_count"]) <= 512 // waves // 8 * 8, (field["name"], field["vgpr_count"])
        assert int(field["group_segment_fixed_size"]) * 4 * waves <= 160 * 1024, field["name"]
        assert int(field["private_segment_fixed_size"]) <= (32 if mode == 4 else 0), field["name"]
        seen += 1
    assert seen == len(names)
