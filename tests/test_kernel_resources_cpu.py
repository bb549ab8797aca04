"""What the built library's kernels take of a CU, from the code objects in it
(the metadata the compiler wrote for this library's own sources): no GEMM kernel
keeps values in scratch memory, where a register spill of the main loop costs it
several times its time."""
import os
import re
import shutil
import struct
import subprocess

import pytest

import mxenc

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects of a shared library's fat binaries."""
    blob = open(path, "rb").read()
    at = blob.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + idlen].decode()
            p += 24 + idlen
            if "gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + len(MAGIC))


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Demangled kernel name -> bytes of scratch per lane."""
    if not os.path.exists(READELF):
        pytest.skip("needs llvm-readelf")
    if not os.path.exists(mxenc.LIB_PATH):
        pytest.skip("the library is not built")
    out = {}
    f = tmp_path_factory.mktemp("co") / "co.elf"
    for co in code_objects(mxenc.LIB_PATH):
        f.write_bytes(co)
        notes = subprocess.run([READELF, "--notes", str(f)], check=True, capture_output=True,
                               text=True).stdout
        # a kernel's entry lists its fields in order of their names
        for name, scratch in re.findall(
                r"\.name:\s+(_Z\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)", notes):
            out[name] = int(scratch)
    names = subprocess.run(["c++filt"], input="\n".join(out), check=True, capture_output=True,
                           text=True).stdout.split("\n")
    return {n.replace("void (anonymous namespace)::", "").split("(")[0]: s
            for n, s in zip(names, out.values())}


def test_gemm_kernels_use_no_scratch(kernels):
    gemm = {n: s for n, s in kernels.items() if n.startswith("gemm_")}
    assert len(gemm) > 100
    # 8 bytes: one register of an epilogue, out of the main loop
    assert not {n: s for n, s in gemm.items() if s > 8}


def test_one_mfma_form_per_tile(kernels):
    """A tile's kernel exists in the MFMA form that its launcher takes, not in
    the other as well."""
    args = lambda name: {n[len(name):] for n in kernels if n.startswith(name + "<")}  # noqa: E731
    for a, b in (("gemm_lds_k", "gemm_lds16_k"), ("gemm_i8_k", "gemm_i8_16_k")):
        assert len(args(a)) > 20 and len(args(b)) > 5
        assert not args(a) & args(b)
