"""The forward kernels keep their state in registers: a spilled one comes back through a wait for the vector-memory counter, which
also waits for the tile copies in flight, and a spilled scalar takes two instructions of the loop.  The compiler notes the spills of
every kernel in the code object of the library."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from psa_hip import _lib

READELF = next((p for p in (shutil.which("llvm-readelf"), "/opt/rocm/llvm/bin/llvm-readelf") if p and os.path.exists(p)), None)


def _kernels(tmp_path):
    """{mangled name: metadata} of every kernel in the library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    with open(_lib.LIB_PATH, "rb") as f:
        blob = f.read()
    res, at = {}, blob.find(magic)
    while at >= 0:
        pos = at + len(magic)
        (n,) = struct.unpack_from("<Q", blob, pos)
        pos += 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, pos)
            ident = blob[pos + 24 : pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" in ident and size:
                path = tmp_path / "code.elf"
                path.write_bytes(blob[at + off : at + off + size])
                notes = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True, text=True).stdout
                for block in re.split(r"\n\s+- \.a(?:gpr_count|rgs):", notes)[1:]:
                    # (the kernel's own name is the last one, behind those of its arguments)
                    meta = dict(re.findall(r"\.(name|[sv]gpr_spill_count|private_segment_fixed_size):\s+(\S+)\s*$", block, re.M))
                    res[meta["name"]] = meta
        at = blob.find(magic, at + 1)
    return res


@pytest.mark.skipif(READELF is None, reason="llvm-readelf of the ROCm toolchain not found")
@pytest.mark.parametrize("kernel,instances", [("psa_fwd_kernel", 20), ("psa_fwd_lds_kernel", 20)])
def test_forward_kernels_do_not_spill(kernel, instances, tmp_path):
    found = {n: m for n, m in _kernels(tmp_path).items() if re.search(r"\d%sI" % kernel, n)}
    assert len(found) == instances, sorted(found)
    spilled = {n: m for n, m in found.items() if any(int(m[c]) for c in ("vgpr_spill_count", "sgpr_spill_count", "private_segment_fixed_size"))}
    assert not spilled, spilled


@pytest.mark.skipif(READELF is None, reason="llvm-readelf of the ROCm toolchain not found")
def test_the_contraction_keeps_its_accumulators(tmp_path):
    """The MFMAs of its large tile are written with their accumulators in place: nothing else may move them in between."""
    found = {n: m for n, m in _kernels(tmp_path).items() if "psa_xattn_gemm_kernel" in n}
    assert len(found) == 15, sorted(found)
    spilled = {n: m for n, m in found.items() if any(int(m[c]) for c in ("vgpr_spill_count", "sgpr_spill_count", "private_segment_fixed_size"))}
    assert not spilled, spilled
