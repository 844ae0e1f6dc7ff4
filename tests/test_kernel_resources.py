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

def _tool(name):
    return next((p for p in (shutil.which(name), "/opt/rocm/llvm/bin/" + name) if p and os.path.exists(p)), None)


READELF, OBJDUMP = _tool("llvm-readelf"), _tool("llvm-objdump")


def _code_objects(tmp_path):
    """Files of the code objects in the library, one after the other."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    with open(_lib.LIB_PATH, "rb") as f:
        blob = f.read()
    at = blob.find(magic)
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
                yield path
        at = blob.find(magic, at + 1)


def _kernels(tmp_path):
    """{mangled name: metadata} of every kernel in the library."""
    res = {}
    for path in _code_objects(tmp_path):
        notes = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True, text=True).stdout
        for block in re.split(r"\n\s+- \.a(?:gpr_count|rgs):", notes)[1:]:
            # (the kernel's own name is the last one, behind those of its arguments)
            meta = dict(re.findall(r"\.(name|[sv]gpr_spill_count|private_segment_fixed_size):\s+(\S+)\s*$", block, re.M))
            res[meta["name"]] = meta
    return res


@pytest.mark.skipif(READELF is None, reason="llvm-readelf of the ROCm toolchain not found")
@pytest.mark.parametrize("kernel,instances", [("psa_fwd_kernel", 20), ("psa_fwd_lds_kernel", 20)])
def test_forward_kernels_do_not_spill(kernel, instances, tmp_path):
    found = {n: m for n, m in _kernels(tmp_path).items() if re.search(r"\d%sI" % kernel, n)}
    assert len(found) == instances, sorted(found)
    spilled = {n: m for n, m in found.items() if any(int(m[c]) for c in ("vgpr_spill_count", "sgpr_spill_count", "private_segment_fixed_size"))}
    assert not spilled, spilled


@pytest.mark.skipif(READELF is None, reason="llvm-readelf of the ROCm toolchain not found")
def test_the_contraction_does_not_spill(tmp_path):
    found = {n: m for n, m in _kernels(tmp_path).items() if "psa_xattn_gemm_kernel" in n}
    assert len(found) == 15, sorted(found)
    spilled = {n: m for n, m in found.items() if any(int(m[c]) for c in ("vgpr_spill_count", "sgpr_spill_count", "private_segment_fixed_size"))}
    assert not spilled, spilled


def _regs(operand, kind):
    """Numbers of the registers of an operand like v7 or v[4:7]."""
    m = re.fullmatch(kind + r"(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return set()
    return {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))


@pytest.mark.skipif(OBJDUMP is None, reason="llvm-objdump of the ROCm toolchain not found")
def test_the_contraction_keeps_its_accumulators(tmp_path):
    """The MFMAs of its large tile are inline assembly with the accumulator in place, and its copies are inline assembly too: the
    compiler knows neither what such an MFMA needs between itself and other users of its registers nor that a copy reads scalar
    registers.  In the code that it made: nothing else touches an accumulator from the first MFMA of the loop to the last, no vector
    instruction right before one writes what it reads, the waits around them are there, and no copy's descriptor comes from the vector
    unit less than five instructions before."""
    found = 0
    for path in _code_objects(tmp_path):
        if b"psa_xattn_gemm_kernel" not in path.read_bytes():
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], check=True, capture_output=True, text=True).stdout
        for fn in re.split(r"\n(?=\S*\s*<[^>]+>:)", text):
            if not re.match(r"\s*\S*\s*<\S*psa_xattn_gemm_kernelILi[345]ENS_5XTileILi8ELi8ELi1EE", fn):
                continue
            found += 1
            code = [re.sub(r"\s*//.*", "", line).strip() for line in fn.splitlines()]
            code = [c for c in code if c and not c.endswith(":")]
            op = [c.split(None, 1)[0] for c in code]
            args = [re.split(r",\s*", c.split(None, 1)[1]) if " " in c else [] for c in code]
            at = [i for i, o in enumerate(op) if o.startswith("v_mfma")]
            assert len(at) == 128
            first, last = at[0], at[-1]
            uses = {}
            for i in at:
                d, a, b, c = args[i]
                assert op[i] == "v_mfma_f32_16x16x32_bf16" and d == c and len(_regs(d, "a")) == 4
                uses[d] = uses.get(d, 0) + 1
                reads = _regs(a, "v") | _regs(b, "v")
                assert len(reads) == 8
                for j in (i - 1, i - 2):
                    if op[j].startswith("v_") and not op[j].startswith("v_mfma"):
                        assert not _regs(args[j][0], "v") & reads, (code[j], code[i])
            assert len(uses) == 64 and set(uses.values()) == {2}
            others = [c for i, c in enumerate(code[first:last + 1], first) if i not in at and re.search(r"accvgpr|\ba\d|\ba\[", c)]
            assert not others, others
            assert not [o for o in op[first:last] if "branch" in o or "setpc" in o]
            # the zeroes before them, the results behind them
            before = max(i for i in range(first) if "accvgpr_write" in op[i])
            assert "s_nop 7" in code[before:first]
            behind = next(i for i in range(last + 1, len(code)) if re.search(r"accvgpr|\ba\d|\ba\[", code[i]))
            assert code[last:behind].count("s_nop 15") >= 2
            copies = [i for i, c in enumerate(code) if op[i].startswith("buffer_load") and c.endswith("lds")]
            assert len(copies) >= 48  # two stages before the loop, one in it
            for i in copies:
                desc = _regs(args[i][1], "s")
                assert len(desc) == 4
                for j in range(max(0, i - 5), i):
                    assert not (op[j].startswith("v_readfirstlane") or op[j].startswith("v_readlane")) or not _regs(args[j][0], "s") & desc, code[j:i + 1]
    assert found == 3
