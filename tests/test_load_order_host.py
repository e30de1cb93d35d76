"""Issue order of the vector-memory operations whose partial waits (vmcnt) rely on it, read from the gfx950 code that
the build left in libmolt_amd.so. The order of a round's own loads is free; no load of one round may be issued among
those of another."""
from __future__ import annotations

import re
import shutil
import struct
import subprocess

import pytest

from molt_amd.build import ARCH, LIB

LLVM = "/opt/rocm/llvm/bin/"
needs_build = pytest.mark.skipif(not (LIB.exists() and shutil.which(LLVM + "llvm-objdump")),
                                 reason="no built library or no llvm-objdump")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects():
    """The gfx950 code objects in the library's offload bundles."""
    data = LIB.read_bytes()
    at = data.find(MAGIC)
    while at >= 0:
        pos = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + n].decode()
            pos += 24 + n
            if name.endswith(ARCH) and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 24)


def _kernels(tmp_path, name: str) -> dict[str, list[str]]:
    """Instructions of every kernel whose symbol contains ``name``."""
    found: dict[str, list[str]] = {}
    for i, code in enumerate(_code_objects()):
        if name.encode() not in code:
            continue
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        text = subprocess.run([LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", str(path)], capture_output=True,
                              text=True, check=True).stdout
        for part in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:]:
            sym, body = part.split(">:", 1)
            if name in sym:
                found[sym] = [ln.split("//")[0].strip() for ln in body.splitlines() if ln.strip()]
    return found


def _memory(instructions: list[str]) -> list[str]:
    """'D' for a DMA into LDS, 'L' for a load into registers, 'W<n>' for a wait of vmcnt(n), '|' for a barrier."""
    out = []
    for t in instructions:
        if re.match(r"(buffer|global)_load_", t):
            out.append("D" if re.search(r"\blds\b", t) else "L")
        elif m := re.search(r"s_waitcnt .*vmcnt\((\d+)\)", t):
            out.append("W" + m.group(1))
        elif t.startswith("s_barrier"):
            out.append("|")
    return out


@needs_build
def test_streamed_gemv_issues_its_rounds_in_order(tmp_path):
    """Up to 8 tokens, several rounds: the first round's wait leaves the youngest two rounds' loads in flight, so the
    prologue must issue X, all of round 0, then all of round 1: the same pattern of DMA and loads twice."""
    kernels = {s: k for s, k in _kernels(tmp_path, "nf4_gemv_lds_kernel").items() if "Lb0E" in s}
    assert len(kernels) == 9, sorted(kernels)          # three scale forms by three adapter forms
    for sym, ins in kernels.items():
        sm, lv = (int(v) for v in re.search(r"ILi(\d)ELi(\d)ELb0E", sym).groups())
        per = 2 + (4, 6, 2)[sm] + (0, 2, 2)[lv]        # two DMAs, statistics, adapter entries
        seq = [e for e in _memory(ins) if e in "DL" or e == f"W{2 * per}"]
        heads = ["".join(seq[max(0, i - 4 - 2 * per):i]) for i, e in enumerate(seq) if e not in "DL"]
        heads = [h for h in heads if h.startswith("DDDD") and "W" not in h]
        assert heads, f"{sym}: no prologue of four X loads and two rounds before a wait of {2 * per}"
        for h in heads:
            rounds = h[4:4 + per], h[4 + per:]
            assert rounds[0].count("D") == rounds[1].count("D") == 2, f"{sym}: {h}"
        # and each further round issues as many operations as its wait counts (merged loads would not be)
        between = "".join(e[0] for e in seq).split("W")
        assert [n for n in map(len, between[-4:-1])] == [per] * 3, f"{sym}: {per} a round, got {between[-4:]}"


@needs_build
def test_streamed_gemv_holds_its_rounds_in_registers(tmp_path):
    """The streamed GEMV spills no vector registers (a spill's reload waits for the weight stream), but for two in the
    form of per-block codes and ranks that are no groups of four."""
    spills = {}
    for i, code in enumerate(_code_objects()):
        if b"nf4_gemv_lds_kernel" in code:
            (tmp_path / f"{i}.co").write_bytes(code)
            notes = subprocess.run([LLVM + "llvm-readelf", "--notes", str(tmp_path / f"{i}.co")], capture_output=True,
                                   text=True, check=True).stdout
            spills.update(re.findall(r"\.name:\s+(\S*nf4_gemv_lds_kernel\S*).*?\.vgpr_spill_count:\s+(\d+)", notes, re.S))
    assert len(spills) == 18
    over = {k: int(v) for k, v in spills.items() if int(v) > (2 if "ILi1ELi2ELb0E" in k else 0)}
    assert not over, over
