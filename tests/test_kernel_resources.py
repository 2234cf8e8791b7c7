"""Registers and scratch of the built kernels, from the metadata of the library's
own code objects: the figures that the kernels' comments state, and no vector
register spilled where they say so."""
import os
import re
import struct
import subprocess

import pytest

import __graft_entry__ as entry

msgpack = pytest.importorskip("msgpack")
LIB = os.path.join(entry.PKG_DIR, "libhp3d_pm.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(blob):
    """The gfx950 code objects of the offload bundles in the library."""
    at = blob.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, k = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + k]
            p += 24 + k
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + len(MAGIC))


def metadata(elf):
    """amdhsa.kernels of a code object: the NT_AMDGPU_METADATA note."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entsize, num = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(num):
        kind, = struct.unpack_from("<I", elf, shoff + i * entsize + 4)
        if kind != 7:   # SHT_NOTE
            continue
        off, size = struct.unpack_from("<QQ", elf, shoff + i * entsize + 0x18)
        end = off + size
        while off < end:
            n, d, t = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (n + 3) // 4 * 4
            if t == 32:
                return msgpack.unpackb(elf[desc:desc + d])["amdhsa.kernels"]
            off = desc + (d + 3) // 4 * 4
    return []


@pytest.fixture(scope="module")
def kernels():
    """{"pm_step_kernel<7, 1, 0, ...>": metadata}"""
    with open(LIB, "rb") as f:
        blob = f.read()
    found = [k for elf in code_objects(blob) for k in metadata(elf)]
    names = subprocess.run(["c++filt"], input="\n".join(k[".name"] for k in found),
                           capture_output=True, text=True, check=True).stdout.split("\n")
    out = {re.sub(r"\(.*|^void |hp3d::", "", s.replace("(anonymous namespace)::", "")): k
           for s, k in zip(names, found)}
    assert len(out) > 100
    return out


def of(kernels, name):
    return {k: v for k, v in kernels.items() if k.startswith(name + "<")}


@pytest.mark.parametrize("name", ["pm_halfpass_kernel", "pm_cost_kernel", "pm_halfpass_split_kernel",
                                  "pm_cost_split_kernel"])
def test_view_kernels_fit_four_waves_without_spills(kernels, name):
    ks = of(kernels, name)
    assert ks
    for k, v in ks.items():
        assert v[".vgpr_spill_count"] == 0, (k, v[".vgpr_spill_count"])
        assert v[".vgpr_count"] <= 128, (k, v[".vgpr_count"])


# forms of pm_step.hip: plain, pooled, start only
SPILL = {("11", "1", "0", "1"), ("7", "1", "0", "1"), ("7", "1", "1", "1")}


def test_step_kernels_fit_four_waves_and_spill_only_where_stated(kernels):
    ks = of(kernels, "pm_step_kernel")
    seen = set()
    for k, v in ks.items():
        nt, st, store, _, _, form = re.findall(r"-?\d+", k.split("<")[1])
        assert v[".vgpr_count"] <= 128, (k, v[".vgpr_count"])
        if v[".vgpr_spill_count"]:
            seen.add((nt, st, store, form))
            assert v[".vgpr_spill_count"] <= 16, k
    assert seen <= SPILL, seen - SPILL


@pytest.mark.parametrize("name", ["pm_halfpass_kernel", "pm_step_kernel"])
def test_smallest_windows_fit_five_waves(kernels, name):
    """2 x 2 taps, and 3 x 3 with FP16 planes: 96 registers."""
    for k, v in of(kernels, name).items():
        nt, st, store = re.findall(r"\d+", k.split("<")[1])[:3]
        if nt == "2" or (nt == "3" and store == "1"):
            assert v[".vgpr_count"] <= 96, (k, v[".vgpr_count"])


def test_initial_cost_issues_a_rows_gathers_together(tmp_path):
    """11 x 11 FP32: the 11 gathers of a row come with no vector arithmetic between
    them, in the masked and in the plain tap loop."""
    objdump = "/opt/rocm/llvm/bin/llvm-objdump"
    if not os.path.exists(objdump):
        pytest.skip("no llvm-objdump")
    with open(LIB, "rb") as f:
        blob = f.read()
    for elf in code_objects(blob):
        name = [k[".name"] for k in metadata(elf) if "pm_cost_kernelILi11ELi1ELi0E" in k[".name"]]
        if name:
            break
    path = tmp_path / "k.elf"
    path.write_bytes(elf)
    text = subprocess.run([objdump, "-d", "--no-show-raw-insn", f"--disassemble-symbols={name[0]}",
                           str(path)], capture_output=True, text=True, check=True).stdout
    ops = re.findall(r"^\s+([a-z]\w+)", text, re.M)
    gathers = [i for i, op in enumerate(ops) if op == "buffer_load_dwordx4"]
    assert len(gathers) == 22
    for row in (gathers[:11], gathers[11:]):
        between = [op for op in ops[row[0]:row[-1]] if op.startswith("v_")]
        assert len(between) <= 2, between
