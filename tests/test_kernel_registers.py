"""Registers of the built kernels, from the metadata in their code objects:
the waves a SIMD holds where the launch bounds and the choice of what is kept
in registers were made for them.  And one order of their instructions."""
import os
import re
import shutil
import struct
import subprocess

import pytest

import philtorch_amd

LIB = os.path.join(os.path.dirname(philtorch_amd.__file__), "libphilscan.so")
msgpack = pytest.importorskip("msgpack")
if not os.path.exists(LIB):  # pragma: no cover
    pytest.skip("libphilscan.so not built", allow_module_level=True)

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def _notes(elf):
    """The (type, descriptor) pairs of an ELF's SHT_NOTE sections."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 0x18)
        while kind == 7 and size >= 12:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (namesz + 3) // 4 * 4
            yield ntype, elf[desc:desc + descsz]
            step = desc + (descsz + 3) // 4 * 4 - off
            off, size = off + step, size - step


def _code_objects():
    """The gfx950 ELFs bundled in the library."""
    data = open(LIB, "rb").read()
    for m in re.finditer(re.escape(MAGIC), data):
        n, = struct.unpack_from("<Q", data, m.end())
        p = m.end() + 8
        if n > 16:  # the magic in another place
            continue
        for _ in range(n):
            off, size, tlen = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + tlen]
            p += 24 + tlen
            if b"gfx950" in triple:
                yield data[m.start() + off:m.start() + off + size]


@pytest.fixture(scope="module")
def kernels():
    """mangled name -> metadata of every kernel of the library."""
    out = {}
    for elf in _code_objects():
        for ntype, desc in _notes(elf):
            if ntype == NT_AMDGPU_METADATA:
                for k in msgpack.unpackb(desc, strict_map_key=False)["amdhsa.kernels"]:
                    out[k[".name"]] = k
    assert out, "no kernel metadata found"
    return out


def _some(kernels, pattern):
    found = {n: k for n, k in kernels.items() if re.search(pattern, n)}
    assert found, pattern
    return found.items()


def test_time_varying_state_space_holds_four_waves(kernels):
    """Orders 1-2, every mode but the gradients' (2): 128 VGPRs.  (The fp32
    forward took 130 to 150 and ran 10 to 19 % slower at order 2.)"""
    for name, k in _some(kernels, r"lpv_ss_kernelINS_6(Scalar|Block2)I[fd]EELb[01]ELi[013]E"):
        assert k[".vgpr_count"] <= 128, (name, k[".vgpr_count"])
        if "EELb0ELi" in name:  # forward in time
            assert k[".vgpr_spill_count"] == 0, name


def test_order1_fp64_filters_hold_five_waves(kernels):
    """The forward (plain, and with its final state) of order 1 fp64: 96 VGPRs
    without spills.  (At 98, four waves, lfilter of 24 x 300000 took 35.2 us
    for 32.7.)"""
    for name, k in _some(kernels, r"[0-9]ss_kernelINS_6ScalarIdEELb0ELi[03]E"):
        assert k[".vgpr_count"] <= 96 and k[".vgpr_spill_count"] == 0, (name, k[".vgpr_count"])


def test_multi_input_order4_does_not_spill(kernels):
    """fp32 with 4 inputs, and fp64's form with few steps a lane."""
    for pattern in (r"mimo_ss_kernelINS_6BlockNIfLi4EEELi4E", r"mimo_ss_kernelINS_6BlockNIdLi4EEELi[34]ELb[01]ELb[01]ELb1E"):
        for name, k in _some(kernels, pattern):
            assert k[".vgpr_spill_count"] == 0, (name, k[".vgpr_spill_count"])


def test_streaming_instantiations(kernels):
    """Stores past the caches: scalar and 2x2 real scans and complex64 scalar
    ones, never the time-invariant forward."""
    names = {re.search(r"scan_kernelINS_(.*?)EELb(.)ELb(.)ELb.ELb1E", n).groups()
             for n, _ in _some(kernels, r"scan_kernelI.*ELb[01]ELb[01]ELb0ELb1E")}
    algs = {"6ScalarIf", "6ScalarId", "6ScalarINS_3c64E", "6Block2If", "6Block2Id"}
    assert names == {(a, tv, rev) for a in algs for tv, rev in (("1", "0"), ("1", "1"), ("0", "1"))}
    # the time-varying state space: the gradient mode (2) of orders 1-2
    modes = {re.search(r"lpv_ss_kernelINS_6(.*?)EELb.ELi(.)ELb1E", n).groups()
             for n, _ in _some(kernels, r"lpv_ss_kernelI.*ELi.ELb1E")}
    assert modes == {(a, "2") for a in ("ScalarIf", "ScalarId", "Block2If", "Block2Id")}


OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_rounds_leave_without_a_wait_between(tmp_path):
    """The time-invariant 2x2 fp32 backward: in a whole tile the second round's
    four stores follow the first's with no wait for memory between them.  (A
    wait for a load there waits for the stores before it: 64 x 500000 steps
    took 180 us for 172.)"""
    names = {f"_ZN3phs11scan_kernelINS_6Block2IfEELb0ELb1ELb0ELb{stream}EEEvNS_8ScanArgsIT_EE" for stream in "01"}
    seen = set()
    for i, elf in enumerate(_code_objects()):
        here = {n for n in names if n.encode() in elf}
        if not here:
            continue
        path = tmp_path / f"{i}.elf"
        path.write_bytes(elf)
        text = subprocess.run([OBJDUMP, "-d", "--disassemble-symbols=" + ",".join(sorted(here)), str(path)],
                              stdout=subprocess.PIPE, text=True, check=True).stdout
        for n in here:
            code = re.split(r"\n[0-9a-f]{16} <", text.split(f"<{n}>:", 1)[1])[0]
            # stores of four words S, narrower ones s, waits for memory W, as they lie
            marks = "".join("W" if w else "S" if kind == "x4" else "s" for w, kind in
                            re.findall(r"s_waitcnt [^/\n]*(vmcnt)|global_store_dword(x4|x3|x2|)\b", code))
            assert "SSSSsSSSS" in marks, (n, marks)
            seen.add(n)
    assert seen == names
