"""The compiled sweeps keep what their speed rests on: scalar buffer
descriptors in the frequency loops (a descriptor that the compiler takes for
divergent turns every access into a loop over the lanes) and the waves per SIMD
that their registers allow.  Read from the library built here; no GPU."""
import os
import re
import struct
import subprocess

import pytest

from umwm_amd import build

msgpack = pytest.importorskip("msgpack")

OBJDUMP = os.path.join(build.ROCM, "llvm", "bin", "llvm-objdump")


def code_objects():
    """The gfx950 code objects of the library (clang offload bundles)."""
    with open(build.LIB, "rb") as f:
        data = f.read()
    at, out = 0, []
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        q = at + 32
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", data, q)
            name = data[q + 24:q + 24 + ln]
            q += 24 + ln
            if b"gfx950" in name and size:
                out.append(data[at + off:at + off + size])
        at += 24
    return out


def kernels(elf):
    """Kernel records of a code object's metadata note."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 24)
        while kind == 7 and size >= 12:  # SHT_NOTE
            ns, ds, nt = struct.unpack_from("<III", elf, off)
            body = off + 12 + (ns + 3) // 4 * 4
            if nt == 32:  # AMDGPU metadata
                return msgpack.unpackb(elf[body:body + ds])["amdhsa.kernels"]
            step = 12 + (ns + 3) // 4 * 4 + (ds + 3) // 4 * 4
            off, size = off + step, size - step
    return []


@pytest.fixture(scope="module")
def sweeps(tmp_path_factory):
    """(code object path, {"k_rates<float, 9, ...>": (symbol, VGPRs)})."""
    if not os.path.exists(build.LIB):
        build.build_library()
    for elf in code_objects():
        names = [k[".name"] for k in kernels(elf)]
        if not any("k_rates" in n for n in names):
            continue
        clean = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True,
                               text=True, check=True).stdout.split("\n")
        table = {}
        for k, c in zip(kernels(elf), clean):
            m = re.search(r"(k_\w+<.*?>)\(", c)
            table[m.group(1)] = (k[".name"], k[".vgpr_count"])
        path = tmp_path_factory.mktemp("code") / "sweeps.co"
        path.write_bytes(elf)
        return path, table
    pytest.fail("no code object with the sweeps")


def lane_loops(path, symbol):
    """Loops of one buffer load each over the lanes' descriptors: the lanes that
    share one are compared out before the access, and the branch back on the
    lanes left comes right after it."""
    r = subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={symbol}", str(path)],
                       capture_output=True, text=True, check=True)
    ops = re.findall(r"^\s+([a-z]\w+)", r.stdout, re.M)
    assert len(ops) > 500
    return sum(op.startswith("buffer_load") and "s_cbranch_execnz" in ops[i + 1:i + 6] and
               any(x.startswith("v_cmp_eq_u64") for x in ops[max(i - 10, 0):i])
               for i, op in enumerate(ops))


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
@pytest.mark.parametrize("kernel", ["k_rates<float, 9, true, false, true, true>",
                                    "k_rates<float, 18, true, true, true, true>",
                                    "k_rates<float, 9, true, false, false, false>",
                                    "k_rates<double, 9, true, false, false, true>",
                                    "k_integrate<float, 9, true, true, false>",
                                    "k_integrate<float, 9, true, false, true>",
                                    "k_integrate<double, 9, true, false, false>"])
def test_scalar_descriptors(sweeps, kernel):
    path, table = sweeps
    assert lane_loops(path, table[kernel][0]) == 0


# registers of a wave on a SIMD's 512, in steps of 8
WAVES = {"k_rates<float, 9, true, false, true, true>": 3, "k_rates<float, 9, false, false, true, true>": 3,
         "k_rates<float, 9, true, false, false, false>": 4, "k_rates<float, 36, true, true, false, false>": 3,
         "k_integrate<float, 9, true, true, false>": 3, "k_integrate<float, 12, true, false, false>": 3,
         "k_integrate<float, 9, true, false, true>": 3, "k_rates<double, 9, true, false, false, true>": 2}


@pytest.mark.parametrize("kernel", WAVES)
def test_waves_per_simd(sweeps, kernel):
    _, table = sweeps
    vgprs = (table[kernel][1] + 7) // 8 * 8
    assert 512 // vgprs >= WAVES[kernel], vgprs
