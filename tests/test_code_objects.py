"""What the compiler made of some kernels, read from the built library's gfx950 code objects (no GPU): properties that a
small change of the source has lost before without any wrong result."""
import functools
import os
import re
import subprocess

import pytest

import mechta_amd as mk

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@functools.lru_cache(None)
def disassembly(tmp):
    """{mangled kernel name: its instructions} of every code object in the library."""
    blob = open(mk.LIB_PATH, "rb").read()
    out = {}
    for m in list(re.finditer(b"\x7fELF", blob))[1:]:  # the first is the library itself
        path = os.path.join(tmp, f"{m.start()}.co")
        with open(path, "wb") as f:
            f.write(blob[m.start():])
        r = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", path], capture_output=True, text=True)
        name = None
        for line in r.stdout.splitlines():
            h = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if h:
                name = h.group(1)
                out[name] = []
            elif name and line.startswith("\t"):
                out[name].append(line.strip())
    return out


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    return disassembly(str(tmp_path_factory.mktemp("co")))


def kernels(code, part):
    found = {n: c for n, c in code.items() if part in n and len(c) > 50}
    assert found, part
    return found


@pytest.mark.parametrize("part", ["11prefill_f16", "11prefill_f32"])
def test_prefill_mask_is_no_scalar_chain(code, part):
    """A tile that crosses a row's window takes one comparison per score (16 a lane). With one for each bound the compiler
    passed every pair through vcc, 16 dependent vector-scalar-vector round trips per tile."""
    for name, ins in kernels(code, part).items():
        chained = [i for i in ins if re.match(r"s_and_b64 vcc, (vcc, s\[|s\[\d+:\d+\], vcc)", i)]
        assert len(chained) < 8, f"{name}: {len(chained)} scalar ands of vcc"


@pytest.mark.parametrize("elem,loads", [("t", 4), ("f", 8)])
def test_rows_into_v_loads_in_flight(code, elem, loads):
    """Rows written into V planes: a thread's chunks (4 of f16, 8 of f32) are all loaded before the first is waited for.
    Behind a branch each, they were loaded one at a time (f32: 230 registers, 4.5 us for 100 positions against 2.3)."""
    for name, ins in kernels(code, f"rows_tileI{elem}").items():
        if "ELi1ELi1E" not in name:  # into the planes, V
            continue
        ops = [i.split()[0] + (" vmcnt" if "vmcnt" in i else "") for i in ins]
        first = ops.index("global_load_dwordx4")
        wait = next(k for k in range(first, len(ops)) if ops[k] == "s_waitcnt vmcnt")
        assert ops[first:wait].count("global_load_dwordx4") == loads, name
