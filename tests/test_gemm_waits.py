"""The built W8A16 GEMMs' waits in the K loop, read from the library's own gfx950 code (no GPU).

A K-step widens the next tile's int8 weights from registers while the loads of the tiles after it are in flight. The
compiler places the waits for those registers, and it counts the loads issued behind them on every path: a branch that
could leave some of those loads out makes it wait for the others too, with the same results but with the loads in flight
for half as long.
"""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

import mako_h3

BIN = Path(shutil.which("hipcc") or "/opt/rocm/bin/hipcc").resolve().parent.parent / "llvm" / "bin"
OBJDUMP = next((p for p in (BIN / "llvm-objdump", Path("/opt/rocm/llvm/bin/llvm-objdump")) if p.exists()), None)
GFX = "hipv4-amdgcn-amd-amdhsa--gfx950"


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    if OBJDUMP is None:
        pytest.skip("llvm-objdump is not installed")
    lib = Path(shutil.copy(mako_h3.LIB_PATH, tmp_path_factory.mktemp("lib") / "lib.so"))
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True)
    return sorted(lib.parent.glob(f"*{GFX}"))


def instructions(code_objects, kernel):
    """(offset, mnemonic and operands, branch target or None) of the kernel whose mangled name holds `kernel`."""
    for obj in code_objects:
        names = subprocess.run([OBJDUMP, "--syms", obj], check=True, capture_output=True, text=True).stdout
        name = next((w for w in re.findall(r"\bF \.text.* (\S+)$", names, re.M) if kernel in w), None)
        if name is None:
            continue
        text = subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={name}", obj], check=True, capture_output=True,
                              text=True).stdout
        out = []
        for line in text.splitlines():
            m = re.match(r"\s+(\S.*?)\s*// ([0-9A-F]+):(?:.*<\S+\+0x([0-9a-f]+)>)?", line)
            if m:
                out.append((int(m[2], 16), m[1], int(m[3], 16) if m[3] else None))
        base = out[0][0]
        return [(at - base, op, to) for at, op, to in out]
    raise AssertionError(f"no kernel {kernel} in the library")


def k_loops(ops):
    """The innermost loops over K-steps: the instructions from a backward branch's target to the branch."""
    found = []
    for at, op, to in ops:
        if to is not None and to < at and "branch" in op:
            body = [o for a, o, _ in ops if to <= a <= at]
            if any(o.startswith("v_mfma") for o in body) and any(o.startswith("s_barrier") for o in body):
                found.append(body)
    return found


def load_waits(body):
    return [int(m[1]) for o in body if (m := re.match(r"s_waitcnt.*vmcnt\((\d+)\)", o))]


@pytest.mark.parametrize("epi", [0, 1, 2, 3])
@pytest.mark.parametrize("rows", [64, 128, 192, 256])
def test_w8a16_widening_leaves_later_loads_in_flight(code_objects, rows, epi):
    # A wave issues rows / 64 loads of x behind its two of w a K-step. Widening w's registers may not wait for them; the
    # one full wait of a step comes after it.
    loops = k_loops(instructions(code_objects, f"gemm_kernelILi{rows}ELi128ELi2ELi4ELi0ELi{epi}E"))
    assert len(loops) == 1
    waits = load_waits(loops[0])
    assert waits[-1] == 0 and len(waits) > 1
    assert min(waits[:-1]) >= rows // 64, waits


@pytest.mark.parametrize("epi", [0, 1, 2, 3])
def test_w8a16_narrow_tile_keeps_two_later_tiles_in_flight(code_objects, epi):
    # Three register sets of w: a step's loads are one of w and two of x, and no wait of the three steps that the loop
    # without branches holds may leave fewer than the two later tiles' six in flight.
    loops = k_loops(instructions(code_objects, f"gemm_kernelILi64ELi32ELi2ELi2ELi0ELi{epi}E"))
    waits = max((load_waits(body) for body in loops), key=min)
    assert len(waits) >= 3 and min(waits) >= 6, [load_waits(body) for body in loops]
