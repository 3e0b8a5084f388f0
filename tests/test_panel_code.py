"""The panel kernel's compiled code (``csrc/w4a16_panel.hip``): its matrix products are inline
asm, whose latency the compiler does not know, and the waits for its LDS DMA count by hand the
loads issued since. Reads the code that this tree built; no GPU needed."""

from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
# cycles after which a VALU may read what a 16x16x32 product (at most eight passes) wrote
WAIT = 11


def _panel_kernels(tmp_path: Path) -> dict[str, list[str]]:
    """The instructions of every panel kernel, by its name."""
    from slipstream_amd import build

    if not OBJDUMP.exists():
        pytest.skip("no llvm-objdump")

    lib = tmp_path / "lib.so"
    shutil.copy(build.OUT_DIR / build.LIB_NAME, lib)
    subprocess.run([OBJDUMP, "--offloading", str(lib)], check=True, capture_output=True, cwd=tmp_path)
    for code in tmp_path.glob("lib.so.*gfx950"):
        if b"w4a16_panel_kernel" not in code.read_bytes():
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(code)], check=True, capture_output=True,
                              text=True).stdout
        kernels = {}
        for part in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:]:
            name, body = part.split(">:", 1)
            if "w4a16_panel_kernel" in name:
                kernels[name] = [line.split("//")[0].strip() for line in body.splitlines() if line.startswith("\t")]
        assert len(kernels) == 20  # two dtypes, five panel heights, two widths
        return kernels
    raise AssertionError("no panel kernel in the library")


def test_accumulators_are_read_after_the_products_latency(tmp_path):
    """The last product and the first instruction that reads an accumulator register (copies
    that the compiler adds included) are at least the product's latency apart, at one cycle an
    instruction and n + 1 for an s_nop n; before that only the products read accumulators."""
    for name, code in _panel_kernels(tmp_path).items():
        products = [i for i, line in enumerate(code) if line.startswith("v_mfma")]
        last = products[-1]
        reads = [i for i, line in enumerate(code) if i > products[0] and not line.startswith("v_mfma")
                 and re.search(r",.*\ba\[?\d", line)]
        assert reads and reads[0] > last, name
        cycles = sum(int(line.split()[1]) + 1 if line.startswith("s_nop") else 1 for line in code[last + 1 : reads[0]])
        assert cycles >= WAIT, f"{name}: {cycles} cycles from {code[last]!r} to {code[reads[0]]!r}"


def test_dma_waits_leave_what_the_half_stage_issued(tmp_path):
    """Each half stage ends with a wait for all but the loads that it issued itself and a
    barrier: the hand-written count is the number of loads between the barriers."""
    for name, code in _panel_kernels(tmp_path).items():
        last = max(i for i, line in enumerate(code) if line.startswith("v_mfma"))
        barriers = [i for i, line in enumerate(code) if line == "s_barrier"]
        second = next(i for i in barriers if i > last)
        k = barriers.index(second)
        for begin, end in ((barriers[k - 2], barriers[k - 1]), (barriers[k - 1], second)):
            loads = sum(line.startswith("buffer_load") for line in code[begin:end])
            wait = next(line for line in reversed(code[begin:end]) if "vmcnt" in line)
            assert int(re.search(r"vmcnt\((\d+)\)", wait)[1]) == loads, (name, wait, loads)
