"""How the products of 17 to 128 rows fetch the parts of a sum that K slices left in memory: all of a group before the first is waited for.  Asked for
two at a time, with a wait in between, they cost a trip to memory a pair and nothing in the results shows it."""
import os
import re
import subprocess

import pytest

from fllm_amd.kernels import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SWIGLU = 4


def runs(kernel: str) -> list:
    """How many part loads (buffer_load_dwordx4) lie in a row without a wait for loads between them, row by row."""
    found, run = [], 0
    for line in kernel.splitlines():
        line = line.strip()
        if line.startswith("buffer_load_dwordx4"):
            run += 1
        elif line.startswith("s_waitcnt") and "vmcnt" in line:
            if run:
                found.append(run)
            run = 0
    return found


def longest_run(kernel: str) -> int:
    return max(runs(kernel), default=0)


@pytest.fixture(scope="module")
def text(tmp_path_factory):
    try:
        hipcc = build._hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    listing = tmp_path_factory.mktemp("listing") / "skinny.s"
    source = os.path.join(ROOT, "fllm_amd", "csrc", "linear_skinny.hip")
    run = subprocess.run([hipcc, *build.HIPCC_FLAGS, "--cuda-device-only", "-S", source, "-o", str(listing)], capture_output=True, text=True, timeout=600)
    assert run.returncode == 0, run.stderr
    return listing.read_text()


def test_the_parts_of_a_group_are_asked_for_together(text):
    kernels = re.findall(r"^(\w*skinny_wide_kernelILi(\d+)ELi(\d+)ELb[01]ELi\d+ELi\d+E\w*):.*?^\.Lfunc_end", text, re.S | re.M)
    assert len(kernels) > 20
    for name, row_tiles, epilogue in kernels:
        row_tiles, tiles = int(row_tiles), 2 if int(epilogue) == SWIGLU else 1          # of activations; of weights a wave
        if row_tiles <= 3:         # all row tiles together, of as many slices as there are registers for
            pieces = row_tiles * tiles
            want = pieces * (8 if pieces <= 2 else 4 if pieces <= 4 else 2)
        else:
            want = tiles * (4 if row_tiles > 4 else 8)
        body = text[text.index(f"\n{name}:"):]
        got = longest_run(body[:body.index(".Lfunc_end")])
        assert got >= want, (name, got, want)


def test_the_parts_of_two_slices_are_asked_for_together(text):
    """The kernel that keeps a slice of the rows in LDS.  Left out are the forms for which the compiler has not done so (q/k/v, and gate and up of 49
    to 64 rows, behind a norm)."""
    kernels = re.findall(r"^(\w*skinny_slab_kernelILi(\d)ELi(\d)ELi(\d)E\w*):", text, re.M)
    assert len(kernels) == 21
    for name, prologue, epilogue, row_tiles in kernels:
        if prologue == "1" and (epilogue == "3" or (epilogue, row_tiles) == (str(SWIGLU), "4")):
            continue
        body = text[text.index(f"\n{name}:"):]
        together = runs(body[:body.index(".Lfunc_end")])
        assert together and min(together) == (4 if int(epilogue) == SWIGLU else 2), (name, together)
