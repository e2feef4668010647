"""Where the dynamic LDS of decode attention begins.  Its merge reads two neighbouring floats at a time, so the area has to begin on 8 bytes; it lies
behind the kernel's own static LDS, whose size the compiler states in the listing and rounds up to what the area is declared to need."""
import os
import re
import subprocess

import pytest

from fllm_amd.kernels import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_decode_attention_reads_pairs_from_an_area_that_begins_on_16_bytes(tmp_path):
    try:
        hipcc = build._hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    listing = tmp_path / "attention.s"
    flags = [f for f in build.HIPCC_FLAGS if f != "-O3"] + ["-O1", "--cuda-device-only", "-S"]
    run = subprocess.run([hipcc, *flags, os.path.join(ROOT, "fllm_amd", "csrc", "attention_mfma.hip"), "-o", str(listing)], capture_output=True, text=True,
                         timeout=300)
    assert run.returncode == 0, run.stderr
    sizes = {name: int(size) for size, name in re.findall(r"\.group_segment_fixed_size: (\d+).*?\.name:\s+(\S+)", listing.read_text(), re.S)}
    decode = {name: size for name, size in sizes.items() if "attn_decode_kernel" in name}
    assert len(decode) == 9                                   # three head sizes, three page sizes
    assert all(size % 16 == 0 for size in decode.values()), decode
