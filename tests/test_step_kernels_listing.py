"""What the compiled kernels of decode steps and prompts are held to where nothing in their results shows it: loads that wait for nothing between
them, registers that leave a compute unit its waves."""
import os
import re
import subprocess

import pytest

from fllm_amd.kernels import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def kernels(source, pattern, tmp_path):
    """(name, text up to the next kernel, the pattern's groups) of every kernel of a source whose name the pattern matches."""
    try:
        hipcc = build._hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    listing = tmp_path / "listing.s"
    run = subprocess.run([hipcc, *build.HIPCC_FLAGS, "--cuda-device-only", "-S", os.path.join(ROOT, "fllm_amd", "csrc", source), "-o", str(listing)],
                         capture_output=True, text=True, timeout=600)
    assert run.returncode == 0, run.stderr
    parts = re.split(r"^(_Z\w+):.*$", listing.read_text(), flags=re.M)
    found = [(name, text, re.search(pattern, name)) for name, text in zip(parts[1::2], parts[2::2])]
    return [(name, text, match.groups()) for name, text, match in found if match]


def longest_run(text):
    """The most 16-bit loads in a row without a wait for loads between them."""
    longest = run = 0
    for line in text.splitlines():
        line = line.strip()
        if line.startswith("global_load_ushort"):
            run += 1
            longest = max(longest, run)
        elif line.startswith("s_waitcnt") and "vmcnt" in line:
            run = 0
    return longest


@pytest.mark.parametrize("source,pattern,instances", [("conv_store.hip", r"20conv_qkv_step_kernelIDF16bLi(\d+)E", 4),
                                                      ("sequence_ops.hip", r"22norm_short_conv_kernelIDF16b", 4),
                                                      ("layer_norms.hip", r"21layernorm_conv_kernelIDF16b", 4)])
def test_entries_of_the_state_are_asked_for_together(tmp_path, source, pattern, instances):
    """bfloat16 entries, three of every piece of a row that a wave has: behind a question each they are awaited one by one."""
    found = kernels(source, pattern, tmp_path)
    assert len(found) == instances
    for name, text, groups in found:
        want = 3 * int(groups[0]) if groups else 3
        assert longest_run(text) >= want, name


# waves a SIMD of prompts' tiles of windows with pooled blocks, (key lanes / 32, value lanes / 16): where asking for a block's keys and values at
# once costs one of them
TILE_WAVES = {(2, 6): 3, (3, 2): 4, (3, 4): 3, (3, 6): 3, (4, 2): 4, (4, 4): 3}


def test_waves_of_prompts_with_pooled_blocks(tmp_path):
    found = kernels("mixer_variants_mfma.hip", r"17mixer_tile_kernelILi(\d)ELi(\d)ELi0ELb[01]ELb0E", tmp_path)
    assert len(found) == 32
    for name, text, (kd, vt) in found:
        waves = int(re.search(r"^; Occupancy: (\d+)", text, re.M).group(1))
        assert waves >= TILE_WAVES.get((int(kd), int(vt)), 2), (name, waves)
