"""Registers of the built kernels, as the code object's metadata states them: kernels that must not
spill or keep anything in scratch memory."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CO = os.path.join(ROOT, "velo-core_amd", "velokv", "velokv_gfx950.co")
READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")

# int8-block stream-K kernels with RoPE: the spills that the 256 registers of two waves per SIMD leave
STREAM_K_SPILLS = {"g2_rope": 2, "g8_rope": 4, "gx_rope": 8, "g2_q0_rope": 4, "g4_q0_rope": 2, "g8_q0_rope": 6, "gx_q0_rope": 8}


@pytest.fixture(scope="module")
def kernels():
    """Kernel name -> (bytes of scratch memory a lane, spilled vector registers)."""
    if not (os.path.exists(CO) and os.path.exists(READELF)):
        pytest.skip("no built code object or no llvm-readelf")
    notes = subprocess.run([READELF, "--notes", CO], capture_output=True, text=True, check=True).stdout
    out, cur = {}, {}
    for line in notes.splitlines():
        m = re.match(r"\s+\.(symbol|private_segment_fixed_size|vgpr_spill_count|wavefront_size):\s+(\S+)", line)
        if m:
            cur[m.group(1)] = m.group(2)
            if m.group(1) == "wavefront_size":  # a kernel's last key
                out[cur["symbol"].removesuffix(".kd")] = (int(cur["private_segment_fixed_size"]), int(cur["vgpr_spill_count"]))
                cur = {}
    assert out
    return out


def test_stream_k_fold_spills(kernels):
    got = {n: v for n, v in kernels.items() if n.startswith("vk_decode_sk_kv3_")}
    assert len(got) == 24
    for n, (_, spills) in got.items():
        assert spills <= STREAM_K_SPILLS.get(n.removeprefix("vk_decode_sk_kv3_"), 0), n


@pytest.mark.parametrize("name", ["vk_decode_merge", "vk_decode_merge_sk"])
def test_merges_use_no_scratch_memory(kernels, name):
    assert kernels[name] == (0, 0)
