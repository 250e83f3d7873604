"""The K-major 256x256 kernel's DMAs into LDS, in the assembly of its device
pass (CPU only): none carries a scalar offset.  What a DMA may read is then
decided by its lane offset and its descriptor's record count alone, also where
the stage stream runs past an operand's end with no records left (a K of one
stage, no next tile)."""
import re
import subprocess
import sys
from pathlib import Path

REPO = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(REPO / "moe-overlap_amd"))
import build_native  # noqa: E402


def test_stage_dmas_have_no_scalar_offset(tmp_path):
    out = tmp_path / "kmajor.s"
    subprocess.run([build_native._hipcc(), *build_native.HIP_FLAGS, "--cuda-device-only", "-S",
                    str(build_native.CSRC / "mgg_gemm_kmajor.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    dmas = re.findall(r"^\s*buffer_load_dwordx4 v\d+, s\[\d+:\d+\], (\S+) offen.* lds",
                      out.read_text(), re.M)
    assert len(dmas) >= 6 * 48  # six instances: two prologue stages and the body's sixteen
    assert set(dmas) == {"0"}
