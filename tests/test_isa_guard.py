"""What the compiler makes of libmgg's device code, read from the assembly of
its device pass (CPU only).

Device code writes through vector stores alone: every scalar instruction is
one that computes, branches or waits, or a scalar memory instruction that only
reads or invalidates.  The list names what is allowed, so an instruction
nobody thought of fails as well.

The K-major 256x256 kernel's DMAs into LDS carry no scalar offset: what one
may read is decided by its lane offset and its descriptor's record count
alone, also where the stage stream runs past an operand's end with no records
left (a K of one stage, no next tile)."""
import functools
import re
import subprocess
import sys
import tempfile
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(REPO / "moe-overlap_amd"))
import build_native  # noqa: E402

READS = r"s_(load|buffer_load)_dword(x\d+)?|s_mem(real)?time|s_dcache_inv(_vol)?"
COMPUTES = (r"s_(mov|movk|cmov|cmovk|not|wqm|brev|abs|sext|getpc|setpc|swappc|bitset[01]|quadmask"
            r"|bcnt[01]|ff[01]|flbit|add|addc|addk|sub|subb|mul|mulk|mul_hi|min|max|cselect"
            r"|and|or|xor|nand|nor|xnor|andn2|orn2|lshl|lshr|ashr|lshl[1-4]_add|bfm|bfe|absdiff"
            r"|bitcmp[01]|cmp_\w+|cmpk_\w+|pack_\w+|(and|or|xor|andn1|andn2|orn1|orn2|nand|nor|xnor)_saveexec)"
            r"(_[biu](16|32|64))*(_i(8|16))?")
CONTROLS = r"s_(waitcnt|nop|barrier|branch|cbranch_\w+|endpgm|sleep|setprio|sendmsg|trap|getreg_b32|setreg\w*)"
ALLOWED = re.compile(f"({READS}|{COMPUTES}|{CONTROLS})$")


@functools.lru_cache(maxsize=None)
def assembly(src):
    with tempfile.TemporaryDirectory() as tmp:
        out = Path(tmp) / "device.s"
        subprocess.run([build_native._hipcc(), *build_native.HIP_FLAGS, "--cuda-device-only", "-S",
                        str(build_native.CSRC / src), "-o", str(out)], check=True, capture_output=True)
        return out.read_text()


@pytest.mark.parametrize("src", build_native.SOURCES)
def test_scalar_instructions_compute_or_read(src):
    used = set(re.findall(r"^\s+(s_\w+)", assembly(src), re.M))
    assert "s_endpgm" in used or "amdhsa_kernel" not in assembly(src)  # (a source without kernels)
    assert [op for op in sorted(used) if not ALLOWED.match(op)] == []


def test_the_list_allows_no_scalar_memory_write():
    """Names made of the memory verbs and every suffix the list knows."""
    for verb in ("store", "atomic", "scratch", "dcache", "atc", "memwrite"):
        for rest in ("", "_dword", "_dwordx4", "_add", "_swap_x2", "_wbinvl", "_probe", "_b32", "_i32"):
            for prefix in ("s_", "s_buffer_"):
                assert not ALLOWED.match(prefix + verb + rest)


def test_stage_dmas_have_no_scalar_offset():
    dmas = re.findall(r"^\s*buffer_load_dwordx4 v\d+, s\[\d+:\d+\], (\S+) offen.* lds",
                      assembly("mgg_gemm_kmajor.hip"), re.M)
    assert len(dmas) >= 6 * 48  # six instances: two prologue stages and the body's sixteen
    assert set(dmas) == {"0"}
