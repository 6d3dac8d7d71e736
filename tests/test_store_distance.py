"""A 12- or 16-byte store reads its data registers after it has been issued: a VALU instruction right behind it that writes one of
them can reach memory in its place.  hipcc keeps the distance for most stores, but not for buffer stores with a scalar offset;
those go through buffer_store16 (gemm_internal.h).  Checked on the compiler's listing of every source.  Needs hipcc, no GPU."""
import re
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "cosmos-rl_amd"))
from cosmos_rl_amd import _build  # noqa: E402

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(), reason="needs hipcc")

_REGS = re.compile(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b")
_STORE = re.compile(r"(buffer|global|flat)_store_dwordx[34]\s+(.*)")


def _regs(operand):
    out = set()
    for m in _REGS.finditer(operand):
        out |= set(range(int(m.group(1)), int(m.group(2)) + 1)) if m.group(1) else {int(m.group(3))}
    return out


def overwritten(lines):
    """(function, store, instruction) where the instruction right behind a wide store writes one of its data registers."""
    found, function, last = [], "", None
    for line in lines:
        label = re.match(r"(_Z\w+):", line)
        if label:
            function = label.group(1)
        text = line.split(";")[0].strip()
        if not text or text[0] in "._" or text.endswith(":"):
            continue
        if last and text.startswith("v_") and not text.startswith("v_cmp"):
            if _regs(text.split(None, 1)[1].split(",")[0]) & last[1]:
                found.append((function, last[0], text))
        m = _STORE.match(text)
        last = (text, _regs(m.group(2).split(",")[0 if m.group(1) == "buffer" else 1])) if m else None
    return found


def _listing(src):
    cmd = [_build.hipcc(), *_build.HIPCC_FLAGS, *_build.EXTRA_FLAGS.get(src, []), f"-I{_build.INCLUDE_DIR}", f"-I{_build.CSRC_DIR}",
           "--cuda-device-only", "-S", str(_build.CSRC_DIR / src), "-o", "-"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return res.stdout.splitlines()


def test_the_check_sees_what_it_looks_for():
    store = "buffer_store_dwordx4 v[4:7], v8, s[0:3], s4 offen"
    assert overwritten([store, "v_and_b32_e32 v5, 8, v9"]) and overwritten([store, "; comment", "v_mfma_f32_16x16x128_f8f6f4 v[6:9], v[0:3], v[0:3], 0"])
    assert not overwritten([store, "s_nop 1", "v_and_b32_e32 v5, 8, v9"]) and not overwritten([store, "v_and_b32_e32 v8, 8, v5"])
    assert overwritten(["global_store_dwordx4 v[0:1], v[4:7], off", "v_mov_b32_e32 v4, 0"]) and not overwritten(["global_store_dwordx4 v[0:1], v[4:7], off", "v_mov_b32_e32 v0, 0"])


def test_no_store_is_overtaken():
    with ThreadPoolExecutor(max_workers=8) as pool:
        found = {src: overwritten(lines) for src, lines in zip(_build.SOURCES, pool.map(_listing, _build.SOURCES))}
    assert not any(found.values()), {src: hits[:3] for src, hits in found.items() if hits}


def test_experts_kernel_stays_in_registers():
    """gemm_experts_kernel counts its vector-memory operations by hand: a spilled register would be one more of them."""
    lines = _listing("gemm_experts.hip")
    assert sum(line.strip().startswith("buffer_load_dwordx4") and " lds" in line for line in lines) > 0
    assert not any(line.strip().startswith("scratch_") for line in lines)
