"""The varlen launches' work order (csrc/fa_common.h), run on the host: every workgroup gets an item of its own, also
where the L2 span times a head's items would pass 32 bits."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_varlen_work_order_is_a_permutation(tmp_path):
    import build_native
    if shutil.which(build_native.HIPCC) is None:
        pytest.skip("no hipcc")
    exe = tmp_path / "work_items_check"
    subprocess.run([build_native.HIPCC, *build_native.COMMON_FLAGS, "-w", f"-I{build_native.CSRC}",
                    str(ROOT / "tests" / "work_items_check.hip"), "-o", str(exe)], check=True, timeout=600)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert out.returncode == 0 and "wrong 0" in out.stdout, out.stdout + out.stderr
