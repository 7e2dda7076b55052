"""The LDS ring of the head-dim-64 prefill kernel: in the code built for gfx950, every barrier after which a ring slot
is refilled comes right behind a wait for all of the wave's LDS reads.  Compiles the kernel to assembly (no GPU)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
FORMS = ("kPpDense, false", "kPpVarlen, false", "kPpVarlen, true", "kPpCache, false", "kPpCache, true")


def test_lds_reads_return_before_the_ring_barriers(tmp_path):
    import build_native
    if shutil.which(build_native.HIPCC) is None:
        pytest.skip("no hipcc")
    src = tmp_path / "d64.hip"
    src.write_text(f'#include "{ROOT}/flash-attn-triton_amd/csrc/fa_prefill_d64.h"\nnamespace fa {{\n' + "".join(
        f"template __global__ void prefill_d64_kernel<F16, {f}>(const FwdParams);\n" for f in FORMS) + "}\n")
    asm = tmp_path / "d64.s"
    subprocess.run([build_native.HIPCC, *build_native.COMMON_FLAGS, "-w", "-S", "--cuda-device-only", str(src), "-o",
                    str(asm)], check=True, timeout=600)
    code = [s for s in (line.split(";")[0].strip() for line in asm.read_text().splitlines())
            if s and not s.startswith(".") and not s.endswith(":")]
    before = [code[i - 1] for i, s in enumerate(code) if s.startswith("s_barrier")]
    # per form: the ring steps (four places in the source), then the barrier ahead of the output staging
    assert len(before) == 5 * len(FORMS)
    ring = [s for i, s in enumerate(before) if i % 5 != 4]
    assert all(re.search(r"s_waitcnt\b.*\blgkmcnt\(0\)", s) for s in ring), ring
