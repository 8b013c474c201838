"""The wait state between a write of m0 and the LDS transfer that reads it: the
hardware needs one, and inside an asm string the compiler inserts none. Read off the
compiled kernels, since a missing one shows on the GPU only now and then."""

import os
import shutil
import subprocess

import pytest

from opsagent_amd.ops import build

WITH_TRANSFERS = [s for s in build.SOURCES + build.MIXER_SOURCES
                  if "lds_transfer16" in open(os.path.join(build.CSRC, s)).read()
                  or "load_lds" in open(os.path.join(build.CSRC, s)).read()]


def test_files():
    assert {"attention_prefill.hip", "fp8_moe.hip", "ring_gemm.hip", "tile_gemm.hip"} <= set(WITH_TRANSFERS)


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
@pytest.mark.parametrize("fname", WITH_TRANSFERS)
def test_wait_state_after_m0(fname, tmp_path):
    out = tmp_path / "k.s"
    subprocess.run([build.HIPCC, f"--offload-arch={build.ARCH}", "-O3", "-std=c++17",
                    *build.HIP_FLAGS, "--cuda-device-only", "-S",
                    os.path.join(build.CSRC, fname), "-o", str(out)],
                   check=True, capture_output=True, timeout=300)
    code = [ln.split(";")[0].split("//")[0].strip() for ln in out.read_text().splitlines()]
    code = [ln for ln in code if ln and not ln.startswith(".") and not ln.endswith(":")]
    loads = [i for i, ln in enumerate(code) if ln.startswith("global_load_lds")]
    assert loads
    for i in loads:
        assert code[i - 1].split()[0] == "s_nop" and code[i - 2].startswith("s_mov_b32 m0,"), code[i - 2:i + 1]
    # m0 is on no clobber list: nothing but the transfers may use it
    writes = [ln for ln in code if "m0" in ln.replace(",", " ").split()]
    assert len(writes) == len(loads), writes
