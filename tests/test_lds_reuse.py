"""A kernel whose waves copy straight into LDS without a barrier in the loop has to await its own reads of a stage before the
copies that overwrite it.  Seen in the assembly that the source gives for gfx950: no GPU needed."""
import importlib.util
import os
import subprocess

import pytest

ROOT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "ojas-engine_amd")


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    spec = importlib.util.spec_from_file_location("ojas_build", os.path.join(ROOT, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc here")
    out = str(tmp_path_factory.mktemp("asm") / "gemm_xl.s")
    src, extra = build.FAMILIES["gemm_xl"]
    subprocess.check_call([build.HIPCC, f"--offload-arch={build.ARCH}", "--cuda-device-only", "-S", *build.DEVICE_FLAGS, *extra,
                           "-o", out, os.path.join(build.KERNELS, src)])
    return open(out).read()


@pytest.mark.parametrize("kernel", ["gemm_mm_q4kl_bdk", "gemm_mm_q4kl_bdk_sk"])
def test_reads_awaited_before_copies(assembly, kernel):
    body = assembly.split(f"\n{kernel}:", 1)[1].split("s_endpgm", 1)[0]
    pending, copies = False, 0
    for line in (t.strip() for t in body.splitlines()):
        if line.startswith("ds_read"):
            pending = True
        elif line.startswith("s_waitcnt") and "lgkmcnt(0)" in line:
            pending = False
        elif line.startswith("global_load_lds"):
            copies += 1
            assert not pending, f"copy {copies} may overwrite LDS that a read has not left yet"
    assert copies > 64                                       # the loop's four unrolled steps were seen
