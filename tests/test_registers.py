"""Vector registers of the few-token kernels, as the built code object states them: no GPU needed.  A SIMD holds 512 per lane, so
two workgroups of eight waves share a CU up to 128 of them, and three waves a SIMD up to 168."""
import os
import re
import subprocess

import pytest

ROOT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "ojas-engine_amd")
FORMATS = ["q8_0", "f16", "iq4nl", "iq4xs", "q40", "q41", "q50", "q51", "mxfp4", "q2k", "q3k"]


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    built, llvm = os.path.join(ROOT, "hsaco", "gemm.hsaco"), "/opt/rocm/llvm/bin/"
    if not os.path.exists(built) or not os.path.exists(llvm + "clang-offload-bundler"):
        pytest.skip("no built code object, or no tool to read it")
    co = str(tmp_path_factory.mktemp("co") / "gemm.co")
    subprocess.check_call([llvm + "clang-offload-bundler", "--type=o", "--unbundle", "--input=" + built,
                           "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--output=" + co])
    notes = subprocess.check_output([llvm + "llvm-readelf", "--notes", co], text=True)
    found = {}
    for body in notes.split("- .agpr_count:")[1:]:
        value = lambda key: re.search(r"\.%s:\s+(\S+)" % key, body).group(1)
        found[value("name")] = (int(value("vgpr_count")), int(value("vgpr_spill_count")))
    return found


@pytest.mark.parametrize("fmt", FORMATS)
def test_no_few_token_kernel_spills(registers, fmt):
    names = [n for n in registers if n.startswith("gemm_few_%s_" % fmt)]
    assert len(names) >= 5 and not [n for n in names if registers[n][1]]


@pytest.mark.parametrize("fmt", [f for f in FORMATS if f != "q3k"])      # (Q3_K: 153 with its block's eight loads)
def test_two_workgroups_of_eight_waves_share_a_cu(registers, fmt):
    assert registers["gemm_few_%s_r4_t2" % fmt][0] <= 128


@pytest.mark.parametrize("fmt", ["q8_0", "iq4nl", "iq4xs"])
def test_grouped_expert_form_keeps_three_waves_a_simd(registers, fmt):
    assert registers["moe_few_%s" % fmt][0] <= 168 and not registers["moe_few_%s" % fmt][1]
