"""What pj_api.cpp decides by itself (line blocks, scratch contents), checked on
the host with the HIP calls and the launches replaced
(tests/cpp/api_state_check.cpp): no GPU and no kernel takes part."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "micronaut3-bug_amd", "csrc")


def test_api_state(tmp_path):
    exe = str(tmp_path / "api_state_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    os.path.join(ROOT, "tests", "cpp", "api_state_check.cpp"), os.path.join(CSRC, "pj_api.cpp"),
                    "-pthread", "-o", exe], check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "api state checks passed" in r.stdout
