"""The PerBit retrieve's ordering between streams and its error exits, on the
CPU: tests/cpp/test_retrieve_streams.cpp runs the library over HIP calls of its
own."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.mark.parametrize("what", ["maxima", "errors"])
def test_perbit_retrieve_streams(tmp_path, what):
    lib = os.path.join(ROOT, "prodm_amd")
    exe = str(tmp_path / "test_retrieve_streams")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-rdynamic",
                    f"-I{ROOT}/include", f"-I{ROCM}/include", os.path.join(ROOT, "tests", "cpp", "test_retrieve_streams.cpp"),
                    "-o", exe, f"-L{lib}", "-lprodm_mdr", f"-Wl,-rpath,{lib}", f"-L{ROCM}/lib", "-lamdhip64",
                    f"-Wl,-rpath,{ROCM}/lib", "-pthread"], check=True)
    r = subprocess.run([exe, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "PASSED" in r.stdout, r.stdout + r.stderr
