"""The order of a call's launches and its use of scratch, on the CPU: the built library with a HIP runtime that only writes down
what it is asked (tests/calls_on_host.cc)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "go-inference_amd", "libaq_mi355.so")


def test_calls_on_host(tmp_path):
    prog = str(tmp_path / "calls_on_host")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cmd = ["g++", "-O1", "-std=c++17", "-Wall", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "go-inference_amd", "csrc"), "-I", os.path.join(rocm, "include"),
           os.path.join(ROOT, "tests", "calls_on_host.cc"), "-o", prog, LIB, "-Wl,-rpath," + os.path.dirname(LIB), "-Wl,-rpath-link," + os.path.join(rocm, "lib"), "-lpthread", "-ldl"]
    built = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert built.returncode == 0, built.stdout
    r = subprocess.run([prog], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout[-4000:]
