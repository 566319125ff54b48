"""Which workgroup of a grid of several matrices works on which tile, on the CPU (tests/tiles_on_host.hip)."""
import importlib.util
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tiles_on_host(tmp_path):
    spec = importlib.util.spec_from_file_location("aq_build", os.path.join(ROOT, "go-inference_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    prog = str(tmp_path / "tiles_on_host")
    build.run([build.hipcc()] + build.COMMON + build.HIPFLAGS + ["--cuda-host-only", "-I", build.CSRC, "-o", prog, os.path.join(ROOT, "tests", "tiles_on_host.hip")])
    r = subprocess.run([prog], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
