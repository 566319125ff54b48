"""The order of the scratch block's users across streams, its growth and its refusals, on the CPU: csrc/aq_workspace.hip
compiled with a HIP runtime that only writes down what it is asked (tests/workspace_on_host.hip)."""
import importlib.util
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_workspace_on_host(tmp_path):
    spec = importlib.util.spec_from_file_location("aq_build", os.path.join(ROOT, "go-inference_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    prog = str(tmp_path / "workspace_on_host")
    sources = [os.path.join(ROOT, "tests", "workspace_on_host.hip"), os.path.join(build.CSRC, "aq_workspace.hip")]
    build.run([build.hipcc()] + build.COMMON + build.HIPFLAGS + ["--cuda-host-only", "-I", build.CSRC, "-o", prog] + sources)
    r = subprocess.run([prog], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
