"""How the SpMM goes about the panels of a weight, on the CPU (tests/cpp/test_spmm_plan.cc, built by __graft_entry__.build())."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_spmm_plan():
    exe = os.path.join(ROOT, "tests", "cpp", "bin", "test_spmm_plan")
    assert os.path.exists(exe), "%s is not built: run __graft_entry__.build()" % exe
    p = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert p.returncode == 0 and "ALL PASSED" in p.stdout, p.stdout[-4000:]
