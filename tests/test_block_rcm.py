"""Reverse Cuthill-McKee orders shared by subdomains of one local graph (CPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_shared_orders(tmp_path):
    src = os.path.join(ROOT, "doug_amd", "csrc")
    exe = str(tmp_path / "rcm_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", src, "-o", exe,
                    os.path.join(ROOT, "tests", "rcm_check.cpp"), os.path.join(src, "doug_setup.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
