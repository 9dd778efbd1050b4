"""The choice of workgroups per subdomain where a work vector does not fit (CPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_choice_equals_asking_outright(tmp_path):
    src = os.path.join(ROOT, "doug_amd", "csrc")
    exe = str(tmp_path / "front_groups_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", src, "-o", exe,
                    os.path.join(ROOT, "tests", "front_groups_check.cpp"), os.path.join(src, "doug_fronts.cpp"),
                    os.path.join(src, "doug_setup.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
