"""The plan-memory pool against a device with little memory (host only, over
fake allocation calls)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_idle_memory_is_given_back(tmp_path):
    csrc, cpp = os.path.join(ROOT, "superman_amd", "csrc"), os.path.join(ROOT, "tests", "cpp")
    out = str(tmp_path / "workspace")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(cpp, "fake_hip"), "-I" + os.path.join(ROOT, "include"),
                    "-I" + csrc, os.path.join(cpp, "workspace_main.cpp"), os.path.join(csrc, "workspace.cpp"), "-lpthread",
                    "-o", out], check=True)
    p = subprocess.run([out], capture_output=True, text=True)
    assert p.returncode == 0 and p.stdout == "ok\n", p.stdout
