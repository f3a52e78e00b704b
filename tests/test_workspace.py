"""The device workspace's growth rules (eb_workspace.h), on the host with a pretend memory: what
holds the least a call can do with is kept when memory is refused, a refusal is not asked for again
by the next calls, and graphs keep the buffers they were captured with."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_growth_rules(tmp_path):
    exe = str(tmp_path / "rules")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    "-I", os.path.join(ROOT, "eyebrowse_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "workspace_rules.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
