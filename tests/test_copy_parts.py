"""The threaded host copy of body state transfers (physkit_amd/csrc/pk_copy.hpp): whole, and no
end of the process, where a thread of its team cannot be allocated."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copy_is_whole_when_threads_cannot_start(tmp_path):
    exe = str(tmp_path / "copy_parts_check")
    subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-Wall", "-Wextra", "-pthread",
                    "-I", os.path.join(ROOT, "physkit_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "copy_parts_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "copy_parts ok" in r.stdout
