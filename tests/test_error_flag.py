"""The words that kernels report errors in: reused after a wait that succeeded,
never after one that failed (a late store would reach another call)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_a_word_is_passed_on_only_after_its_wait(tmp_path):
    exe = tmp_path / "error_flag"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(HERE, "..", "rustyneedle_amd", "csrc"),
                    os.path.join(HERE, "c", "error_flag.cpp"), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
