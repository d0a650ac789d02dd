"""The resident loop's wait for the other blocks' words, run on the CPU: a word
missing on any line ends the wait for the whole wave, not only for the lanes
that poll it."""
import os
import subprocess

from conftest import ROOT


def test_a_missing_word_on_any_line_ends_the_wait(tmp_path):
    exe = str(tmp_path / "exchange_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wno-unknown-pragmas",
                    os.path.join(ROOT, "tests", "cpp", "exchange_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
