"""The number of the resident steps' messages: tests/mail_count.cpp built against
cppimpact_amd/csrc/host.cpp (plain C++, no GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_messages_are_counted_past_32_bits(tmp_path):
    exe = str(tmp_path / "mail_count")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", os.path.join(ROOT, "tests", "mail_count.cpp"),
                    os.path.join(ROOT, "cppimpact_amd", "csrc", "host.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True, timeout=300)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout + p.stderr
