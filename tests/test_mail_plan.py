"""The resident steps' messages on the host: tests/mail_plan.cpp built against
cppimpact_amd/csrc/host.cpp (plain C++, no GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_messages_reach_their_blocks_in_slot_order(tmp_path):
    exe = str(tmp_path / "mail_plan")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", os.path.join(ROOT, "tests", "mail_plan.cpp"),
                    os.path.join(ROOT, "cppimpact_amd", "csrc", "host.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True, timeout=300)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout + p.stderr
    assert p.stdout.count("ok ") == 7
