"""No exchange tag is 0: a claim word is a bare tag, so in zeroed scratch memory a launch with tag 0
would find every chunk claimed, nobody would compute the missing ones and the row would become NaN.
Host-only (tests/call_tag_check.cc)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "atex_amd", "csrc")


def test_tags_are_never_zero_and_differ_from_call_to_call(tmp_path):
    exe = str(tmp_path / "call_tag_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, os.path.join(HERE, "call_tag_check.cc"), "-o", exe],
                   check=True, capture_output=True, text=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stdout
