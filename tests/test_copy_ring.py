"""The ring that carries large results to the caller's buffers, on the CPU, with
a transfer engine that fails or refuses at a chosen chunk: a buffer gets bytes
of its own copy and nothing else, in particular not what the ring's chunks held
before, and every copy ends.  And the rule by which the ring is made at all."""

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_copy_ring(tmp_path):
    exe = str(tmp_path / "copy_ring")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I",
                    os.path.join(HERE, "..", "gdistger-re_amd", "csrc"), os.path.join(HERE, "copy_ring_main.cpp"),
                    "-o", exe, "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert r.stdout.count("ok ") == 18
