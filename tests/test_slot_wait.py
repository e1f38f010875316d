"""CPU check of the host's wait for a staged batch to be read
(fast-rbd-gradients_amd/csrc/slot_wait.hpp): it ends when the word arrives,
when the stream has failed and when the stream has drained without it."""
import os
import subprocess

import common


def test_wait_ends(tmp_path):
    exe = str(tmp_path / "slot_wait")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror",
                    os.path.join(common.HOSTCHECK, "slot_wait.cpp"), "-o", exe, "-lpthread"], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
