"""The staged transfers (csrc/upf_stage.h) on the host, against a stand-in for
the runtime: every byte arrives, also when threads cannot start, pinned memory
is refused or events are."""
import os
import subprocess

import unifiedparticleframeworkcuda_amd as upf

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "stage")


def test_transfers_without_threads_pinned_memory_or_events(tmp_path):
    exe = str(tmp_path / "stage_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-pthread", "-I" + HERE,
                           "-I" + os.path.join(os.path.dirname(upf.__file__), "csrc"),
                           os.path.join(HERE, "stage_check.cpp"), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[-300:] + r.stderr[-300:]
