"""Pointers that the lanes treat as global memory (csrc/de_common.h, global_ptr)
are never addresses of a lane's own stack: the event lanes of every kind of method
run on the host with each such pointer checked, through the integration, the root
pass over their brackets and the bookkeeping pass."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_no_lane_reads_its_stack_as_global_memory():
    subprocess.check_call(["make", "-s", "-C", os.path.join(HERE, "cpp"), "_build/global_ptr_check"])
    out = subprocess.run([os.path.join(HERE, "cpp", "_build", "global_ptr_check")],
                         capture_output=True, timeout=300, text=True)
    assert out.returncode == 0, out.stdout[-4000:]
