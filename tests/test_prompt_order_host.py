"""The order in which a prompt's pieces are numbered (sru_layer.h), walked on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_piece_once_with_rows_and_behind_what_it_reads(tmp_path):
    """A piece without rows would have no barrier between the read of a workgroup's next number and its next write."""
    program = str(tmp_path / "prompt_order")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1", "-I" + os.path.join(rocm, "include"),
                           "-I" + os.path.join(ROOT, "sru_amd", "csrc"), os.path.join(ROOT, "tests", "prompt_order.cpp"), "-o", program])
    proc = subprocess.run([program], stdout=subprocess.PIPE, text=True, timeout=100)
    assert proc.returncode == 0, proc.stdout
