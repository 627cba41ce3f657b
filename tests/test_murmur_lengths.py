"""The hashes of cudf_amd/csrc/murmur.cuh, compiled for the host, at lengths around their blocks and just below 2^32 bytes, where a
32-bit place of a block wraps: there the loop over the blocks of the 64-bit hash never ended."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_hashes_of_any_length_against_the_published_algorithm(tmp_path):
    exe = tmp_path / "murmur_lengths"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-I" + os.path.join(ROOT, "cudf_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "murmur_lengths.cpp"), "-o", str(exe)])
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stdout
