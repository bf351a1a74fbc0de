"""A handle whose record buffers could not be allocated at one call (a sample dump or a surrogate
on a single-pass handle asks for them late) has all of them, or fails again, at the next
(tests/cxx/alloc_records.cpp: the driver's own function with an allocator that fails)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_failed_allocation_leaves_no_half_set(tmp_path):
    exe = str(tmp_path / "alloc_records")
    # the kernels' entry points that the driver's table names stay unresolved: none is called
    r = subprocess.run(["/opt/rocm/bin/hipcc", "--offload-host-only", "-std=c++17", "-O1",
                        "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "ppkmhd_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cxx", "alloc_records.cpp"), "-o", exe,
                        "-Wl,--unresolved-symbols=ignore-all"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
