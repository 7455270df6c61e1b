"""Device memory on a failing allocation: the memory kept from dropped graphs
goes back and the allocation is tried again, whichever call makes it."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sstgraph_amd", "csrc")


def test_kept_blocks_over_a_small_device(tmp_path):
    """The allocator against a device of 64 MiB made of host functions."""
    exe = str(tmp_path / "device_memory_test")
    subprocess.run(
        ["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__",
         "-I/opt/rocm/include", f"-I{CSRC}", "-x", "c++",
         os.path.join(ROOT, "tests", "cpp", "device_memory_test.cpp"),
         os.path.join(CSRC, "device_memory.hip"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout


def test_every_allocation_can_take_the_kept_memory():
    """No file but the allocator's own calls hipMalloc."""
    for f in sorted(os.listdir(CSRC)):
        text = open(os.path.join(CSRC, f)).read()
        found = re.findall(r"\bhipMalloc(?:Async|Managed|Pitch)?\s*\(", text)
        assert f == "device_memory.hip" or not found, f
