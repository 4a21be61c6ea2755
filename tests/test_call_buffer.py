"""The memory that calls keep between them, over an allocator that refuses: a solve whose ray
pairs' parts find no memory keeps the tables' buffer instead of freeing and allocating it in
every call (tests/cpp/call_buffer.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_refused_parts_leave_the_buffer(tmp_path):
    exe = str(tmp_path / "call_buffer")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I" + os.path.join(ROOT, "magritte_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "call_buffer.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
