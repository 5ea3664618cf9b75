"""How the read-back cuts arrays into chunks and what it does without pinned
memory (tests/cpp/readback_plan_test.cpp, host only): 32 MB chunks, 1 MB chunks
when there is no memory for those, an error from the caller's allocator when
there is none at all."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_plan_covers_every_row(tmp_path):
    exe = str(tmp_path / "plan")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-fsanitize=address,undefined", "-I",
                    os.path.join(ROOT, "edegpredict-engine-rotary_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "readback_plan_test.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr[-2000:]
