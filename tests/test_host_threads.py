"""Host work where the system starts no more threads."""
import os
import subprocess

import onegraph_amd as og

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_work_runs_on_the_threads_there_are(tmp_path):
    og.lib()  # the library is built
    exe, libdir = str(tmp_path / "threads"), os.path.dirname(og.LIB_PATH)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-o", exe, os.path.join(HERE, "integration", "threads.cpp"),
                        "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(libdir, "csrc"), "-L" + libdir,
                        "-lonegraph", "-Wl,-rpath," + libdir, "-ldl", "-lpthread"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout + r.stderr)
