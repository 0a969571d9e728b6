"""Which partial slices the reduce adds up: tests/c_abi/reduce_check.cpp, host arithmetic only."""
import os
import subprocess
import sys

BINARY = os.path.join(os.path.dirname(os.path.abspath(__file__)), "c_abi", "reduce_check.out")


def test_slices_of_the_reduce():
    if not os.path.isfile(BINARY):
        recipe = os.path.join(os.path.dirname(BINARY), "build.py")
        subprocess.run([sys.executable, "-c", f"import runpy; runpy.run_path({recipe!r})['build_reduce']()"], check=True,
                       timeout=300)
    run = subprocess.run([BINARY], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout.strip() == "all slices ok", (run.returncode, run.stdout)
