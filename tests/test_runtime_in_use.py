"""The tests run on the HIP runtime the library is linked against.  A package that brings a runtime
of its own under the same name (torch does) takes its place when it is imported first, for every
test of the process."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import importlib, os, sys
sys.path.insert(0, os.getcwd())
for f in sorted(os.listdir("tests")):
    if f.endswith(".py"):
        importlib.import_module("tests." + f[:-3])
import exanbody_amd
exanbody_amd.load()
print([l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l][0])
"""


def test_test_modules_bring_no_other_runtime():
    alone = "import exanbody_amd; exanbody_amd.load()\n" + PROGRAM[PROGRAM.index("print("):]
    runtimes = [subprocess.run([sys.executable, "-c", p], cwd=ROOT, capture_output=True, text=True, check=True).stdout.strip()
                for p in (alone, PROGRAM)]
    assert runtimes[0] and runtimes[1] == runtimes[0]
