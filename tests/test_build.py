"""What the documented build lines need: the library hipcc alone, the Python module a target of its own."""
import os
import re
import subprocess

from conftest import ROOT


def planned(*args):
    r = subprocess.run(["make", "-C", os.path.join(ROOT, "my-nn-engine_amd", "csrc"), "-B", "-n", "--no-print-directory", *args], capture_output=True, text=True,
                       timeout=60)
    return r.returncode, r.stdout


def test_the_library_is_built_without_python():
    rc, commands = planned("PYTHON=/bin/false", "CXX=/bin/false")
    assert rc == 0 and "libmynn_hip.so" in commands
    assert "_host_ops" not in commands and "/bin/false" not in commands


def test_the_python_module_is_a_target_of_its_own():
    rc, commands = planned("host_ops")
    assert rc == 0 and "_host_ops.so" in commands and "hipcc" not in commands


def test_every_launch_role_of_the_benchmark_is_a_kernel_of_the_library():
    """(rocprofv3's figures of a launch are found by the pattern of its kernel's name)"""
    import sys

    sys.path.insert(0, ROOT)
    import bench

    lib = open(os.path.join(ROOT, "my-nn-engine_amd", "lib", "libmynn_hip.so"), "rb").read()
    assert len(bench.ROLE_PATTERNS) >= 13
    assert not [role for role, pattern in bench.ROLE_PATTERNS.items() if not re.search(pattern.encode(), lib)]
