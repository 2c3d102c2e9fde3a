"""What of the process environment reaches the compiled library."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bmtk_amd", "csrc")


def test_kernels_are_steered_by_no_variable_but_the_documented_one():
    """A plan read from a variable any shell may hold gives wrong sums, or a division by zero, without an error."""
    names = {}
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        with open(path) as f:
            for argument in re.findall(r"getenv\s*\(\s*([^)]*?)\s*\)", f.read()):
                names.setdefault(argument, []).append(os.path.basename(path))
    assert names == {'"BMTK_AMD_PLAIN_LAUNCH"': ["resident.hip", "resident_batch.hip"]}
