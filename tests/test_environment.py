"""What of the process environment reaches the compiled library."""
import glob
import os
import re
import types

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bmtk_amd", "csrc")


def test_kernels_are_steered_by_no_variable_but_the_documented_one():
    """A plan read from a variable any shell may hold gives wrong sums, or a division by zero, without an error."""
    names = {}
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        with open(path) as f:
            for argument in re.findall(r"getenv\s*\(\s*([^)]*?)\s*\)", f.read()):
                names.setdefault(argument, []).append(os.path.basename(path))
    assert names == {'"BMTK_AMD_PLAIN_LAUNCH"': ["resident.hip", "resident_batch.hip"]}


@pytest.mark.parametrize("compiler", ["false", "/nonexistent/compiler"])
def test_pointer_checks_that_cannot_be_compiled_are_a_warning(monkeypatch, tmp_path, compiler):
    from bmtk_amd.csrc import build
    stale = tmp_path / os.path.basename(build.PTR)
    stale.write_bytes(b"of another build")
    monkeypatch.setattr(build, "PTR", str(stale))
    monkeypatch.setenv("CXX", compiler)
    with pytest.warns(UserWarning, match="ptr.cpp was not compiled"):
        assert build.build_ptr() is None
    assert not stale.exists()


def test_pointer_checks_of_another_torch_are_not_used(monkeypatch):
    import torch

    import bmtk_amd
    from bmtk_amd import ops

    def general():
        pass
    given = []
    for built_for, used in ((str(torch.__version__), True), ("0.0", False), (None, False)):
        fake = types.SimpleNamespace(ptr=object(), set_general=given.append)
        if built_for is not None:
            fake.built_for = built_for
        monkeypatch.setattr(bmtk_amd, "_ptr", fake, raising=False)
        assert ops._native(general) is (fake.ptr if used else general)
    assert given == [general]
