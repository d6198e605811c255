"""The tests' switches are no part of the public interface."""
import os
import re

from conftest import ROOT


def test_switches_are_exported_but_not_declared_publicly():
    from psvwave_amd import _lib
    declared = re.findall(r"^int (psv_\w+)\(", open(os.path.join(
        ROOT, "psvwave_amd", "csrc", "psv_testing.h")).read(), re.M)
    public = open(os.path.join(ROOT, "include", "psvwave.h")).read()
    assert declared
    for name in declared:
        assert hasattr(_lib.load(), name)
        assert name not in public and name not in _lib._SIGNATURES
