"""The host build of the library (tests/emu) is rebuilt when any of its sources changes: a header that is
missing from its list would leave the checks of the kernels on old code."""
import glob
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(__file__), "emu"))


def test_every_source_and_header_is_a_dependency():
    import build

    present = {f for pat in ("*.hip", "*.h") for f in glob.glob(os.path.join(build.CSRC, pat))}
    present.add(os.path.join(build.ROOT, "include", "jaxfluids_amd.h"))
    assert len(present) > len(build.SOURCES)
    assert present - {os.path.abspath(d) for d in build.DEPS} == set()
