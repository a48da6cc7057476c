"""The host layer's library and the C++ programs of the tests: compiled against LibNTC's own public header where that tree
lies (rtxntc-library_amd/host/Makefile, tests/Makefile), so not on every machine."""
import os

import pytest

HEADER = os.path.join(os.environ.get("NTC_REFERENCE", "/root/reference"), "include", "libntc", "ntc.h")


def built(path):
    """`path`, if it is there.  A test fails where it could have been built, and is skipped where it could not."""
    if not os.path.exists(path):
        if os.path.exists(HEADER):
            pytest.fail(f"{path} is not built; run __graft_entry__.build()")
        pytest.skip(f"{os.path.basename(path)} is compiled against LibNTC's include/libntc/ntc.h, which this machine does not have")
    return path
