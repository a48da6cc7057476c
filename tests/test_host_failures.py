"""Host code of the C ABI (csrc/ntc_hip_api.cpp) where the runtime fails or is late, on the CPU: the file's object linked
with a runtime on host memory (fake_hip_runtime.cpp) whose calls can be made to fail and whose launches stay outstanding
until they are waited for."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rtxntc-library_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not found")
    out = tmp_path_factory.mktemp("fake")
    flags = ["-O1", "-std=c++17", "-fPIC", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-x", "hip"]
    sources = [os.path.join(CSRC, "ntc_hip_api.cpp"), os.path.join(HERE, "fake_hip_runtime.cpp")]
    objects = [str(out / f"{i}.o") for i in range(2)]
    builds = [subprocess.Popen([HIPCC, *flags, "-c", s, "-o", o], stderr=subprocess.PIPE) for s, o in zip(sources, objects)]
    for b in builds:
        text = b.communicate(timeout=300)[1]
        assert b.returncode == 0, text.decode()
    path = str(out / "libntc_fake.so")
    subprocess.run(["g++", "-shared", "-Wl,-z,defs", "-Wl,-Bsymbolic", "-o", path, *objects], check=True, timeout=300)
    return path


@pytest.fixture
def fake(ntc, library):
    """The library with its exports typed and a context made, both gone after the test."""
    lib = C.CDLL(library)
    for name, restype, argtypes in ntc.abi.EXPORTS:
        getattr(lib, name).restype, getattr(lib, name).argtypes = restype, argtypes
    lib.fake_reset()
    handle = C.c_void_p()
    assert lib.ntc_hip_create(0, C.byref(handle)) == 0, lib.ntc_hip_last_error()
    lib.context = handle
    yield lib
    lib.ntc_hip_destroy(handle)
    assert lib.fake_allocations() == 0


def test_tables_of_a_device_are_complete_before_its_first_context(fake):
    """Contexts have streams of their own: nothing orders one's first launch behind tables that another's call fills."""
    fake.fake_launches.restype = C.c_char_p
    first = fake.fake_launches().decode().split()[:3]
    assert sorted(first[:2]) == ["launch_color_tables", "launch_transfer_tables"] and first[2] == "complete"


def test_contexts_leave_the_null_stream_alone(fake):
    """Work on the null stream waits for every blocking stream of the device, and they for it."""
    handle = C.c_void_p()
    assert fake.ntc_hip_create(0, C.byref(handle)) == 0
    fake.ntc_hip_destroy(handle)
    assert fake.fake_null_stream_uses() == 0                            # since the library was loaded


def loss(lib, width=64, height=64, mask=-1):
    """-> (return code, the 16 values)"""
    a, b = np.zeros(width * height * 16, dtype=np.float16), np.zeros(width * height * 16, dtype=np.float16)
    out = (C.c_float * 16)()
    code = lib.ntc_hip_ctx_image_loss(lib.context, a.ctypes.data, b.ctypes.data, a.nbytes, width, height, 16, 0xFFFF, mask, 0, out)
    return code, list(out)


EXPECTED = [float(c + 1) for c in range(16)]


@pytest.mark.parametrize("mask", [-1, 3])
@pytest.mark.parametrize("size", [1, 64, 512, 1024])
def test_image_loss_whose_sums_do_not_arrive_is_an_error(fake, size, mask):
    assert loss(fake, size, size, mask) == (0, EXPECTED)
    fake.fake_drop_rows(1)
    code, _ = loss(fake, size, size, mask)
    assert code != 0 and b"image_loss" in fake.ntc_hip_last_error()
    assert loss(fake, size, size, mask) == (0, EXPECTED)                # and the next call is whole again
    assert fake.fake_dirty_counters() == 0


@pytest.mark.parametrize("mask", [-1, 3])
def test_image_loss_is_synchronous(fake, mask):
    """What the stream held, the launch included, is complete when the call returns, and an error of it is the call's."""
    for _ in range(2):
        assert loss(fake, mask=mask) == (0, EXPECTED)
        assert fake.fake_outstanding() == 0
    fake.fake_fail(b"hipEventSynchronize", 1)
    assert loss(fake, mask=mask)[0] != 0
    assert loss(fake, mask=mask) == (0, EXPECTED) and fake.fake_dirty_counters() == 0


@pytest.mark.parametrize("call", [1, 2, 3])
@pytest.mark.parametrize("name", ["hipMalloc", "launch_fill", "hipEventCreate", "hipHostMalloc", "hipHostGetDevicePointer", "launch_image_loss"])
def test_image_loss_after_a_set_up_that_failed(fake, name, call):
    """The first calls meet a failing allocation or launch (the n-th of its kind; a larger image grows the partial sums):
    each such call returns an error, and the first one without it finds the working memory whole."""
    fake.fake_fail(name.encode(), call)
    codes = []
    for size in (32, 1024, 4096, 64):
        code, values = loss(fake, size, size)
        codes.append(code)
        if code != 0:
            code, values = loss(fake, size, size)
        assert code == 0 and values == EXPECTED, (name, size)
    assert sum(c != 0 for c in codes) <= 1
    fake.fake_fail(name.encode(), 1 << 30)
    assert fake.fake_dirty_counters() == 0
