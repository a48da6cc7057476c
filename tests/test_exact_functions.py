"""The kernels' shortcuts - divisions by corrected reciprocals, colour encoding by approximation with a test for certainty,
products and shifts for quotients - give the operation's own bits for every operand they are used on: all of them are
tried on the GPU (tests/exact_functions.hip, compiled with the kernel files themselves), but for quotient_by(), whose
operands are too many."""
import ctypes as C
import os

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))


class Report(C.Structure):
    _fields_ = [("tried", C.c_uint64), ("wrong", C.c_uint64), ("example", C.c_uint64)]


@pytest.mark.parametrize("subject,function,cases", [
    ("copy", "encoded_half_srgb", 1 << 32), ("copy", "encoded_half_hlg", 1 << 32),
    ("copy", "put_unorm8", 1 << 32), ("copy", "divide_by_255", (1 << 23) + 256), ("copy", "divide_by_65535", (1 << 23) + 65536),
    ("bc", "code_quotient", 96), ("bc", "bc4_palette", 65536), ("bc", "bc4_positions", 1 << 20), ("bc", "bc4_refit", 1 << 24),
    ("bc6", "quotient_of_integers", (1 << 17) * ((1 << 17) - 1)), ("bc6", "quotient_of_log2", None),
    ("bc6", "quotient_of_msle", 0x7c00 * (0x7c00 + 256 + 65536 + 65505)), ("bc6", "log_estimate", 34 << 23), ("bc6", "quotient_of_codes", 3 * 65536 + 64),
    ("bc6", "quotient_of_diagonals", 1 << 30), ("decode", "texel_centre", (1 << 15) * 65537),
    ("decode", "floors_of", 0x43800000), ("decode", "filtered_features", 1 << 26)])
def test_gpu_shortcut_equals_the_operation(device, subject, function, cases):
    path = os.path.join(HERE, f"libexact_{subject}.so")
    assert os.path.exists(path), f"{path} is not built; run __graft_entry__.build() (make -C tests)"
    report = Report()
    print(function, flush=True)
    assert getattr(C.CDLL(path), "exact_" + function)(C.byref(report)) == 0
    assert report.wrong == 0, f"{report.wrong} of {report.tried} cases differ, case {report.example:#x} among them"
    assert report.tried == cases if cases else report.tried > 1 << 23
