"""How the gated block's kernel cuts a shape (shadow_amd/csrc/gate_shape.h): what every cut has to
keep to, and which form the shapes of the GPU tests get."""
import ctypes
import os

import pytest

from tests.native import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def native():
    path = os.path.join(HERE, "native", "gate_shape.so")
    if not os.path.exists(path):
        build.build()
    return ctypes.CDLL(path)


@pytest.mark.parametrize("rows", [1, 2, 255, 512, 513, 1023, 1024, 1025, 2047, 2048, 4096, 4097, 8192, 16384, 65536, 1 << 20])
def test_every_cut_fits_the_kernel(native, rows):
    assert native.gate_shape_scan(rows, 15360) == 0


def cut(native, rows, length):
    out = (ctypes.c_uint * 7)()
    native.gate_shape(rows, length, out)
    lanes, pieces, group, chunk, _, slots, together = out
    return {"lanes": 1 << lanes, "turns": group * (1 << lanes) // 256, "slots": slots, "chunked": chunk != pieces,
            "cut_group": rows % group != 0, "together": bool(together)}


def test_forms_of_the_gpu_shapes(native):
    """The shapes of test_gpu_gate.py reach the forms they are there for."""
    from tests.test_gpu_gate import FORMS
    for (n, c, h, w), form in FORMS.items():
        got = cut(native, n * c, h * w)
        assert {k: got[k] for k in form} == form, (n, c, h, w, got)
    assert {f["slots"] for f in FORMS.values()} == {1, 4, 8, 16}


# groups of 4, 8, 12 and 16 rows, longer and shorter than the rule asks for, and few workgroups of four
@pytest.mark.parametrize("rows,length,together", [
    (6700, 784, True), (6700, 400, True), (6700, 384, True), (6700, 383, False), (6700, 225, False), (4096, 225, True), (4097, 225, False),
    (13000, 784, True), (13000, 767, False), (10000, 289, False), (13000, 225, False), (30000, 49, False), (30000, 289, False),
    (300, 49, False), (300, 81, True), (1000, 12543, True), (2000, 6561, True)])
def test_which_rows_are_walked_together(native, rows, length, together):
    assert cut(native, rows, length)["together"] is together


def test_which_kernel_the_gpu_shapes_get(native):
    """Forms of whole vectors reach both kernels: with all parts some are whole_squeeze_gate_kernel's, with one left out none."""
    from tests.test_gpu_gate import FORMS, GENERIC, WHOLE

    def whole(shape, stats=True, relu=True, residual=True):
        return native.gate_takes_whole(shape[0] * shape[1], shape[2] * shape[3], stats, relu, residual) == 1
    vectors = [s for s in FORMS if s[2] * s[3] % 4 == 0]
    assert {s for s in FORMS if whole(s)} == {(516, 1, 84, 84), (2060, 1, 44, 44), (2061, 1, 60, 60), (600, 1, 112, 112), (3, 2, 112, 112),
                                              (8201, 1, 28, 28), (4101, 1, 16, 24), (13003, 1, 20, 20)}
    assert all(whole(s) for s in WHOLE)
    for parts in GENERIC + [dict(residual=False)]:
        assert not any(whole(s, **parts) for s in vectors + WHOLE)
    # what is left to squeeze_gate_kernel: every number of vectors a lane and both walks
    forms = [cut(native, s[0] * s[1], s[2] * s[3]) for s in vectors]
    assert {(f["slots"], f["chunked"], f["turns"] > 1) for f in forms} >= {
        (4, False, False), (4, False, True), (8, False, True), (8, True, False), (8, True, True), (16, False, False), (16, True, False)}
    assert {(f["slots"], f["together"]) for f in forms} >= {(4, False), (4, True), (8, False), (8, True), (16, True)}


@pytest.mark.parametrize("rows", [1, 2, 255, 1023, 1024, 1025, 4095, 4096, 8192, 16384, 65536])
def test_every_cut_of_whole_rows_fits_its_kernel(native, rows):
    assert native.gate_whole_scan(rows, 15360) == 0


def test_whole_rows_of_the_gpu_shapes(native):
    """The shapes of test_gpu_gate.py take every number of vectors a lane and every number of lanes a row."""
    from tests.test_gpu_gate import WHOLE
    out = (ctypes.c_uint * 3)()
    got = []
    for n, c, h, w in WHOLE:
        assert native.gate_whole(n * c, h * w, out) == 1, (n, c, h, w)
        got.append((out[0], out[1], n * c % out[2] != 0))
    assert {p for _, p, _ in got} == set(range(1, 16))
    assert {lanes for lanes, _, _ in got} == {16, 32, 64, 256}
    assert {lanes for lanes, _, cut in got if cut} == {16, 32, 64}
