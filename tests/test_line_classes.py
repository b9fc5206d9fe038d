"""The classes of the batched line kernels (chunk length, threads per row), on
the CPU: every class that the shape rule or a tuning table can choose has a
kernel in the launch of several classes, and the host knows the others from
these (a workgroup of an unknown class would do nothing)."""
import ctypes

import pytest

mg = pytest.importorskip("mgpoisson2d_amd.capi")

KERNELS = {(2, 64), (4, 64), (8, 64), (2, 128), (4, 128), (8, 128), (2, 256), (4, 256), (8, 256), (16, 256)}


def native(name, *argtypes, res=ctypes.c_int):
    f = getattr(mg.lib, name)
    f.restype, f.argtypes = res, argtypes
    return f


def test_known_classes():
    known = native("_ZN3mgp17xline_batch_classEii", ctypes.c_int, ctypes.c_int, res=ctypes.c_bool)
    got = {(C, t) for C in range(1, 65) for t in (32, 64, 128, 256, 512, 1024) if known(C, t)}
    assert got == KERNELS


def test_chosen_classes_are_known():
    shape = native("_ZN3mgp17xline_batch_shapeEiRiS0_", ctypes.c_int, ctypes.POINTER(ctypes.c_int),
                   ctypes.POINTER(ctypes.c_int), res=None)
    chunk = native("_ZN3mgp17xline_batch_chunkEiim", ctypes.c_int, ctypes.c_int, ctypes.c_size_t)
    for nx in range(4, 4112):
        C, t = ctypes.c_int(), ctypes.c_int()
        shape(nx, ctypes.byref(C), ctypes.byref(t))
        assert (C.value, t.value) in KERNELS, nx
        for width in (64, 128, 256):
            for elem in (4, 8):
                c = chunk(nx, width, elem)
                assert c == 0 or (c, width) in KERNELS, (nx, width, elem)
