"""Which kernel the batched GEMM runs (host rules; no GPU): the choice with weights
that do not start on a dword, and a group's launch against what it announces."""

import ctypes
import itertools
import os

import pytest

import oracle

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mini-llama-cpp-release_amd",
                   "libmlq_hip.so")
TYPES = {oracle.Q8_0: "q8_0", oracle.Q4_0: "q4_0", oracle.Q4_1: "q4_1"}


class Shape(ctypes.Structure):
    _fields_ = [(f, ctypes.c_int) for f in ("qtype", "M", "K", "nb", "rows")]


@pytest.fixture(scope="module")
def gemm():
    """The library's C++ entry points (csrc/mlq_kernels.h) by their exported names."""
    lib = ctypes.CDLL(LIB)
    name = lib._ZN3mlq16gemm_kernel_nameERKNS_11LinearShapeEb
    name.restype = ctypes.c_char_p
    name.argtypes = [ctypes.POINTER(Shape), ctypes.c_bool]
    group = lib._ZN3mlq20gemm_group_supportedERKNS_11LinearShapeEiPKPKvPKi
    group.restype = ctypes.c_bool
    group.argtypes = [ctypes.POINTER(Shape), ctypes.c_int, ctypes.POINTER(ctypes.c_void_p), ctypes.POINTER(ctypes.c_int)]

    need = lib._ZN3mlq20gemm_workspace_bytesERKNS_11LinearShapeE
    need.restype = ctypes.c_size_t
    need.argtypes = [ctypes.POINTER(Shape)]

    class Gemm:
        @staticmethod
        def workspace(qt, m, k, rows):
            return need(ctypes.byref(Shape(qt, m, k, (k + 31) // 32, rows)))

        @staticmethod
        def kernel(qt, m, k, rows, dword=True):
            return name(ctypes.byref(Shape(qt, m, k, (k + 31) // 32, rows)), dword).decode()

        @staticmethod
        def grouped(qt, ms, k, rows, at):
            ptrs = (ctypes.c_void_p * len(ms))(*([4096 + at] * len(ms)))
            return group(ctypes.byref(Shape(qt, 0, k, (k + 31) // 32, rows)), len(ms), ptrs, (ctypes.c_int * len(ms))(*ms))

    return Gemm


ROWS = (2, 16, 17, 64, 129, 333, 512, 2048)


@pytest.mark.parametrize("qt", list(TYPES), ids=list(TYPES.values()))
def test_weights_off_a_dword_run_the_chunk_kernel(gemm, qt):
    """The large-tile kernel copies weights to LDS by dwords; the chunk kernel loads
    them from any address, so it takes every call that its shape allows."""
    tiles = 0
    for rows, m, k in itertools.product(ROWS, (1, 300, 4096, 11008), (64, 256, 896, 4090, 4096, 4160, 11008)):
        nb = (k + 31) // 32
        chunked = nb % 4 == 0 and nb >= 8 and k == 32 * nb
        at = gemm.kernel(qt, m, k, rows, True)
        off = gemm.kernel(qt, m, k, rows, False)
        assert ("_chunk_" in off) == chunked and "_tile_" not in off, (rows, m, k, off)
        assert ("_chunk_" in at or "_tile_" in at) == chunked, (rows, m, k, at)
        if "_tile_" not in at:
            assert at == off, (rows, m, k)
        tiles += "_tile_" in at
    assert tiles > 20


@pytest.mark.parametrize("qt", list(TYPES), ids=list(TYPES.values()))
def test_group_of_weights_off_a_dword(gemm, qt):
    """A group launches for weights at any address where each weight but the last is
    whole row tiles of the kernel that the plan names."""
    for rows, (ms, k) in itertools.product(ROWS, [((4096, 4096, 4096), 4096), ((896, 128, 128), 896),
                                                  ((11008, 11008), 4096), ((2048, 300), 2048), ((192, 64), 896),
                                                  ((300, 2048), 2048), ((256, 256), 4160)]):
        nb = k // 32
        for at in (0, 2):
            name = gemm.kernel(qt, sum(ms), k, rows, at == 0)
            whole = nb % 4 == 0 and all(m % int(name.split("_bm")[1].split("_")[0]) == 0 for m in ms[:-1])
            assert gemm.grouped(qt, ms, k, rows, at) == whole, (rows, ms, k, at, name)


@pytest.mark.parametrize("qt,m,k,rows,need", [
    (oracle.Q4_0, 4096, 4096, 16, 2629888), (oracle.Q4_0, 4096, 4096, 128, 19202560),
    (oracle.Q4_0, 4096, 4096, 129, 22381312), (oracle.Q8_0, 4096, 4096, 300, 26641664),
    (oracle.Q8_0, 4096, 4096, 512, 25692160), (oracle.Q4_1, 11008, 4096, 512, 8914944),
    (oracle.Q4_0, 12790, 384, 130, 16900352), (oracle.Q8_0, 2121, 11264, 292, 45769984),
    (oracle.Q4_0, 300, 4160, 200, 7113728), (oracle.Q4_1, 70, 4092, 33, 1487104)])
def test_workspace_of_a_shape_stays(gemm, qt, m, k, rows, need):
    """A shape's workspace is part of the interface: it says which calls fit the fixed
    scratch of mlq_hip_quant_linear_noalloc and a workspace that graphs recorded."""
    assert gemm.workspace(qt, m, k, rows) == need
