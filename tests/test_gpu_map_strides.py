"""dg_map and dg_map_noalloc with the coordinates in a part of longer rows, and the
projection written into a part of longer rows: the values of contiguous arrays, and
nothing else touched.  Of the long rows only the coordinates themselves count: rows
8 GiB apart (address space alone) are as good as any."""
import ctypes as C
import mmap

import numpy as np
import pytest

import dagtm_gpu as dg

pytestmark = pytest.mark.gpu
dp = C.POINTER(C.c_double)


def _engine(prec, N, K):
    rng = np.random.default_rng(N + K)
    T = rng.normal(size=(N, 7))
    e = dg.Engine(precision=prec)
    e.upload(T, np.ones((K, 1)), rng.normal(size=(K, 7)), 0.7)
    e.estep(True, 1.4)
    return e, rng


def _raw(e, name, X, L, ldX, M, ldM):
    f = getattr(C.CDLL(dg.LIB_PATH), name)       # its own prototype: plain addresses
    f.argtypes = [C.c_void_p, dp, C.c_int, C.c_long, dp, C.c_long]
    e._chk(f(e.h, X, L, ldX, M, ldM))


@pytest.mark.parametrize("prec", [dg.FP64, dg.MIXED])
@pytest.mark.parametrize("L,ldX,ldM", [(1, 5, 1), (2, 2, 9), (3, 70, 4)])
def test_padded_rows(L, ldX, ldM, prec):
    N, K = 1500, 130
    print(f"case: map, padded rows, precision={prec} L={L} ldX={ldX} ldM={ldM}", flush=True)
    e, rng = _engine(prec, N, K)
    with e:
        X = rng.normal(size=(K, ldX))
        want = e.map(np.ascontiguousarray(X[:, :L]))
        for name in ("dg_map", "dg_map_noalloc"):
            M = np.full((N, ldM), 123.0)
            _raw(e, name, X.ctypes.data_as(dp), L, ldX, M.ctypes.data_as(dp), ldM)
            assert np.array_equal(M[:, :L], want) and np.all(M[:, L:] == 123.0)


def test_rows_far_apart():
    N, K, L, step = 600, 40, 2, 1 << 30
    print("case: map, rows 8 GiB apart", flush=True)
    e, rng = _engine(dg.FP64, N, K)
    noreserve = 0x4000
    room = mmap.mmap(-1, ((K - 1) * step + L) * 8, flags=mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS | noreserve)
    with e:
        X = np.ndarray((K, L), buffer=room, strides=(8 * step, 8))
        X[:] = rng.normal(size=(K, L))
        want = e.map(np.ascontiguousarray(X))
        M = np.zeros((N, L))
        _raw(e, "dg_map", X.ctypes.data_as(dp), L, step, M.ctypes.data_as(dp), L)
        assert np.array_equal(M, want)
    del X
    room.close()
