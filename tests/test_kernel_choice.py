"""Which kernel phase 1 plans for a shape (mhcPreExecutorKernel before a launch), without a GPU."""
from __future__ import annotations

import ctypes

import pytest

from test_host_api import _descs


@pytest.fixture(scope="module")
def lib(pkg):
    return pkg.load_library()


def _kernel(pkg, lib, **shape):
    mk = lambda v: None if v is None else ctypes.byref(pkg.make_tensor(*v))
    d = _descs(pkg, **shape)
    ws, exe, name = ctypes.c_uint64(0), ctypes.c_void_p(None), ctypes.c_char_p()
    st = lib.mhcPreGetWorkspaceSize(*[mk(d[k]) for k in ("x", "phi", "alpha", "bias", "gamma")],
                                    ctypes.c_float(1e-6), ctypes.c_float(1e-6),
                                    *[mk(d[k]) for k in ("hIn", "hPost", "hRes")],
                                    ctypes.byref(ws), ctypes.byref(exe))
    assert st == 0
    assert lib.mhcPreExecutorKernel(exe, ctypes.byref(name)) == 0
    lib.mhcPreExecutorDestroy(exe)
    return name.value.decode()


@pytest.mark.parametrize("n,D,S,want", [
    (4, 256, 128, "cell"), (4, 7168, 16, "cell"), (4, 7168, 128, "rows"), (4, 7168, 8192, "strip"),
    (4, 1200, 777, "strip"), (4, 400, 2048, "split"), (4, 64, 8192, "split"),
    (6, 1024, 64, "cell"), (6, 1024, 2048, "slab"), (6, 5120, 37, "rows"), (6, 2000, 300, "slab"),
    (6, 8192, 4096, "rows"), (8, 1024, 32, "cell"), (8, 7168, 64, "rows"), (8, 1024, 1024, "split"),
])
def test_planned_kernel(pkg, lib, n, D, S, want):
    assert _kernel(pkg, lib, n=n, D=D, S=S) == want


@pytest.mark.parametrize("n,D,S,want", [(4, 7168, 8192, "strip"), (6, 4096, 4096, "slab"), (8, 16384, 64, "rows"),
                                        (4, 256, 128, "cell")])
def test_set_slice_width_keeps_to_the_grid(pkg, lib, monkeypatch, n, D, S, want):
    """MHCPRE_CELL sets the cell kernel's slices where the kernel is made for
    the grid that comes of it, and changes nothing elsewhere."""
    monkeypatch.setenv("MHCPRE_CELL", "1")
    assert _kernel(pkg, lib, n=n, D=D, S=S) == want


@pytest.mark.parametrize("n,D,S,want", [(6, 2000, 1 << 21, "slab"), (6, 2000, 1 << 23, "split"),
                                        (4, 7056, 200000, "strip"), (4, 7056, 400000, "split"),
                                        (4, 7168, 1 << 23, "strip")])
def test_computing_an_expired_wait_is_bounded(pkg, lib, n, D, S, want):
    """A slab or strip launch in place of kernels that wait for nobody has at
    most 2^17 strips of rows per wave to compute alone (about a second)."""
    assert _kernel(pkg, lib, n=n, D=D, S=S) == want
