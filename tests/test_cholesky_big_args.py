"""The large solve keeps -g in its matrix's strict upper triangle, which has no room for it below three
unknowns: refused before anything is launched (no entry point gets there: fewer than 113 take the small one)."""
import ctypes
import importlib

import pytest

tdi = importlib.import_module("3di_amd.tdi")
abi = importlib.import_module("3di_amd.abi")


@pytest.mark.parametrize("K", [1, 2, 4097])
def test_sizes_without_room_are_refused(K):
    lib = ctypes.CDLL(tdi.lib()._name)
    solve = getattr(lib, "_ZN3tdi19launch_cholesky_bigEiiPKfS1_PfPiP12ihipStream_t")
    solve_f64 = getattr(lib, "_ZN3tdi23launch_cholesky_big_f64EiiPdPKdS0_PiP12ihipStream_t")
    null = ctypes.c_void_p()
    assert solve(1, K, null, null, null, null, null) == abi.TDI_ERR_ARG
    assert solve_f64(1, K, null, null, null, null, null) == abi.TDI_ERR_ARG
