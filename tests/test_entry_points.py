"""C entry points of the kernel modules refuse what no kernel computes, before anything is launched (no GPU needed)."""
import ctypes
import glob
import os

import pytest
import torch

import pilottai_amd

FOUND = glob.glob(os.path.join(os.path.dirname(pilottai_amd.__file__), "_hybrid.*.so"))


@pytest.mark.skipif(not FOUND or torch.cuda.is_available(), reason="not built, or operands that are not there could be read")
@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("epi", [1, 2])
def test_dense_grouped_rows_have_no_gated_unit(fp32, epi):
    """A gated unit or a square of relu of dense rows (no tiles) is refused, in both types alike."""
    f = ctypes.CDLL(FOUND[0]).pa_grouped_gemm
    n, z = None, ctypes.c_float(0)
    rc = f(fp32, n, n, n, ctypes.c_longlong(0), 1, 64, 0, 64, 0, 16, 4, 2, n, 0, n, n, 0, 0, 16, epi, z, z, z, z, n, n, 0, 0, 0, 0,
           n, n, 0, n, n, 0, 0, 0, n)
    assert rc == -1


@pytest.mark.skipif(not glob.glob(os.path.join(os.path.dirname(pilottai_amd.__file__), "_C.*.so")), reason="not built")
@pytest.mark.parametrize("M", [0, -1, -300, 1])
@pytest.mark.parametrize("N", [0, 128, 3072, 28672])
def test_plan_of_a_product_without_rows(M, N):
    """The plan of no rows is empty, with the width by N, whoever leaves the width open."""
    from pilottai_amd import _C

    full, S, ws, bn = _C.prefill_gemm_plan(M, N, 768)
    assert (full, S, ws) == (N // bn if M > 0 else 0, 1, 0) and (bn == (256 if N > 6144 else 128) or M > 0)
    lib, n = ctypes.CDLL(_C.__file__), [ctypes.c_int(-1), ctypes.c_int(-1)]
    lib.pa_prefill_gemm_plan(M, N, 768, 0, ctypes.byref(n[0]), ctypes.byref(n[1]))
    assert [n[0].value, n[1].value] == [full, S]
    floats = lib.pa_prefill_gemm_ws_floats
    floats.restype = ctypes.c_longlong
    assert floats(M, N, 0, full, S) == ws
