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
