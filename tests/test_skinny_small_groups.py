"""Experts' gated products of few rows: 16 + 16 rows of W and four waves a workgroup."""
import pytest
import torch

from test_kernels import ops, run_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (7, 112, 320), (16, 144, 1088), (33, 528, 192)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("glu,grouped", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("tiled", [False, True])
def test_sixteen_rows_and_four_waves(M, N, K, out_dtype, glu, grouped, tiled):
    def fn(a, w, y, *args, **kw):
        ops().gemm_skinny(a, ops().operand_order(w) if tiled else w, y, *args, tiled=tiled, variant=5, **kw)
    run_gemm(fn, torch.bfloat16, out_dtype, M, N, K, glu, grouped)
