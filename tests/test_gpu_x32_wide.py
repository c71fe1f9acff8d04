"""GPU parity of int32 rows of many tiles against the oracle, on 64x320 tiles (deep K, a last round of two blocks a
CU that is filled) and on the 64x128 ones that shallow K keeps: ragged rows and columns, K of one partial step up to
several, every form of the epilogue."""
import numpy as np
import pytest

from tests.test_gpu_gemm import Case
from vela_amd import gemm as vg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(24513, 320, 4), (24576, 318, 68), (24577, 320, 64), (32768, 320, 132), (12225, 637, 192),
                                   (8143, 958, 36), (24512, 320, 64)])
def test_shapes(M, N, K):
    """383 to 512 tiles of 64x320, all of them with too shallow a K: 64x128 tiles."""
    Case(vg.SRC_X32, M, N, K, seed=M + K, residual=N % 4 == 0, rowmax=True).check(what=f"X32 {M}x{K}x{N}")


@pytest.mark.parametrize("shift", [0, 16, 24])
@pytest.mark.parametrize("kw", [dict(), dict(s_range=(4, 60)), dict(m_range=(1 << 28, (1 << 31) - 1)), dict(b_range=(-(2**31), 2**31))])
def test_forms(kw, shift):
    """shift 24 and 16: 8-bit rows (no row shift) and 16-bit rows; the block's forms differ by them and by cst (64x128 tiles)."""
    c = Case(vg.SRC_X32, 24520, 320, 72, seed=shift, rowmax=True, **kw)
    c.x >>= shift
    c.xrm = np.abs(c.x.astype(np.int64)).max(1).astype(np.uint32)
    c.kw = dict(x=c.x, xrowmax=c.xrm, K=c.K)
    c.check(what=f"X32 forms {kw} >> {shift}")


@pytest.mark.parametrize("M,N,K", [(24513, 320, 644), (24576, 318, 640), (31745, 320, 320), (14300, 637, 772), (8143, 958, 1284)])
def test_deep_k(M, N, K):
    """Shapes that the rule on K sends to the wide tile (one column of tiles, two and three)."""
    Case(vg.SRC_X32, M, N, K, seed=M + K, residual=N % 4 == 0, rowmax=True).check(what=f"X32 {M}x{K}x{N}")


@pytest.mark.parametrize("shift", [0, 16, 24])
@pytest.mark.parametrize("kw", [dict(), dict(s_range=(4, 60)), dict(m_range=(1 << 28, (1 << 31) - 1)), dict(b_range=(-(2**31), 2**31))])
def test_forms_full_round(kw, shift):
    """The forms again at K = 320 and a full round of tiles, which the rule sends to the wide tile."""
    c = Case(vg.SRC_X32, 31800, 320, 320, seed=shift, rowmax=True, **kw)
    c.x >>= shift
    c.xrm = np.abs(c.x.astype(np.int64)).max(1).astype(np.uint32)
    c.kw = dict(x=c.x, xrowmax=c.xrm, K=c.K)
    c.check(what=f"X32 forms {kw} >> {shift}")
