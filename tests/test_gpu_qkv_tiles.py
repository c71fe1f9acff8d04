"""GPU parity of the QKV epilogue on both of its tile shapes (64x128 up to one 128x128 tile a CU, 128x128
beyond) and in both of its requantisations (double; 64-bit past its bounds, in some or all of a wave's columns),
and of k_quant_rows on rows of every register length."""
import numpy as np
import pytest
import torch

import oracle
from tests.conftest import assert_equal, to_np
from tests.test_gpu_gemm import Case, dev, rand_bits
from tests.test_gpu_qkv_gn import check_qkv
from vela_amd import gemm as vg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,T,B", [(1, 1, 1), (1, 63, 1), (3, 129, 1), (5, 1056, 4), (2, 333, 13)])
@pytest.mark.parametrize("src", [vg.SRC_I16, vg.SRC_I8])
def test_tile_shapes(gpu, src, heads, T, B):
    """(5, 1056, 4): 33 x 8 = 264 128x128 tiles; the others at most 256."""
    check_qkv(src, heads, T, B=B, K=64, seed=heads + T, s_range=(18, 24), e_max=4)


@pytest.mark.parametrize("kw", [dict(s_range=(18, 30), e_max=6), dict(s_range=(4, 60), e_max=9), dict(s_range=(52, 60), e_max=3),
                                dict(s_range=(20, 40), m_range=(1 << 22, (1 << 31) - 1)), dict(s_range=(16, 20), b_range=(-(2**31), 2**31))])
@pytest.mark.parametrize("K", [64, 1280])
def test_forms(gpu, K, kw):
    check_qkv(vg.SRC_I8, 2, 130, B=1, K=K, seed=K, **kw)


FORMS = [dict(s_range=(18, 30), e_max=6), dict(s_range=(4, 60), e_max=9), dict(s_range=(52, 60), e_max=3), dict(s_range=(-2, 40), m_range=(1, 1 << 20)),
         dict(s_range=(20, 40), m_range=(1 << 22, (1 << 31) - 1)), dict(s_range=(16, 20), b_range=(-(2**31), 2**31))]


@pytest.mark.parametrize("kw", FORMS)
@pytest.mark.parametrize("src,K", [(vg.SRC_I16, 64), (vg.SRC_I8, 64), (vg.SRC_I8, 640)])
def test_forms_of_the_larger_tile(gpu, src, K, kw):
    """264 128x128 tiles, two row groups a wave: double, 64-bit and mixed columns, rows of y from 0 to saturation."""
    check_qkv(src, 5, 1056, B=4, K=K, seed=K, **kw)


@pytest.mark.parametrize("heads,T,B", [(2, 130, 1), (5, 1056, 4)])
def test_int_min_rows(gpu, heads, T, B):
    """Head rows that hold INT_MIN (shift 17, where the saturating add of the narrower shifts is not exact)."""
    kw = dict(s_range=(16, 18), b_range=(-(2**31), -(2**31) + 2))
    M, C = B * T, 64 * heads
    Y, _ = Case(vg.SRC_I8, M, 3 * C, 64, seed=9, **kw).reference()
    assert (Y[:, : 2 * C] == -(2**31)).any(1).all()
    check_qkv(vg.SRC_I8, heads, T, B=B, K=64, seed=9, **kw)


@pytest.mark.parametrize("K", [4, 252, 260, 516, 1020, 2044, 2052, 2500, 2560, 2564, 5116, 5120, 5124])
def test_quant_rows_lengths(gpu, K):
    r = np.random.default_rng(K)
    M, Kp = 37, (K + 15) // 16 * 16
    X = rand_bits(r, (M, K))
    hi = torch.full((64, Kp), 0x5A, dtype=torch.int8, device="cuda")
    lo = torch.full_like(hi, 0x5A)
    e = torch.full((64,), 0x5A, dtype=torch.int32, device="cuda")
    vg.k_quant_rows(dev(X), M, K, K, hi, lo, e, Kp)
    torch.cuda.synchronize()
    wh, wl, we = oracle.quant_rows(X, M, K, K, Kp)
    assert_equal(to_np(hi)[:len(wh)], wh, "hi")
    assert_equal(to_np(lo)[:len(wl)], wl, "lo")
    assert_equal(to_np(e)[:M], we[:M], "e")
