"""GPU parity of the attention's forms against the oracle: key counts around every change of form (scores
kept by one, two or four waves, or recomputed; 64-key tiles with and without a remainder; more keys than
fit the LDS constants at once), full and causal, with the integer arithmetic and with the general one
(large shifts, or a table that starts below 2^30 or rises); and the forms of the operand
producers."""
import numpy as np
import pytest
import torch

import oracle
from tests.conftest import assert_equal, to_np
from tests.test_gpu_attention import dev, gpu_heads, gpu_v, host
from vela_amd import attention as va

pytestmark = pytest.mark.gpu

EXP = oracle.exp_table()
RISING = EXP[::-1].copy()          # not monotone falling: the general form
SMALL = (EXP >> 8).copy()          # starts at 2^22: r needs more than 32 bits


def check(B, heads, Tq, Tk, causal, scale=70000, table=EXP, seed=0, big_keys=False):
    r = np.random.default_rng(seed + 1000 * Tq + Tk)
    C = heads * 64
    X = [r.normal(0, scale, (B * n, C)).astype(np.int32) for n in (Tq, Tk, Tk)]
    X[0][::5] = (X[0][::5] * 0.01).astype(np.int32)      # other shifts among the rows
    X[1][::7] = (X[1][::7] * 0.02).astype(np.int32)
    if big_keys:
        X[1][1] = 1 << 29                                 # eq + ek > 12 for every query
    check_rows(X, B, heads, Tq, Tk, causal, table)


def check_rows(X, B, heads, Tq, Tk, causal, table=EXP):
    C = heads * 64
    Tqp, Tkp = (Tq + 63) // 64 * 64, (Tk + 63) // 64 * 64
    q, k, v = gpu_heads(X[0], B, Tq, C, heads, Tqp), gpu_heads(X[1], B, Tk, C, heads, Tkp), gpu_v(X[2], B, Tk, C, heads, Tkp)
    out = torch.full((B * Tq, C), 0x5a5a5a5a, dtype=torch.int32, device="cuda")
    rm = torch.zeros(B * Tq, dtype=torch.int32, device="cuda")
    va.k_fused_attention(*q[:5], k[0], k[1], k[2], k[5], *v, B, heads, Tq, Tqp, Tk, Tkp, causal, dev(table), C, None, None, out, rm)
    torch.cuda.synchronize()
    qh, kh, vh = host(q), host(k), host(v)
    wrm = np.zeros(B * Tq, np.uint32)
    want = oracle.attention(qh[0], qh[1], qh[2], kh[0], kh[1], kh[2], vh[0], vh[1], vh[2], B, heads, Tq, Tqp, Tk, Tkp, causal, table, C, rowmax=wrm)
    what = f"Tq {Tq} Tk {Tk} causal {causal}"
    assert_equal(to_np(out), want, what + " out")
    assert_equal(to_np(rm).view(np.uint32), wrm, what + " rowmax")


def edge_rows(r, shape):
    X = r.normal(0, 60000, shape).astype(np.int32)
    X[:: 9] = r.integers(-(2**31), 2**31, X[::9].shape, dtype=np.int64).astype(np.int32)
    X[3:: 11] = r.integers(-3, 4, X[3::11].shape)
    X[5:: 50] = -(2**31)
    return X


@pytest.mark.parametrize("B,T,heads,C,Tp,shift", [(1, 1, 1, 64, 64, 0), (2, 77, 3, 192, 128, 0), (1, 50, 2, 130, 64, 0), (1, 50, 2, 128, 64, 1),
                                                  (8, 1000, 5, 324, 1024, 0), (3, 33, 12, 768, 35, 0)])
def test_quant_heads_forms(gpu, B, T, heads, C, Tp, shift):
    """Aligned rows and planes, odd widths, a source off 16 bytes (shift elements), few and many rows."""
    X = edge_rows(np.random.default_rng(T + C), (B * T, C))
    flat = torch.zeros(B * T * C + 4, dtype=torch.int32, device="cuda")
    Xd = flat[shift : shift + B * T * C]
    Xd.copy_(dev(X).reshape(-1))
    n = B * heads * Tp
    got = [torch.full((n, 64), 0x5a, dtype=torch.int8, device="cuda") for _ in range(2)] + [torch.full((n,), 7, dtype=torch.int32, device="cuda")]
    got += [torch.full((n,), 7, dtype=torch.int64, device="cuda") for _ in range(3)]
    va.k_quant_heads(Xd, B, T, C, heads, Tp, *got)
    torch.cuda.synchronize()
    for g, w, name in zip(got, oracle.quant_heads(X, B, T, C, heads, Tp), ("hi", "lo", "e", "hs", "ls", "tsum")):
        assert_equal(to_np(g), w, name)


@pytest.mark.parametrize("B,Tk,heads,C,Tkp", [(1, 1, 1, 64, 64), (2, 64, 2, 128, 64), (2, 65, 2, 130, 128), (1, 100, 3, 192, 256), (2, 128, 1, 65, 128),
                                              (2, 129, 2, 128, 192), (1, 700, 5, 320, 704)])
def test_quant_v_forms(gpu, B, Tk, heads, C, Tkp):
    """One block a group and rows split over blocks, remainders of both, twice into the same buffers."""
    r = np.random.default_rng(Tk)
    G = B * heads
    got = [torch.full((G * 64, Tkp), 0x5a, dtype=torch.int8, device="cuda") for _ in range(2)]
    got += [torch.full((G * 64,), 99, dtype=torch.int32, device="cuda"), torch.full((G * 64,), 99, dtype=torch.int64, device="cuda")]
    for scale in (60000, 900):
        X = (edge_rows(r, (B * Tk, C)) if scale > 1000 else r.normal(0, scale, (B * Tk, C)).astype(np.int32))
        va.k_quant_v(dev(X), B, Tk, C, heads, Tkp, *got)
        torch.cuda.synchronize()
        for g, w, name in zip(got, oracle.quant_v(X, B, Tk, C, heads, Tkp), ("vthi", "vtlo", "ev", "vsum")):
            assert_equal(to_np(g), w, name)


@pytest.mark.parametrize("Tk", [1, 64, 65, 128, 129, 192, 256, 257, 448, 512, 513, 1000, 1024, 1025, 1217, 4096, 4161])
def test_key_counts(gpu, Tk):
    check(1, 2, 37, Tk, False)


@pytest.mark.parametrize("T", [1, 17, 64, 130, 257, 300, 513, 700, 1100])
def test_causal(gpu, T):
    check(1, 2, T, T, True)


@pytest.mark.parametrize("Tk", [77, 250, 400, 900, 1090])
@pytest.mark.parametrize("kw", [dict(table=RISING), dict(table=SMALL), dict(big_keys=True)])
def test_general_form(gpu, Tk, kw):
    check(1, 1, 20, Tk, False, **kw)


def test_dominant_key(gpu):
    """One key takes a row's whole probability (sum of E = 2^30, r = 2^32, P = 32768 before the clamp)."""
    for Tk in (3, 200, 1100):
        check(1, 1, 33, Tk, False, scale=600000)


@pytest.mark.parametrize("Tk", [1, 3, 20, 63, 64])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kw", [dict(), dict(table=RISING), dict(table=SMALL), dict(scale=20000000)])
def test_one_tile(gpu, Tk, causal, kw):
    """Keys of one tile, in the integer arithmetic and in the general one."""
    check(2, 3, 70, Tk, causal, **kw)


@pytest.mark.parametrize("T", [150, 300, 700, 1100])
@pytest.mark.parametrize("kw", [dict(table=RISING), dict(table=SMALL), dict(big_keys=True)])
def test_general_form_causal(gpu, T, kw):
    check(1, 1, T, T, True, **kw)


@pytest.mark.parametrize("kw", [dict(), dict(table=SMALL)])
def test_causal_past_the_staged_keys(gpu, kw):
    """More keys than the LDS constants hold at a time, causal: queries on both sides of the restaging."""
    check(1, 1, 4170, 4170, True, **kw)


@pytest.mark.parametrize("total", [12, 13])
@pytest.mark.parametrize("Tk", [20, 77, 200, 400, 1000, 1100])
def test_dominant_key_by_form(gpu, Tk, total):
    """test_dominant_key with the shifts held: eq + ek = 12 at most, the last sum of the integer arithmetic (where r =
    2^32 is taken as 2^32 - 1), and 13, the first of the general one, for every form by the number of keys."""
    r = np.random.default_rng(Tk)
    Tq, lo, hi = 33, 1 << 20, (1 << 21) - 1            # shift 6
    sign = r.choice([-1, 1], 64)
    Xq, Xk = r.integers(lo, hi, (Tq, 64)) * sign, r.integers(-hi, hi, (Tk, 64))
    Xk[:, 0] = r.choice([-1, 1], Tk) * r.integers(lo, hi, Tk)
    top = [0, Tk // 2, Tk - 1][Tk % 3]
    Xk[top] = hi * sign
    if total == 13:
        Xk[(top + 1) % Tk, 3] = hi + 1                 # shift 7
    eq, ek = oracle.quant_heads(Xq.astype(np.int32), 1, Tq, 64, 1, 64)[2], oracle.quant_heads(Xk.astype(np.int32), 1, Tk, 64, 1, (Tk + 63) // 64 * 64)[2]
    assert eq[:Tq].min() == eq[:Tq].max() == 6 and eq.max() + ek.max() == total
    # scores in Q16, a margin of 1 % for the rounding: all but one key 16 e-folds and more below, so that sum E = 2^30
    S = np.sort((Xq.astype(np.float64) @ Xk.T.astype(np.float64)) / 2**19, axis=1)
    assert (S[:, -1] - S[:, -2] > 1.01 * 2**20).all() and EXP[0] == 1 << 30
    check_rows([Xq.astype(np.int32), Xk.astype(np.int32), r.integers(-(2**31), 2**31, (Tk, 64), dtype=np.int64).astype(np.int32)], 1, 1, Tq, Tk, False)
