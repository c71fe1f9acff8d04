"""GPU parity of the sixteen-row row-stationary kernel on rows with shifts, against the oracle: each form of
its requantisation (the integer form up to the largest shift its columns allow, the form in double one past
it and for wide scales, the general one), each epilogue, at the edges of its row stripes and column chunks;
and the automatic route to it."""
import pytest

from tests.test_gpu_gemm import Case
from vela_amd import gemm as vg

pytestmark = pytest.mark.gpu

FORMS = [
    ("integer", dict(s_range=(23, 26), e_max=7)),
    ("integer, at its limit", dict(s_range=(23, 23), m_range=(1 << 14, 1 << 15), e_max=7)),
    ("double, one past it", dict(s_range=(23, 23), m_range=(1 << 14, 1 << 15), e_max=8)),
    ("double", dict(s_range=(16, 24), e_max=11)),
    ("double, b near 2^31", dict(s_range=(18, 30), e_max=5, b_range=(-(2**31), 2**31))),
    ("double, large y", dict(s_range=(17, 18), m_range=(1 << 16, 1 << 18), e_max=15)),
    ("double, deep shifts", dict(s_range=(40, 52), e_max=3)),
    ("general", dict(s_range=(3, 12), e_max=17)),
]


@pytest.fixture(autouse=True)
def _reset(gpu):
    yield
    vg.set_variant(-1)


@pytest.mark.parametrize("name,kw", FORMS, ids=[f[0] for f in FORMS])
@pytest.mark.parametrize("epi", [vg.EPI_PLAIN, vg.EPI_GEGLU, vg.EPI_GELU])
@pytest.mark.parametrize("src", [vg.SRC_I16, vg.SRC_I8])
def test_forms(src, epi, name, kw):
    vg.set_variant(6)
    for i, (M, N, K) in enumerate([(300, 200, 320), (129, 72, 72)]):
        Case(src, M, N, K, epi=epi, seed=11 * i + epi, rowmax=i == 0, **kw).check(what=f"{name} {src} {epi} {M}x{K}x{N}")


@pytest.mark.parametrize("M,N,K", [(1, 8, 16), (127, 64, 320), (128, 136, 304), (257, 2568, 320), (1000, 320, 160)])
@pytest.mark.parametrize("epi", [vg.EPI_PLAIN, vg.EPI_GEGLU])
def test_edges(epi, M, N, K):
    vg.set_variant(6)
    Case(vg.SRC_I8, M, N, K, epi=epi, seed=M + K, rowmax=True, s_range=(23, 26), e_max=6).check(what=f"edges {epi} {M}x{K}x{N}")


@pytest.mark.parametrize("e_max", [0, 6, 11])
def test_automatic_route(e_max):
    """3100 x 320 x 2560: 980 tiles of 64x128, the row-stationary kernel without shifts and, with two chunks a block, the tile
    kernels with them."""
    Case(vg.SRC_I8, 3100, 2560, 320, epi=vg.EPI_GEGLU, seed=5 + e_max, rowmax=True, s_range=(23, 26), e_max=e_max).check(what=f"auto e {e_max}")


@pytest.mark.parametrize("epi,M,N,K", [(vg.EPI_GEGLU, 3520, 2560, 320), (vg.EPI_GEGLU, 6592, 2560, 304), (vg.EPI_PLAIN, 20544, 320, 160), (vg.EPI_GELU, 7040, 1280, 320),
                                       (vg.EPI_GELU, 8320, 1280, 64)])
def test_automatic_route_by_ranges(epi, M, N, K):
    """Grids of one round and of more that the rule on a block's chunks sends to the row-stationary kernel."""
    Case(vg.SRC_I8, M, N, K, epi=epi, seed=M, rowmax=True, s_range=(23, 26), e_max=6).check(what=f"auto {epi} {M}x{K}x{N}")
