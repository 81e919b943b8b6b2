"""Where Q is quantised: the rule on the host (tests/capi_host/routes.cpp).  The groups of wavefronts and the selection kernel take Q as codes,
so the calls that have them keep Q in front."""
import pytest

from test_gpu_q_in_place import BATCHED, MASKS
from test_forward_routes import CDF, MASK, TOPK, pytestmark, routes  # noqa: F401


@pytest.mark.parametrize("kw,in_front", [
    (dict(H=36, N=2048, Nk=4096), 1), (dict(H=37, N=2048, Nk=4096), 0), (dict(H=577, N=1, Nk=3000), 0), (dict(H=577, N=128, Nk=8192, selection=CDF), 0),
    (dict(H=577, N=128, Nk=8193, selection=CDF), 1), (dict(H=32, Hkv=8, N=4096), 0), (dict(H=577, N=128, Nk=3000, pv_f16=1), 0),
    (dict(H=11, N=4096, selection=MASK), 1), (dict(H=11, N=4097, selection=MASK), 0), (dict(H=48, N=16384, selection=MASK), 0),
    (dict(H=48, N=16384, D=64), 1), (dict(H=48, N=16384, D=64, selection=MASK), 1), (dict(H=48, N=8192, D=64), 1), (dict(H=700, N=128, Nk=256), 0)])
def test_where_q_is_quantised(routes, kw, in_front):  # noqa: F811
    assert routes(**kw)[4] == in_front


@pytest.mark.parametrize("kw,in_front", [
    (dict(H=24, N=2048), 1), (dict(H=28, N=2304), 1), (dict(H=28, N=2432), 0), (dict(H=48, N=1024), 1), (dict(H=80, N=1024), 0),
    (dict(H=44, N=2048, Nk=500), 1), (dict(H=28, N=2688, Nk=1000), 1), (dict(H=36, N=4608, Nk=800), 0), (dict(H=60, N=1024, Nk=9000), 1),
    (dict(H=61, N=1024, Nk=9000), 0), (dict(H=32, Hkv=8, N=1408), 1), (dict(H=32, Hkv=8, N=1409), 0)])
def test_masks_over_many_heads_keep_q_in_front_of_small_grids(routes, kw, in_front):  # noqa: F811
    """In front of a grid that its reads do not fill, the blocks of Q cost nothing: 24 heads N2048 took 49.8 us a call, 53.0 in place."""
    assert routes(selection=MASK, **kw)[4] == in_front


def test_groups_never_meet_q_in_place(routes):  # noqa: F811
    for H, N in ((1, 32768), (2, 16384), (256, 128), (4, 8192)):
        for sel in (TOPK, CDF, MASK):
            for Nk in (64, 800, 4096, 8192, 20000):
                r = routes(H=H, N=N, Nk=Nk, selection=sel)
                assert r[3] == 1 or r[4] == 1


@pytest.mark.parametrize("kw", [dict(H=24, N=3200, Nk=640), dict(H=24, N=3200, Nk=640, selection=CDF), dict(H=32, Hkv=8, N=2688, Nk=1024)])
def test_the_workspace_serves_every_similarity_threshold(routes, kw):  # noqa: F811
    """A workspace is sized once for a shape; with a similarity threshold short heads take another route."""
    a, b = routes(sim=-0.1, **kw), routes(sim=0.3, **kw)
    assert a[4] != b[4] and a[5] == b[5]


def test_the_tests_of_q_in_place_reach_it(routes):  # noqa: F811
    for B, H, Hkv, N, Nk, _ in BATCHED:
        for kw in (dict(selection=TOPK), dict(selection=CDF, sim=0.4), dict(selection=TOPK, pv_f16=1)):
            assert routes(B=B, H=H, Hkv=Hkv, N=N, Nk=Nk, **kw)[4] == 0
    for B, H, Hkv, N, Nk in MASKS:
        assert routes(B=B, H=H, Hkv=Hkv, N=N, Nk=Nk, selection=MASK)[4] == 0
    assert routes(H=40, N=4608, Nk=512, selection=MASK)[4] == 0          # (output over q)
