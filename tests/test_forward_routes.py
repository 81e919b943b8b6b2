"""Which launches a call of the whole operator takes: the rules themselves, on the host (tests/capi_host/routes.cpp).

Queries and keys can differ in number, so a rule about K and V has to hold for any number of Q blocks beside them."""
import os
import subprocess

import pytest
import torch

from spargeattn_amd import _lib, core

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not found")
TOPK, CDF, MASK = 0, 1, 2


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("routes") / "routes")
    r = subprocess.run([HIPCC, "--cuda-host-only", "-x", "hip", "-O1", "-std=c++17", "-Wno-unused-command-line-argument",
                        f"-I{os.path.join(ROOT, 'spargeattn_amd', 'csrc')}", os.path.join(ROOT, "tests", "capi_host", "routes.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]

    def route(B=1, H=1, Hkv=0, N=128, Nk=0, D=128, selection=TOPK, pv_f16=0, sim=-0.1, level=0.5, causal=0, pv=50):
        line = f"{B} {H} {Hkv or H} {N} {Nk or N} {D} {selection} {pv_f16} {sim} {level} {causal} {pv}\n"
        out = subprocess.run([exe], input=line, capture_output=True, text=True, timeout=60)
        assert out.returncode == 0
        return [int(x) for x in out.stdout.split()]
    return route


@pytest.mark.parametrize("kw", [dict(H=24, Nk=512), dict(H=8, Nk=512, B=3), dict(H=36, Nk=400, D=64), dict(H=30, Nk=512, pv_f16=1),
                                dict(H=20, Nk=700, selection=CDF, sim=0.3), dict(H=40, Nk=256, selection=MASK), dict(H=32, Hkv=8, Nk=700)])
def test_short_heads_take_one_launch_up_to_1024_q_blocks(routes, kw):
    """The blocks of Q decide beyond 1024 of them: 24 heads of 32760 queries over 512 keys ran 183.5 us in one launch, 172.6 in two."""
    most = 1024 // (kw.get("B", 1) * kw["H"])
    assert routes(N=128, **kw)[0] == 1
    assert routes(N=128 * most, **kw)[0] == 1
    assert routes(N=128 * most + 1, **kw)[0] == 0
    assert routes(N=32760, **kw)[0] == 0


# heads, queries, keys, head size -> partial sums combined by the back kernel: sixteen chunks of up to 2048 rows have to have blocks
# of Q beside them, and the rows of all heads, which read them, have to be few.  Both sides of each line.
@pytest.mark.parametrize("H,N,Nk,D,kw,combined", [
    (12, 130, 32768, 128, {}, 0), (12, 1280, 20000, 128, {}, 0), (12, 1281, 20000, 128, {}, 1), (11, 20000, 20000, 128, {}, 0),
    (18, 16384, 16384, 128, {}, 1), (18, 16385, 16385, 128, {}, 0), (32, 32768, 32768, 128, {}, 0), (16, 12288, 12288, 128, dict(selection=MASK), 0),
    (16, 128, 8200, 128, {}, 1), (24, 10000, 10000, 128, dict(pv_f16=1), 1), (2, 130, 12287, 128, {}, 1), (40, 130, 8192, 128, {}, 1),
    (16, 128, 9216, 64, {}, 1), (15, 128, 9216, 64, {}, 0), (16, 128, 9217, 64, {}, 0), (16, 3968, 9217, 64, {}, 0), (16, 3969, 9217, 64, {}, 1),
    (12, 12288, 12288, 64, {}, 0), (12, 16384, 16384, 64, {}, 1), (24, 4096, 32768, 64, dict(selection=MASK), 1), (24, 4096, 32769, 64, {}, 0),
    (25, 4096, 32768, 64, {}, 0), (12, 130, 32768, 64, {}, 0), (30, 17776, 17776, 64, {}, 1), (64, 12288, 12288, 64, dict(Hkv=16), 1),
    (64, 12288, 12288, 64, dict(Hkv=8), 0)])
def test_sixteen_chunks_need_queries_beside_them(routes, H, N, Nk, D, kw, combined):
    assert routes(H=H, N=N, Nk=Nk, D=D, **kw)[2] == combined


def test_chunks_hold_every_row_of_a_head(routes):
    for H, Nk, D in ((1, 1, 64), (1, 65, 128), (12, 8193, 128), (24, 10921, 128), (1, 24576, 64), (3, 100000, 128), (3000, 8200, 64)):
        n = routes(H=H, N=512, Nk=Nk, D=D)[1]
        rows = -(-Nk // n)
        assert n >= 1 and n * rows >= Nk and (n - 1) * rows < Nk


@pytest.mark.parametrize("H,N", [(1, 1), (1, 128), (3, 200), (7, 128), (8, 128), (2, 16384)])
@pytest.mark.parametrize("D,pv_f16,long", [(64, 0, 4), (64, 1, 4), (128, 0, 3), (128, 1, 2)])
def test_groups_follow_the_row_not_the_number_of_rows(routes, H, N, D, pv_f16, long):
    groups = [routes(H=H, N=N, Nk=64 * nk, D=D, pv_f16=pv_f16)[3] for nk in (11, 12, 64, 65, 8192)]
    assert groups == [1, 2, 2, long, long]


def test_grids_beyond_one_row_per_cu_have_no_groups(routes):
    assert [routes(H=2, N=n, Nk=20000, D=64)[3] for n in (16384, 16385)] == [4, 1]


# rows x nk, share of the blocks -> in chunks.  Whole rows: the longest is what top-k keeps; a partial last Q block keeps everything.
@pytest.mark.parametrize("kw,chunks", [
    (dict(H=8, N=128, Nk=64 * 132, level=0.2), 0), (dict(H=8, N=128, Nk=64 * 132, level=0.35), 1), (dict(H=8, N=1024, Nk=64 * 132, level=0.5), 1),
    (dict(H=8, N=2048, Nk=64 * 288, level=0.2), 0), (dict(H=8, N=2048, Nk=64 * 288, level=0.5), 1), (dict(H=8, N=22 * 128, Nk=64 * 512, level=1.0), 0),
    (dict(H=8, N=32 * 128, Nk=64 * 512, level=0.5), 0), (dict(N=17776, D=64, selection=CDF), 1), (dict(N=17776, level=0.5), 1), (dict(N=24000, causal=1), 1),
    (dict(N=64 * 257, Nk=64 * 600, level=0.3), 1), (dict(N=8192 * 4, level=0.5), 0), (dict(N=128 * 256 + 1, level=0.5), 1), (dict(N=128 * 257, level=0.5), 0),
    # beyond 256 rows: a partial last Q block only, and not where the rest takes as long
    (dict(H=4, N=17776, D=64, level=0.5), 1), (dict(H=4, N=17776, D=64, level=0.7), 0), (dict(H=4, N=17776, level=0.3), 1), (dict(H=4, N=17776, level=0.5), 0),
    (dict(H=4, N=17792, D=64, level=0.5), 0), (dict(H=8, N=17776, D=64, level=0.15), 1), (dict(H=9, N=17776, D=64, level=0.15), 0), (dict(H=3, N=17776, D=64, selection=MASK), 0),
    (dict(H=2, N=17776, selection=CDF), 1), (dict(H=2, N=17776, D=64, selection=CDF), 1), (dict(H=3, N=17776, D=64, selection=CDF), 0),
    (dict(H=8, N=128, Nk=64 * 128, level=1.0), 0), (dict(H=2, N=128, Nk=64 * 36, selection=MASK), 0),
    # masks: never, since a sparse one loses
    (dict(H=8, N=128, Nk=64 * 128, selection=MASK), 0), (dict(N=12000, D=64, selection=MASK), 0), (dict(H=8, N=1024, Nk=64 * 256, D=64, selection=MASK), 0),
    (dict(H=8, N=1024, Nk=64 * 256, selection=MASK), 0), (dict(N=1024, Nk=64 * 512, D=64, selection=MASK), 0), (dict(N=200, Nk=64 * 300, selection=MASK, pv_f16=1), 0),
    (dict(H=5, N=1665, Nk=64 * 1000, D=64, selection=MASK), 0), (dict(N=33000, D=64, selection=MASK), 0), (dict(N=33024, D=64, selection=MASK), 0),
    (dict(H=4, N=8300, Nk=60000, D=64, selection=MASK), 0)])
def test_few_long_rows_go_over_several_workgroups(routes, kw, chunks):
    assert routes(**kw)[7] == chunks


# A causal selection: the XCD with the last rows of a head has more than its share of the blocks, so chunks pay less than the number of blocks says.
@pytest.mark.parametrize("kw,chunks", [
    (dict(N=16000, level=0.6), 1), (dict(N=22400, level=1.0), 1), (dict(N=25600, level=0.6), 0), (dict(N=25600, level=1.0), 0), (dict(N=25600, D=64, level=1.0), 1),
    (dict(N=32768, level=1.0), 0), (dict(N=32768, D=64, level=1.0), 0), (dict(H=2, N=12800, D=64, level=1.0), 1), (dict(H=2, N=16000, D=64, level=1.0), 0),
    (dict(H=2, N=16000, level=1.0), 0), (dict(N=31950, level=0.35), 1), (dict(N=31950, level=1.0), 0), (dict(N=31950, D=64, level=0.6), 1), (dict(N=31950, D=64, level=1.0), 0),
    (dict(H=4, N=17776, D=64, level=0.6), 1), (dict(H=4, N=17776, D=64, level=1.0), 0), (dict(N=60001, D=64, level=1.0), 0)])
def test_causal_chunks_end_with_the_longest_rows(routes, kw, chunks):
    assert routes(causal=1, **kw)[7] == chunks == routes(causal=1, pv_f16=1, **kw)[7]


def test_rows_of_one_chunk_are_not_cut(routes):
    assert [routes(N=12800, Nk=64 * 1000, level=level)[7] for level in (0.097, 0.1)] == [0, 1]         # 98 blocks to a chunk


# Top-k with a similarity threshold of 0 or more may keep every block: in chunks only where that pays with all of them, too.
@pytest.mark.parametrize("kw,chunks", [
    (dict(H=8, N=17776, D=64, level=0.15), 0), (dict(H=4, N=17776, D=64, level=0.3), 0), (dict(H=6, N=8300, D=64, level=0.15), 0), (dict(H=2, N=17776, D=64, level=0.15), 1),
    (dict(H=8, N=17776, level=0.15), 0), (dict(H=2, N=17776, level=0.15), 1), (dict(N=17776, level=0.15), 1), (dict(N=30000, level=0.15), 0), (dict(N=30000, D=64, level=0.15), 0),
    (dict(N=24001, D=64, level=0.5), 1), (dict(N=24001, D=64, level=0.5, pv_f16=1), 0), (dict(N=24001, level=0.5), 0), (dict(N=28001, D=64, level=0.5, causal=1), 1),
    (dict(H=2, N=17776, level=0.15, pv_f16=1), 0), (dict(H=8, N=1024, Nk=64 * 288, level=0.5), 1), (dict(N=16000, level=0.6, causal=1), 1),
    (dict(N=22400, level=1.0, causal=1), 0)])
def test_a_similarity_threshold_may_keep_everything(routes, kw, chunks):
    assert routes(sim=0.0, **kw)[7] == chunks == routes(sim=0.6, **kw)[7] == routes(sim="nan", **kw)[7]
    assert routes(sim=-0.1, **kw)[7] == 1
    if os.path.exists(_lib.LIB_PATH):           # the stage-by-stage path takes the same route
        shape, causal, pv_f16 = (1, kw.get("H", 1), kw["N"], kw.get("D", 128)), bool(kw.get("causal")), bool(kw.get("pv_f16"))
        for sim, want in ((0.0, chunks), (None, chunks), (-0.1, 1)):
            got = _lib.few_rows_route(shape, kw.get("Nk", kw["N"]), pv_f16, core._selected(None, kw["level"], causal, torch.zeros(2) if sim is None else sim, 50.0))
            assert got[0] == (_lib.ROWS_BY_BLOCKS if want else _lib.ROWS_ONE_WORKGROUP)


# So may a CDF threshold.  (A level per head is a negative share to the rule, as a CDF threshold is.)
@pytest.mark.parametrize("kw,chunks", [
    (dict(N=31595, causal=1), 0), (dict(N=31887, causal=1, pv_f16=1), 0), (dict(N=30000, D=64), 0), (dict(N=24001, D=64), 1), (dict(N=17776), 1), (dict(N=24001), 0),
    (dict(H=2, N=40573, D=64, causal=1), 0), (dict(H=2, N=24001, D=64), 1), (dict(H=2, N=17776, pv_f16=1), 0), (dict(N=24064), 0),
    # whole rows may keep next to nothing
    (dict(N=12800), 0), (dict(N=12800, D=64), 0), (dict(N=9088, causal=1), 0), (dict(N=16000, D=64, causal=1), 0), (dict(H=8, N=1024, Nk=64 * 288), 1),
    (dict(H=8, N=1024, Nk=64 * 287), 0), (dict(H=65, N=128, Nk=64 * 400, D=64), 0), (dict(H=64, N=128, Nk=64 * 400, D=64), 1), (dict(H=2, N=128, Nk=64 * 140, D=64), 0)])
def test_a_cdf_threshold_may_keep_everything(routes, kw, chunks):
    for sim in (-0.1, 0.6):
        assert routes(selection=CDF, sim=sim, **kw)[7] == chunks


def test_workspace_does_not_depend_on_the_level(routes):
    for kw in (dict(H=8, N=128, Nk=64 * 132), dict(N=17776, D=64), dict(H=8, N=2048, Nk=64 * 288, pv_f16=1), dict(H=4, N=17776)):
        assert len({routes(level=level, **kw)[5] for level in (0.05, 0.5, 1.0)}) == 1


# N17776 has a partial last Q block and N17792 has not, which makes 16 queries of difference where there are no chunks
@pytest.mark.parametrize("kw", [dict(H=8, selection=CDF), dict(H=8, selection=MASK), dict(H=4, selection=MASK, D=64), dict(H=3, selection=CDF, D=64, pv_f16=1),
                                dict(H=5, selection=CDF, causal=1)])
def test_no_scratch_where_no_call_is_cut(routes, kw):
    a, b = routes(N=17776, **kw), routes(N=17792, **kw)
    assert a[6] > 1 and a[9] == 0 and a[5] <= b[5]
    a, b = routes(H=2, N=16384), routes(H=2, N=16385)            # whole rows, as many as there are CUs: whatever top-k keeps
    assert a[6] > 1 and a[9] == 0 and a[5] < b[5] - (20 << 20)


def test_scratch_wherever_a_call_is_cut(routes):
    for sel, H, N, Nk, D, causal, pv_f16 in ((TOPK, 8, 17776, 0, 64, 0, 0), (TOPK, 4, 17776, 0, 128, 1, 0), (TOPK, 1, 12800, 0, 64, 1, 0), (TOPK, 1, 26000, 0, 128, 1, 1),
                                             (TOPK, 8, 1024, 64 * 288, 64, 0, 0), (TOPK, 24, 1024, 64 * 288, 128, 0, 0), (TOPK, 3, 30001, 0, 64, 1, 0), (TOPK, 16, 9000, 0, 128, 0, 0),
                                             (TOPK, 12, 12001, 0, 64, 0, 1), (CDF, 1, 17776, 0, 64, 0, 0), (CDF, 2, 17776, 0, 128, 0, 1), (MASK, 8, 1024, 64 * 256, 64, 0, 0),
                                             (MASK, 8, 1024, 64 * 255, 64, 0, 0), (MASK, 1, 17777, 0, 128, 0, 0)):
        cut = {routes(selection=sel, H=H, N=N, Nk=Nk, D=D, causal=causal, pv_f16=pv_f16, level=level, sim=sim)[7]
               for level in (0.0, 0.05, 0.15, 0.3, 0.5, 0.7, 0.9, 1.0, 1.5) for sim in (-0.1, 0.0)}
        assert max(cut) == routes(selection=sel, H=H, N=N, Nk=Nk, D=D, causal=causal, pv_f16=pv_f16)[9], (sel, H, N, Nk, D)


@pytest.mark.parametrize("D,most", [(64, 1536), (128, 1024)])
def test_chunks_of_a_row_are_bounded(routes, D, most):
    for H, N, nk in ((1, 1, 8192), (1, 128, 37), (8, 128, 2048), (1, 17776, 278), (2, 16384, 8192)):
        rows, n = H * -(-N // 128), routes(H=H, N=N, Nk=64 * nk, D=D, selection=MASK)[6]
        assert 1 < n <= 64 and n <= -(-nk // 16) and rows * (n - 1) <= most
    assert routes(H=2, N=128 * 129, Nk=64 * 512, D=D)[6] == routes(H=8, N=128 * 150 + 1, Nk=64 * 512, D=D)[6] == 1
    for H, N, nk in ((2, 16385, 512), (8, 128 * 150 - 1, 8192), (8, 128 * 150 - 1, 129)):
        rows, n = H * -(-N // 128), routes(H=H, N=N, Nk=64 * nk, D=D)[6]
        assert 2 < n <= 64 and n <= -(-nk // 16) and rows * (n - 1) <= 3072


@pytest.mark.parametrize("kw,wgs", [
    (dict(H=4, N=128, Nk=64 * 5), 0), (dict(H=4, N=128, Nk=64 * 6), 4), (dict(H=8, N=1024, Nk=64 * 128), 4), (dict(H=8, N=1024, Nk=64 * 129), 0),
    (dict(H=13, N=640, Nk=64 * 12), 2), (dict(H=13, N=640, Nk=64 * 11), 0), (dict(H=8, N=2048, Nk=64 * 100), 2), (dict(H=8, N=2049, Nk=64 * 100), 0),
    (dict(H=8, N=2048, Nk=64 * 100, pv_f16=1), 0), (dict(H=8, N=2048, Nk=64 * 100, D=64, pv_f16=1), 2), (dict(H=8, N=1024, Nk=64 * 100, pv_f16=1), 4),
    (dict(H=8, N=1024, pv=44.9), 0), (dict(H=8, N=1024, pv=45), 4), (dict(H=8, N=1024, pv=0), 0), (dict(H=8, N=1024, pv="nan"), 0)])
def test_few_short_rows_have_several_workgroups(routes, kw, wgs):
    assert routes(**kw)[8] == wgs
