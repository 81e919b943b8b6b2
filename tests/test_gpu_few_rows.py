"""Few short rows: the queries of a row go over several workgroups and its blocks over the wavefronts of each.

The general kernel (which a call that asks for PV counts gets) walks the same lists block by block.  P is rounded against the same running
maxima; O and the denominator are summed per group of blocks: at most a few binary32 roundings, 1e-5 of the largest output with margin, and
then one rounding to the output type, which may fall on the other side (one unit in the last place: 2^-10 fp16, 2^-7 bf16)."""
import pytest
import torch

import spargeattn_amd as sa
from spargeattn_amd import _lib, core

pytestmark = pytest.mark.gpu


# heads, queries, K blocks: four workgroups to a row and two, whole and partial Q blocks, quarters without a row, one block to all 128
@pytest.mark.parametrize("H,N,nk", [(4, 1147, 6), (4, 1044, 40), (2, 300, 128), (8, 1300, 64), (8, 2043, 12), (8, 1928, 128)])
@pytest.mark.parametrize("D,dtype,f16v,gran,causal", [(64, torch.float16, False, 1, True), (128, torch.bfloat16, False, 2, False),
                                                      (128, torch.float16, False, 1, True), (64, torch.bfloat16, True, 2, False), (128, torch.float16, True, 1, True)])
def test_equal_the_sequential_walk(D, dtype, f16v, gran, causal, H, N, nk):
    g = torch.Generator().manual_seed(D + nk)
    B, nq, Nk, Hkv = 1, (N + 127) // 128, 64 * nk - 9, H // 2
    selected = (_lib.SELECT_MASK, None, False, 50.0)
    if _lib.few_rows_route((B, H, N, D), Nk, f16v, selected)[0] != _lib.ROWS_BY_QUERIES:
        assert f16v and D == 128 and H * nq > 64
        pytest.skip("FP16 PV at D = 128: up to 64 rows")
    q8 = torch.randint(-127, 128, (B, H, N, D), generator=g, dtype=torch.int8).cuda()
    k8 = torch.randint(-127, 128, (B, Hkv, Nk, D), generator=g, dtype=torch.int8).cuda()
    # scales spread over two decades: maxima that rise late in the list, blocks far below the running maximum, both forms of the exponent
    qs = (0.01 + 0.03 * torch.rand((B, H, nq * (4 if gran == 2 else 1)), generator=g)).cuda()
    ks = (0.04 * 10 ** (-2 * torch.rand((B, Hkv, nk), generator=g))).cuda()
    # lists of every length around the numbers of groups, none and all of the blocks
    lengths = [min(n, nk) for n in (0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 15, 16, 17, 25, 63, 64, 65, 66, nk - 1, nk)]
    lut = torch.zeros((B, H, nq, nk), dtype=torch.int32)
    valid = torch.tensor((lengths * (H * nq))[:H * nq], dtype=torch.int32).reshape(B, H, nq)
    for h in range(H):
        for i in range(nq):
            cols = torch.randperm(nk, generator=g)[:valid[0, h, i]].sort().values.to(torch.int32)
            lut[0, h, i, :len(cols)] = torch.diff(cols, prepend=torch.zeros(1, dtype=torch.int32))
            lut[0, h, i, len(cols):] = 1000000          # entries behind the list are not used
    lut, valid = lut.cuda(), valid.cuda()
    thr = torch.full((H,), 50.0, device="cuda")
    v = torch.randn((B, Hkv, Nk, D), generator=g).to(torch.float16).cuda()

    def run(count):
        o = torch.full((B, H, N, D), 7.0, dtype=dtype, device="cuda")
        if f16v:
            return o, _lib.block_sparse_attn_f16v(q8, k8, _lib.v_tiles_f16_swizzled(v), o, lut, valid, thr, qs, ks, D ** -0.5,
                                                  is_causal=causal, return_pv_count=count, qk_quant_gran=gran, selected=selected)
        v8, vs = _lib.v_quant_fp8(v)
        return o, _lib.block_sparse_attn(q8, k8, v8, o, lut, valid, thr, qs, ks, vs, D ** -0.5, is_causal=causal,
                                         return_pv_count=count, qk_quant_gran=gran, selected=selected)

    want, _ = run(True)
    got, _ = run(False)
    assert (got[0, 0, :128] == 7.0).all()                               # a row without blocks stays unwritten
    w, o = want.double(), got.double()
    ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    assert ((o - w).abs() <= ulp * w.abs() + 1e-5 * w.abs().max()).all()
    assert (o - w).norm() <= 3e-4 * w.norm() * (1 if dtype == torch.float16 else 8)


# four workgroups to a row and two; the smallest threshold of the route and the usual one
@pytest.mark.parametrize("H,N,nk", [(2, 256, 9), (8, 1920, 30)])
@pytest.mark.parametrize("D,f16v", [(64, False), (128, False), (64, True), (128, True)])
@pytest.mark.parametrize("thr", [45.0, 50.0])
def test_a_skipped_block_is_not_touched(D, f16v, thr, H, N, nk):
    """What stands in V of a block that the PV threshold skips for every query, or a K scale that is not finite, changes nothing, as in the walk."""
    g = torch.Generator().manual_seed(nk)
    B, nq, Nk = 1, (N + 127) // 128, 64 * nk
    selected = (_lib.SELECT_MASK, None, False, thr)
    if _lib.few_rows_route((B, H, N, D), Nk, f16v, selected)[0] != _lib.ROWS_BY_QUERIES:
        assert f16v and D == 128 and H * nq > 64
        pytest.skip("FP16 PV at D = 128: up to 64 rows")
    # scores of blocks 0, 4, 8, ... are 0.002 * 64 * 60^2 * 0.125 * log2(e) = 83 (D = 128: 117) to 5 % more, those of the others minus as much
    q8 = torch.randint(60, 62, (B, H, N, D), generator=g, dtype=torch.int8)
    k8 = torch.randint(60, 62, (B, H, Nk, D), generator=g, dtype=torch.int8)
    sign = torch.where(torch.arange(nk) % 4 == 0, 1, -1).to(torch.int8).repeat_interleave(64)
    k8 *= sign[None, None, :, None]
    qs, ks = torch.full((B, H, nq), 0.1), torch.full((B, H, nk), 0.02)
    v = torch.randn((B, H, Nk, D), generator=g).to(torch.float16)
    v[:, :, 64 * 1 + 3, 5] = float("nan")
    if f16v:                                            # (with FP8 PV an infinity is the scale of its channel)
        v[:, :, 64 * 2 + 60, 1] = float("inf")
        v[:, 0, 64 * 5] = float("-inf")
    ks[:, :, 6], k8[:, :, 64 * 6:64 * 7] = float("inf"), 0            # (what a block with an infinity in it is quantised to)
    q8, k8, qs, ks, v = (t.cuda() for t in (q8, k8, qs, ks, v))
    lut, valid = torch.ones((B, H, nq, nk), dtype=torch.int32), torch.full((B, H, nq), nk, dtype=torch.int32)
    lut[..., 0] = 0
    lut, valid, pv = lut.cuda(), valid.cuda(), torch.full((H,), thr, device="cuda")

    def run(count):
        o = torch.empty((B, H, N, D), dtype=torch.float16, device="cuda")
        if f16v:
            return o, _lib.block_sparse_attn_f16v(q8, k8, _lib.v_tiles_f16_swizzled(v), o, lut, valid, pv, qs, ks, D ** -0.5,
                                                  return_pv_count=count, selected=selected)
        v8, vs = _lib.v_quant_fp8(v)
        return o, _lib.block_sparse_attn(q8, k8, v8, o, lut, valid, pv, qs, ks, vs, D ** -0.5, return_pv_count=count, selected=selected)

    want, count = run(True)
    got, _ = run(False)
    # blocks 0, 4, 8, ... and the last two of the row
    assert (count == len({b for b in range(nk) if b % 4 == 0} | {nk - 2, nk - 1})).all() and want.isfinite().all()
    w, o = want.double(), got.double()
    assert ((o - w).abs() <= 2.0 ** -10 * w.abs() + 1e-5 * w.abs().max()).all()


@pytest.mark.parametrize("H,N,Nk", [(3, 129, 64 * 6), (3, 700, 64 * 64 - 3), (2, 1025, 64 * 65), (9, 1025, 64 * 128 - 1), (2, 128, 64 * 100)])
@pytest.mark.parametrize("D,f16v", [(64, False), (128, False), (64, True), (128, True)])
def test_selection_in_place_equals_the_stages(D, f16v, H, N, Nk):
    g = torch.Generator().manual_seed(N)
    q, k, v = (torch.randn((1, H, n, D), generator=g).bfloat16().cuda().transpose(1, 2).contiguous() for n in (N, Nk, Nk))
    topk = sa.spas_sage_attn_meansim_topk_cuda if f16v else sa.spas_sage2_attn_meansim_topk_cuda
    cdf = sa.spas_sage_attn_meansim_cuda if f16v else sa.spas_sage2_attn_meansim_cuda
    for fn in (lambda: topk(q, k, v, topk=0.4, tensor_layout="NHD", return_sparsity=True),
               lambda: cdf(q, k, v, cdfthreshd=0.9, simthreshd1=0.1, attention_sink=True, tensor_layout="NHD", is_causal=N == Nk, qk_quant_gran=2, return_sparsity=True)):
        o, s = fn()
        core._stage_hook = lambda name: None
        try:
            o2, s2 = fn()
        finally:
            core._stage_hook = None
        assert s == s2
        assert torch.equal(o.view(torch.int16), o2.view(torch.int16))
