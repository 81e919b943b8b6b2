"""Few long rows go over several workgroups, each with a stretch of the row's list.

The general kernel (which a call that asks for PV counts gets) walks the same lists block by block.  The chunks start from the same running
maxima, so the rounded P and the skipped blocks are the same; O and the denominator are summed per chunk and rescaled once more: at most a few
binary32 roundings, 1e-5 of the largest output with margin, and then one rounding to the output type, which may fall on the other
side (one unit in the last place: 2^-10 fp16, 2^-7 bf16)."""
import pytest
import torch

import spargeattn_amd as sa
from gpu_common import tag_of, to_np
from oracle import api as oapi, attention as oat
from spargeattn_amd import _lib

pytestmark = pytest.mark.gpu


def lists(B, H, nq, nk, lengths, g):
    lut = torch.zeros((B, H, nq, nk), dtype=torch.int32)
    valid = torch.tensor((lengths * (B * H * nq))[:B * H * nq], dtype=torch.int32).reshape(B, H, nq)
    for h in range(H):
        for i in range(nq):
            cols = torch.randperm(nk, generator=g)[:valid[0, h, i]].sort().values.to(torch.int32)
            lut[0, h, i, :len(cols)] = torch.diff(cols, prepend=torch.zeros(1, dtype=torch.int32))
            lut[0, h, i, len(cols):] = 1000000          # entries behind the list are not used
    return lut.cuda(), valid.cuda()


# heads, Q blocks, K blocks, what is said of the lists: chunks of 16 blocks, and of more where rows are many or long (beyond 256 rows, and at their most)
@pytest.mark.parametrize("H,nq,nk,share", [(4, 9, 129, 1.0), (4, 9, 300, 1.0), (8, 27, 150, 0.05), (1, 2, 1100, 0.9), (8, 33, 150, 0.05), (8, 150, 141, 0.05)])
@pytest.mark.parametrize("D,dtype,f16v,gran,causal", [(64, torch.float16, False, 1, True), (128, torch.bfloat16, False, 2, False), (64, torch.bfloat16, True, 2, False),
                                                      (128, torch.float16, True, 1, True)])
def test_chunks_equal_the_sequential_walk(D, dtype, f16v, gran, causal, H, nq, nk, share):
    g = torch.Generator().manual_seed(D + nk)
    B, N, Nk, Hkv = 1, 128 * nq - 5, 64 * nk - 9, H // 2 if H > 1 else 1
    q8 = torch.randint(-127, 128, (B, H, N, D), generator=g, dtype=torch.int8).cuda()
    k8 = torch.randint(-127, 128, (B, Hkv, Nk, D), generator=g, dtype=torch.int8).cuda()
    # scales spread over two decades: maxima that rise late in the list, and blocks far below the running maximum
    qs = (0.01 + 0.03 * torch.rand((B, H, nq * (4 if gran == 2 else 1)), generator=g)).cuda()
    ks = (0.04 * 10 ** (-2 * torch.rand((B, Hkv, nk), generator=g))).cuda()
    # lists of every length around one and a few chunks, none and all of the blocks
    lut, valid = lists(B, H, nq, nk, [0, 1, 2, 3, 15, 16, 17, 18, 31, 32, 33, 34, 47, 48, 49, 64, 65, 97, nk - 1, nk], g)
    thr = torch.tensor([50.0, 2.0, 0.5, 0.0] * 2, device="cuda")[:H].contiguous()
    v = torch.randn((B, Hkv, Nk, D), generator=g).to(torch.float16).cuda()
    selected = (_lib.SELECT_TOPK, share, False, None)
    assert _lib.few_rows_route(q8.shape, Nk, f16v, selected)[0] == _lib.ROWS_BY_BLOCKS

    def run(count):
        o = torch.full((B, H, N, D), 7.0, dtype=dtype, device="cuda")
        if f16v:
            return o, _lib.block_sparse_attn_f16v(q8, k8, _lib.v_tiles_f16_swizzled(v), o, lut, valid, thr, qs, ks, D ** -0.5,
                                                  is_causal=causal, return_pv_count=count, qk_quant_gran=gran, selected=selected)
        v8, vs = _lib.v_quant_fp8(v)
        return o, _lib.block_sparse_attn(q8, k8, v8, o, lut, valid, thr, qs, ks, vs, D ** -0.5, is_causal=causal,
                                         return_pv_count=count, qk_quant_gran=gran, selected=selected)

    want, count = run(True)
    got, _ = run(False)
    if H > 1:
        assert (count.reshape(B, H, nq, 4)[..., 0] < valid).any()      # some blocks are skipped
    assert (got[0, 0, :128] == 7.0).all()                               # a row without blocks stays unwritten
    w, o = want.double(), got.double()
    ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    assert ((o - w).abs() <= ulp * w.abs() + 1e-5 * w.abs().max()).all()
    assert (o - w).norm() <= 3e-4 * w.norm() * (1 if dtype == torch.float16 else 8)


@pytest.mark.parametrize("D,dtype,f16v", [(64, torch.bfloat16, False), (128, torch.float16, False), (64, torch.float16, True), (128, torch.bfloat16, True)])
def test_chunks_of_batches_write_by_strides(D, dtype, f16v):
    """Two batches, grouped heads, an output laid out (B, N, heads, D) with a head more than the call has: the walk's values, and nothing beside them."""
    g = torch.Generator().manual_seed(D)
    B, H, Hkv, nq, nk = 2, 4, 2, 5, 200
    N, Nk = 128 * nq - 100, 64 * nk - 1
    q8 = torch.randint(-127, 128, (B, H, N, D), generator=g, dtype=torch.int8).cuda()
    k8 = torch.randint(-127, 128, (B, Hkv, Nk, D), generator=g, dtype=torch.int8).cuda()
    qs, ks = (0.01 + 0.03 * torch.rand((B, H, nq), generator=g)).cuda(), (0.04 * 10 ** (-2 * torch.rand((B, Hkv, nk), generator=g))).cuda()
    per_batch = [lists(1, H, nq, nk, [17, nk, 0, 33, 64, 16, 97, 150, 1], g) for _ in range(B)]
    lut, valid = (torch.cat(t) for t in zip(*per_batch))
    thr, v = torch.full((H,), 50.0, device="cuda"), torch.randn((B, Hkv, Nk, D), generator=g).to(torch.float16).cuda()
    selected = (_lib.SELECT_TOPK, 1.0, False, None)
    assert _lib.few_rows_route(q8.shape, Nk, f16v, selected)[0] == _lib.ROWS_BY_BLOCKS

    def run(count, o):
        if f16v:
            return _lib.block_sparse_attn_f16v(q8, k8, _lib.v_tiles_f16_swizzled(v), o, lut, valid, thr, qs, ks, D ** -0.5, return_pv_count=count, selected=selected)
        v8, vs = _lib.v_quant_fp8(v)
        return _lib.block_sparse_attn(q8, k8, v8, o, lut, valid, thr, qs, ks, vs, D ** -0.5, return_pv_count=count, selected=selected)

    want = torch.full((B, H, N, D), 7.0, dtype=dtype, device="cuda")
    run(True, want)
    whole = torch.full((B, N, H + 1, D), 7.0, dtype=dtype, device="cuda")
    got = whole[:, :, :H].transpose(1, 2)
    run(False, got)
    assert (whole[:, :, H] == 7.0).all()
    empty = (valid == 0).repeat_interleave(128, 2)[:, :, :N]
    assert empty.any() and (got[empty] == 7.0).all()
    w, o = want.double(), got.double()
    ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    assert ((o - w).abs() <= ulp * w.abs() + 1e-5 * w.abs().max()).all()


@pytest.mark.parametrize("D,dtype,sage1,gran", [(64, torch.bfloat16, False, 2), (128, torch.float16, False, 1), (64, torch.float16, True, 1), (128, torch.bfloat16, True, 2)])
@pytest.mark.parametrize("mode", ["topk", "cdf"])
def test_cut_rows_against_the_oracle(D, dtype, sage1, gran, mode):
    """The operator on a call whose rows are cut, from selection to output, two batches and an (B, N, H, D) layout."""
    g = torch.Generator().manual_seed(D + gran)
    B, H, Hkv, Nq, Nk = 2, 2, 1, 200, 64 * 150 - 7
    q, k, v = (torch.randn((B, h, n, D), generator=g).to(dtype) for h, n in ((H, Nq), (Hkv, Nk), (Hkv, Nk)))
    level, sim = (0.6, -0.1) if mode == "topk" else (0.7, 0.3)
    assert _lib.few_rows_route(q.shape, Nk, sage1, (_lib.SELECT_TOPK if mode == "topk" else _lib.SELECT_CDF, level if mode == "topk" else None, False, 20.0, sim))[0] == _lib.ROWS_BY_BLOCKS
    want = (oapi.spas_sage_attn_meansim_topk if sage1 else oapi.spas_sage2_attn_meansim_topk)(
        to_np(q), to_np(k), to_np(v), tag_of(dtype), simthreshd1=sim, pvthreshd=20.0, qk_quant_gran=gran,
        **(dict(topk=level, cdfthreshd=None) if mode == "topk" else dict(topk=None, cdfthreshd=level)))
    op = {("topk", False): sa.spas_sage2_attn_meansim_topk_cuda, ("cdf", False): sa.spas_sage2_attn_meansim_cuda,
          ("topk", True): sa.spas_sage_attn_meansim_topk_cuda, ("cdf", True): sa.spas_sage_attn_meansim_cuda}[mode, sage1]
    o, sparsity = op(*(t.transpose(1, 2).contiguous().cuda() for t in (q, k, v)), simthreshd1=sim, pvthreshd=20.0, qk_quant_gran=gran, tensor_layout="NHD",
                     return_sparsity=True, **{"topk" if mode == "topk" else "cdfthreshd": level})
    assert abs(sparsity - want["sparsity"]) < 1e-6
    met = oat.precision_metric(to_np(o.transpose(1, 2)), want["out"])
    assert met["Cossim"] >= 0.999 and met["L1"] <= 1e-2, met


@pytest.mark.parametrize("level", [0.2, 0.9])
def test_a_captured_call_replays(level):
    """Scratch of the chunks is written anew by every replay."""
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn((1, 4, n, 64), generator=g).bfloat16().cuda() for n in (300, 64 * 200 - 3, 64 * 200 - 3))
    want = [sa.spas_sage2_attn_meansim_topk_cuda(s * q, k, v, topk=level) for s in (1, 2, 3)]
    static = q.clone()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        sa.spas_sage2_attn_meansim_topk_cuda(static, k, v, topk=level)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = sa.spas_sage2_attn_meansim_topk_cuda(static, k, v, topk=level)
    for s in (2, 1, 3, 2):
        static.copy_(s * q)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want[s - 1].view(torch.int16))
        sa.spas_sage2_attn_meansim_topk_cuda(3 * q, k, v, topk=0.5)
