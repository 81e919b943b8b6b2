"""Rows that have a CU to themselves are worked on by groups of wavefronts that take the row's blocks in turn.

The general kernel (which a call that asks for PV counts gets) walks the same lists block by block.  The groups use the same
running maxima, so the rounded P and the skipped blocks are the same; O and the denominator are summed in another order and
rescaled fewer times: at most a few binary32 roundings per rescaling, 1e-5 of the largest output with margin, and then one
rounding to the output type, which may fall on the other side (one unit in the last place: 2^-10 fp16, 2^-7 bf16)."""
import pytest
import torch

import spargeattn_amd as sa
from spargeattn_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("Nk", [64 * 24 - 9, 64 * 70])
@pytest.mark.parametrize("D,dtype,f16v", [(64, torch.float16, False), (128, torch.bfloat16, False), (64, torch.bfloat16, True),
                                          (128, torch.float16, True)])
def test_groups_equal_the_sequential_walk(D, dtype, f16v, Nk, causal):
    g = torch.Generator().manual_seed(D + Nk)
    B, H, N = 1, 4, 128 * 9 - 5
    nq, nk = 9, (Nk + 63) // 64
    q8 = torch.randint(-127, 128, (B, H, N, D), generator=g, dtype=torch.int8).cuda()
    k8 = torch.randint(-127, 128, (B, H, Nk, D), generator=g, dtype=torch.int8).cuda()
    # scales spread over two decades: maxima that rise late in the list, and blocks far below the running maximum
    qs = (0.01 + 0.03 * torch.rand((B, H, nq), generator=g)).cuda()
    ks = (0.04 * 10 ** (-2 * torch.rand((B, H, nk), generator=g))).cuda()
    # lists of every length around the numbers of groups and ring slots, none and all of the blocks
    lengths = [0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 19, 20, 21, 22, nk - 1] + [nk] * 12
    lut = torch.zeros((B, H, nq, nk), dtype=torch.int32)
    valid = torch.tensor(lengths, dtype=torch.int32).reshape(B, H, nq)
    for h in range(H):
        for i in range(nq):
            cols = torch.randperm(nk, generator=g)[:valid[0, h, i]].sort().values.to(torch.int32)
            lut[0, h, i, :len(cols)] = torch.diff(cols, prepend=torch.zeros(1, dtype=torch.int32))
            lut[0, h, i, len(cols):] = 1000000          # entries behind the list are not used
    lut, valid = lut.cuda(), valid.cuda()
    thr = torch.tensor([50.0, 2.0, 0.5, 0.0], device="cuda")
    v = torch.randn((B, H, Nk, D), generator=g).to(torch.float16).cuda()

    def run(count):
        o = torch.full((B, H, N, D), 7.0, dtype=dtype, device="cuda")
        if f16v:
            return o, _lib.block_sparse_attn_f16v(q8, k8, _lib.v_tiles_f16_swizzled(v), o, lut, valid, thr, qs, ks, D ** -0.5,
                                                  is_causal=causal, return_pv_count=count)
        v8, vs = _lib.v_quant_fp8(v)
        return o, _lib.block_sparse_attn(q8, k8, v8, o, lut, valid, thr, qs, ks, vs, D ** -0.5, is_causal=causal,
                                         return_pv_count=count)

    want, count = run(True)
    got, _ = run(False)
    assert (count.reshape(B, H, nq, 4)[..., 0] < valid).any()          # some blocks are skipped
    assert (got[0, 0, :128] == 7.0).all()                               # a row without blocks stays unwritten
    w, o = want.double(), got.double()
    ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    assert ((o - w).abs() <= ulp * w.abs() + 1e-5 * w.abs().max()).all()
    assert (o - w).norm() <= 3e-4 * w.norm() * (1 if dtype == torch.float16 else 8)


@pytest.mark.parametrize("nk", [64, 65, 128, 129])
def test_long_rows_at_both_sides_of_the_line(nk):
    """D = 128 takes three groups beyond 64 blocks; a row's bits do not depend on how many others the grid holds."""
    test_groups_equal_the_sequential_walk(128, torch.bfloat16, False, 64 * nk - 3, False)
    g = torch.Generator().manual_seed(nk)
    Nk, D = 64 * nk - 3, 128
    q, k, v = (torch.randn((1, 12, n, D), generator=g).bfloat16().cuda() for n in (130, Nk, Nk))
    many = sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=0.7)
    for h in (0, 11):
        few = sa.spas_sage2_attn_meansim_topk_cuda(*(t[:, h:h + 1].contiguous() for t in (q, k, v)), topk=0.7)
        assert torch.equal(few.view(torch.int16), many[:, h:h + 1].view(torch.int16))
