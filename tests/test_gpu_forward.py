"""The whole operator in one native call (spg_sparse_attn) against the same stages launched one by one: same bits.

The stages are checked against the oracle elsewhere; what can go wrong here is which workgroup does what - chunk and role
boundaries, the combination of partial sums, workspace offsets, strides, and where the hyper-parameters come from."""
import pytest
import torch

import spargeattn_amd as sa
from spargeattn_amd import _lib, core
from gpu_common import rand_T

pytestmark = pytest.mark.gpu


def _both(fn):
    whole = fn()
    core._stage_hook = lambda name: None
    try:
        staged = fn()
    finally:
        core._stage_hook = None
    return whole, staged


def _bits(t):
    return t.view(torch.int16)


@pytest.mark.parametrize("Nk", [300, 4096])
def test_ties_and_extreme_levels_in_place(Nk):
    """Equal probabilities (the lower column wins), levels that keep one block, all of them, or nothing but dissimilar ones."""
    q = rand_T((1, 2, 256, 64), torch.float16, 1)
    k = rand_T((1, 2, 1, 64), torch.float16, 2).expand(1, 2, Nk, 64).contiguous()
    k[:, :, 130:200] = rand_T((1, 2, 70, 64), torch.float16, 4)
    v = rand_T((1, 2, Nk, 64), torch.float16, 3)
    for kw in (dict(topk=0.0), dict(topk=1.0), dict(topk=0.5), dict(topk=0.37, is_causal=True), dict(topk=5.0),
               dict(topk=0.2, simthreshd1=0.9)):
        (o, s), (o2, s2) = _both(lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, return_sparsity=True, **kw))
        assert torch.equal(_bits(o), _bits(o2)) and s == s2, kw
    for cdf in (0.0, 0.5, 1.0):
        (o, s), (o2, s2) = _both(lambda: sa.spas_sage2_attn_meansim_cuda(q, k, v, cdfthreshd=cdf, simthreshd1=0.5, return_sparsity=True))
        assert torch.equal(_bits(o), _bits(o2)) and s == s2, cdf


# key/value lengths: one block, the edges of a 64- and a 128-row workgroup, one row more than sixteen full chunks of 64,
# the last length whose rows the attention kernel selects by itself (4096) and the first beyond it, the last whose partial
# results every workgroup combines for itself (8192) and the first beyond it
@pytest.mark.parametrize("Nk", [64, 65, 127, 129, 1025, 4096, 4097, 8192, 8193])
@pytest.mark.parametrize("D,dtype,vdtype", [(128, torch.bfloat16, torch.bfloat16), (64, torch.float16, torch.float16),
                                            (128, torch.float16, torch.bfloat16)])
def test_one_call_equals_the_stages(Nk, D, dtype, vdtype):
    B, H, Hkv, N = 2, 4, 2, 257
    q, k = rand_T((B, H, N, D), dtype, 1), rand_T((B, Hkv, Nk, D), dtype, 2, shift=0.4)
    v = rand_T((B, Hkv, Nk, D), vdtype, 3)
    sim = torch.tensor([0.3, 0.3, -0.1, -0.1], device="cuda")
    level, pv = torch.linspace(0.3, 0.9, H, device="cuda"), torch.tensor([50.0, 3.0, 10.0, 50.0], device="cuda")
    for fn in (lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=0.5, return_sparsity=True),
               lambda: sa.spas_sage2_attn_meansim_cuda(q, k, v, cdfthreshd=level, simthreshd1=sim, pvthreshd=pv, is_causal=True,
                                                       attention_sink=True, qk_quant_gran=2, return_sparsity=True),
               lambda: sa.spas_sage_attn_meansim_topk_cuda(q, k, v, topk=level, simthreshd1=0.2, return_sparsity=True),
               lambda: sa.spas_sage_attn_meansim_cuda(q, k, v, cdfthreshd=0.9, is_causal=Nk == 257, return_sparsity=True)):
        (o, s), (o2, s2) = _both(fn)
        assert torch.equal(_bits(o), _bits(o2)) and s == s2


@pytest.mark.parametrize("nk", [4, 256, 257, 4097])
@pytest.mark.parametrize("kind", [torch.bool, torch.int32, torch.bfloat16])
def test_own_mask_in_one_call(nk, kind):
    """Mask rows up to 4096 blocks are turned into the LUT beside the quantisation, longer ones in a launch of their own."""
    H, N, D = 2, 200, 64
    q, k, v = (rand_T((1, H, n, D), torch.bfloat16, 5 + i) for i, n in enumerate((N, 64 * nk - 3, 64 * nk - 3)))
    mask = (torch.rand((1, H, 2, nk), generator=torch.Generator().manual_seed(nk)) < 0.3).cuda()
    mask[..., 0] = True
    o, o2 = _both(lambda: sa.block_sparse_sage2_attn_cuda(q, k, v, mask_id=mask.to(kind), return_sparsity=True))
    assert torch.equal(_bits(o[0]), _bits(o2[0])) and o[1] == o2[1]


def test_layouts_and_copied_inputs():
    """(B,N,H,D) tensors, slices of a fused QKV tensor, broadcast heads and float32 inputs give what contiguous copies give,
    in the memory layout the stages give it; a second call with the same shapes and other data is independent of the first."""
    B, H, N, D = 1, 3, 300, 64
    fused = rand_T((B, N, 3, H, D), torch.float16, 9)
    q, k, v = (fused[:, :, i] for i in range(3))
    for args in ((q, k, v), (q.contiguous(), k.contiguous(), v.contiguous()), (q.float(), k.float(), v.float()),
                 (q, k[:, :, :1].expand(B, N, H, D), v)):
        o, o2 = _both(lambda: sa.spas_sage2_attn_meansim_topk_cuda(*args, topk=0.4, tensor_layout="NHD"))
        assert o.stride() == o2.stride() and o.dtype == o2.dtype and torch.equal(_bits(o), _bits(o2))
    other = tuple(t.contiguous() * 0.5 for t in (q, k, v))
    o, o2 = _both(lambda: sa.spas_sage2_attn_meansim_topk_cuda(*other, topk=0.4, tensor_layout="NHD"))
    assert torch.equal(_bits(o), _bits(o2))


@pytest.mark.parametrize("H,N,Nk", [(2, 700, 4300), (3, 400, 4200), (9, 4200, 4200), (7, 1000, 1500), (5, 300, 3000)])
def test_reported_sparsity_has_the_same_bits(H, N, Nk):
    """Block counts that are not powers of two: the quotient and the product with the reciprocal differ in the last bit."""
    q, k, v = rand_T((1, H, N, 64), torch.bfloat16, 1), rand_T((1, H, Nk, 64), torch.bfloat16, 2, shift=0.3), rand_T((1, H, Nk, 64), torch.bfloat16, 3)
    mask = (torch.rand((1, H, (N + 127) // 128, (Nk + 63) // 64), generator=torch.Generator().manual_seed(4)) < 0.4).cuda()
    fns = [lambda: sa.block_sparse_sage2_attn_cuda(q, k, v, mask_id=mask, return_sparsity=True)]
    for topk in (0.1, 0.3, 0.5, 0.6):
        fns.append(lambda topk=topk: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=topk, return_sparsity=True))
        fns.append(lambda topk=topk: sa.spas_sage_attn_meansim_topk_cuda(q, k, v, topk=topk, is_causal=N == Nk, return_sparsity=True))
    for fn in fns:
        (_, s), (_, s2) = _both(fn)
        assert s == s2


@pytest.mark.parametrize("H", [1, 3, 8, 9, 17])
@pytest.mark.parametrize("N", [128, 200, 640, 1100])
def test_every_row_is_placed_once(H, N):
    """Workgroups are dealt over eight XCDs with the longest rows of all heads first: every (head, row) pair has to come up
    exactly once, whatever the counts are multiples of.  Without a causal selection only a partial last row is moved; a row
    that is missed would keep the fill value, one that is computed for another would differ."""
    q, k, v = (rand_T((1, H, N, 64), torch.bfloat16, 20 + i) for i in range(3))
    for causal in (False, True):
        o, o2 = _both(lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=0.6, is_causal=causal))
        assert torch.equal(_bits(o), _bits(o2))
        assert torch.isfinite(o.float()).all() and (o != 0).any(-1).all()


@pytest.mark.parametrize("op,H,N,D,causal", [("topk", 31, 16500, 64, False), ("topk", 48, 16384, 64, False), ("topk16", 49, 8300, 128, False),
                                             ("topk", 25, 16500, 128, True), ("topk16", 25, 16384, 128, True), ("mask", 31, 16500, 64, False)])
def test_long_grids_place_every_row_once(op, H, N, D, causal):
    """Grids whose rows are handed out from counters (384 rows per XCD and more, of more than 16384 K-block channels), with counts
    that do and do not divide by eight, and beside the line: the same bits as the stages, whose rows have fixed places."""
    q, k, v = (rand_T((1, 1, N, D), torch.bfloat16, 40 + i).expand(1, H, N, D) * (1 + torch.arange(H, device="cuda").view(1, H, 1, 1) / H).bfloat16()
               for i in range(3))
    mask = (torch.rand((1, H, (N + 127) // 128, (N + 63) // 64), generator=torch.Generator().manual_seed(1)) < 0.1).cuda()
    mask[..., 0] = True
    fn = {"topk": lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=0.2, is_causal=causal),
          "topk16": lambda: sa.spas_sage_attn_meansim_topk_cuda(q, k, v, topk=0.2, is_causal=causal),
          "mask": lambda: sa.block_sparse_sage2_attn_cuda(q, k, v, mask_id=mask)}[op]
    torch.full_like(q, float("nan"))                     # an output row that is missed would not keep the value of an earlier call
    o, o2 = _both(fn)
    assert torch.isfinite(o.float()).all() and torch.equal(_bits(o), _bits(o2))


@pytest.mark.parametrize("Nk", [8193, 12288, 12289])
@pytest.mark.parametrize("D", [64, 128])
def test_few_long_heads_combine_partial_sums(D, Nk):
    """Up to 24576 key/value rows in all, longer heads get 32 chunks that every workgroup adds up (here up to 12288 rows of two
    heads, at D = 64); one row more goes through the launch in between."""
    q = rand_T((1, 2, 130, D), torch.bfloat16, 31)
    k, v = rand_T((1, 2, Nk, D), torch.bfloat16, 32, shift=0.3), rand_T((1, 2, Nk, D), torch.float16, 33)
    for fn in (sa.spas_sage2_attn_meansim_topk_cuda, sa.spas_sage_attn_meansim_topk_cuda):
        o, o2 = _both(lambda: fn(q, k, v, topk=0.3, simthreshd1=0.1))
        assert torch.equal(_bits(o), _bits(o2))


@pytest.mark.parametrize("H,Nk,D", [(1, 24575, 64), (1, 24576, 64), (2, 12287, 128), (1, 12288, 128)])
def test_long_heads_go_through_the_launch_in_between(H, Nk, D):
    """The other end of the same rule: the last length of a head whose partial sums every workgroup adds up (24575 at D = 64,
    12287 at D = 128) and the first beyond it."""
    q = rand_T((1, H, 130, D), torch.float16, 34)
    k, v = rand_T((1, H, Nk, D), torch.float16, 35, shift=0.3), rand_T((1, H, Nk, D), torch.bfloat16, 36)
    for fn in (sa.spas_sage2_attn_meansim_topk_cuda, sa.spas_sage_attn_meansim_topk_cuda):
        o, o2 = _both(lambda: fn(q, k, v, topk=0.3, simthreshd1=0.1))
        assert torch.equal(_bits(o), _bits(o2))


@pytest.mark.parametrize("Nk,D,Hkv", [(1, 64, 1), (1216, 128, 2), (1217, 128, 2), (2432, 64, 2), (2433, 64, 2), (2048, 128, 1), (2049, 128, 1),
                                      (4096, 64, 2), (4097, 64, 2), (250, 64, 40), (250, 64, 42), (700, 128, 16)])
def test_short_heads_in_one_launch(Nk, D, Hkv):
    """Heads of up to 155648 elements (262144 with a similarity threshold) go from the inputs to the selection in one launch whose
    workgroups sum and search the whole head; one row or one head more takes two.  Both sides of each line against the stages, with
    non-finite elements in K and V, strided inputs, and a mask of the caller's own."""
    N, Nk = 140, max(Nk, 128)
    q, k, v = (rand_T((1, n, Hkv, D), torch.bfloat16, 50 + i, shift=0.2).transpose(1, 2) for i, n in enumerate((N, Nk, Nk)))
    k[0, 0, Nk // 2, 3], v[0, 0, Nk - 1, 5], v[0, Hkv - 1, 0, 7] = float("nan"), float("nan"), float("inf")
    mask = (torch.rand((1, Hkv, 2, (Nk + 63) // 64), generator=torch.Generator().manual_seed(Nk)) < 0.5).cuda()
    mask[..., 0] = True
    for fn in (lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=0.4, return_sparsity=True),
               lambda: sa.spas_sage2_attn_meansim_cuda(q, k, v, cdfthreshd=0.8, simthreshd1=0.1, return_sparsity=True,
                                                       qk_quant_gran=2 if D == 128 else 1),
               lambda: sa.spas_sage_attn_meansim_topk_cuda(q, k, v, topk=0.6, return_sparsity=True),
               lambda: sa.block_sparse_sage2_attn_cuda(q, k, v, mask_id=mask, return_sparsity=True)):
        (o, s), (o2, s2) = _both(fn)
        assert torch.equal(_bits(o), _bits(o2)) and s == s2


@pytest.mark.parametrize("H,Nk,D", [(11, 8200, 128), (12, 8200, 128), (12, 32768, 64), (12, 32769, 64)])
def test_many_heads_combine_partial_sums(H, Nk, D):
    """From twelve heads on and up to 32768 rows a head has sixteen chunks that every workgroup adds up; both sides of either line."""
    q = rand_T((1, H, 130, D), torch.bfloat16, 61)
    k, v = rand_T((1, H, Nk, D), torch.bfloat16, 62, shift=0.3), rand_T((1, H, Nk, D), torch.float16, 63)
    for fn in (sa.spas_sage2_attn_meansim_topk_cuda, sa.spas_sage_attn_meansim_topk_cuda):
        o, o2 = _both(lambda: fn(q, k, v, topk=0.3, simthreshd1=0.1))
        assert torch.equal(_bits(o), _bits(o2))


@pytest.mark.parametrize("Nk", [4097, 6000, 8192])
@pytest.mark.parametrize("D", [64, 128])
def test_two_columns_per_lane_in_place(Nk, D):
    """Rows of 65 to 128 blocks are selected by the attention kernel with two columns per lane: equal probabilities on both sides of
    column 64, levels that keep one block, all of them, or nothing but dissimilar ones, in the general kernel and with groups."""
    for H in (2, 130):
        q = rand_T((1, H, 256, D), torch.bfloat16, 71)
        k = rand_T((1, H, 1, D), torch.bfloat16, 72).expand(1, H, Nk, D).contiguous()
        k[:, :, 130:200], k[:, :, 4000:4160] = rand_T((1, H, 70, D), torch.bfloat16, 74), rand_T((1, H, 160, D), torch.bfloat16, 75)[:, :, :Nk - 4000]
        v = rand_T((1, H, Nk, D), torch.bfloat16, 73)
        for kw in (dict(topk=0.0), dict(topk=1.0), dict(topk=0.5), dict(topk=0.37, is_causal=True), dict(topk=0.2, simthreshd1=0.9),
                   dict(topk=0.3, attention_sink=True)):
            (o, s), (o2, s2) = _both(lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, return_sparsity=True, **kw))
            assert torch.equal(_bits(o), _bits(o2)) and s == s2, (H, kw)
        for cdf in (0.0, 0.5, 0.97, 1.0):
            (o, s), (o2, s2) = _both(lambda: sa.spas_sage2_attn_meansim_cuda(q, k, v, cdfthreshd=cdf, simthreshd1=0.5, return_sparsity=True))
            assert torch.equal(_bits(o), _bits(o2)) and s == s2, (H, cdf)


@pytest.mark.parametrize("N", [16384, 16385])
@pytest.mark.parametrize("D", [64, 128])
def test_many_queries_over_short_heads(N, D):
    """1024 Q blocks over short heads are the last that go through one launch in front of the attention; one row more takes two."""
    q = rand_T((1, 8, N, D), torch.bfloat16, 81)
    k, v = rand_T((1, 8, 500, D), torch.bfloat16, 82, shift=0.3), rand_T((1, 8, 500, D), torch.float16, 83)
    for fn in (lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=0.3, return_sparsity=True),
               lambda: sa.spas_sage_attn_meansim_cuda(q, k, v, cdfthreshd=0.8, simthreshd1=0.1, return_sparsity=True)):
        (o, s), (o2, s2) = _both(fn)
        assert torch.equal(_bits(o), _bits(o2)) and s == s2


@pytest.mark.parametrize("H,N,Nk,D", [(12, 1280, 8300, 128), (12, 1281, 8300, 128), (12, 1281, 24576, 128), (12, 1281, 24577, 128), (16, 130, 9216, 64),
                                      (16, 130, 9217, 64), (16, 3968, 9300, 64), (16, 3969, 9300, 64), (24, 2700, 32768, 64), (24, 2700, 32769, 64)])
def test_many_heads_with_queries_beside_them(H, N, Nk, D):
    """Both sides of the lines from which on sixteen chunks a head are combined by every workgroup of the back kernel."""
    q = rand_T((1, H, N, D), torch.bfloat16, 91)
    k, v = rand_T((1, H, Nk, D), torch.bfloat16, 92, shift=0.3), rand_T((1, H, Nk, D), torch.float16, 93)
    for fn in (sa.spas_sage2_attn_meansim_topk_cuda, sa.spas_sage_attn_meansim_topk_cuda):
        o, o2 = _both(lambda: fn(q, k, v, topk=0.1))
        assert torch.equal(_bits(o), _bits(o2))


# partial sums combined by the back kernel, and by a launch of their own; a tail of one row, an odd number of blocks; 512 and 256 threads
@pytest.mark.parametrize("H,N,Nk,D", [(2, 200, 3000, 128), (4, 300, 8321, 128), (30, 2049, 1601, 128), (3, 200, 3009, 64), (26, 1300, 8260, 64)])
@pytest.mark.parametrize("vdtype", [torch.float16, torch.bfloat16])
def test_fp16_tiles_beside_the_blocks_of_k(H, N, Nk, D, vdtype):
    """V^T tiles come from the launch that quantises K, with a selection and with a mask: the stages' bits, and the same for all blocks."""
    q, k, v = rand_T((1, H, N, D), vdtype, 50), rand_T((1, H, Nk, D), vdtype, 51, shift=0.4), rand_T((1, H, Nk, D), vdtype, 52)
    o, o2 = _both(lambda: sa.spas_sage_attn_meansim_topk_cuda(q, k, v, topk=1.0))
    assert torch.equal(_bits(o), _bits(o2))
    mask = torch.ones((1, H, (N + 127) // 128, (Nk + 63) // 64), dtype=torch.bool, device="cuda")
    got = torch.empty_like(q)
    plan = _lib.ForwardPlan(q, k, v, got, mask, _lib.SELECT_MASK, True, False, False, False, 1, D ** -0.5)
    plan.run(q, k, v, got, mask, 0.0, 0.0, 50.0)
    if _lib.few_rows_route(q.shape, Nk, True, (_lib.SELECT_TOPK, 1.0, False, 50.0)) == _lib.few_rows_route(q.shape, Nk, True, (_lib.SELECT_MASK, None, False, 50.0)):
        assert torch.equal(_bits(got), _bits(o))
    else:
        # few long rows: cut into chunks where top-k names the share, not with a mask, whose density is not known.  The same P are summed in another order: a
        # few binary32 roundings, 1e-5 of the largest output with margin, and one rounding to the output type that may fall on the other side
        assert (H, N, Nk) == (4, 300, 8321)
        a, b = got.double(), o.double()
        assert ((a - b).abs() <= (2.0 ** -10 if vdtype == torch.float16 else 2.0 ** -7) * b.abs() + 1e-5 * b.abs().max()).all()


def test_interrupted_wait_for_counts(monkeypatch):
    """A call that is interrupted while it waits for its counts ends only after the kernels that store them."""
    q, k, v = (rand_T((1, 8, 8192, 128), torch.bfloat16, s) for s in (1, 2, 3))
    call = lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, return_sparsity=True)  # noqa: E731
    out, sparsity = call()

    class Interrupted:
        def __getattr__(self, name):
            return getattr(_lib.load(), name)

        def spg_wait_counts(self, *args):
            raise KeyboardInterrupt
    for plan in core._plans.values():
        monkeypatch.setattr(plan, "_lib", Interrupted())
    torch.cuda.synchronize()
    with pytest.raises(KeyboardInterrupt):
        call()
    assert torch.cuda.current_stream().query()
    monkeypatch.undo()
    again, sparsity2 = call()
    assert torch.equal(_bits(out), _bits(again)) and sparsity == sparsity2


@pytest.mark.parametrize("op,kw", [(sa.spas_sage2_attn_meansim_topk_cuda, dict(topk=0.4)), (sa.spas_sage2_attn_meansim_cuda, dict(cdfthreshd=0.9, simthreshd1=0.2))])
def test_counts_under_a_default_device(op, kw):
    """A program that makes its tensors on the GPU by default (torch.set_default_device) gets its sparsity as any other."""
    q, k, v = (rand_T((1, 3, 1000, 64), torch.float16, s) for s in (1, 2, 3))
    o, sparsity = op(q, k, v, return_sparsity=True, **kw)
    with torch.device("cuda"):
        o2, sparsity2 = op(q, k, v, return_sparsity=True, **kw)
    assert torch.equal(_bits(o), _bits(o2)) and sparsity == sparsity2


def test_counts_behind_queued_work():
    """Counts that do not come within the time that the host looks for them."""
    q, k, v = (rand_T((1, 3, 1000, 64), torch.float16, s) for s in (1, 2, 3))
    call = lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=0.4, return_sparsity=True)  # noqa: E731
    o, sparsity = call()
    torch.cuda._sleep(50_000_000)                       # some 20 ms
    o2, sparsity2 = call()
    assert torch.equal(_bits(o), _bits(o2)) and sparsity == sparsity2
