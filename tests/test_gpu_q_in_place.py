"""Q quantised, and pooled for a selection in place, by the attention kernel's own workgroups: same bits as the stages one by one.

Grids around the line where the route changes, partial last Q blocks of one row, 32-row groups without rows, tensors that are read through
strides, thresholds that need the normalised rows, blocks with zero rows, NaN and infinities."""
import pytest
import torch

import spargeattn_amd as sa
from spargeattn_amd import _lib
from test_gpu_forward import _both, _bits
from gpu_common import rand_T

pytestmark = pytest.mark.gpu


def _qkv(H, Hkv, N, Nk, D, dtype, nhd, seed):
    q, k, v = rand_T((1, H, N, D), dtype, seed), rand_T((1, Hkv, Nk, D), dtype, seed + 1, shift=0.4), rand_T((1, Hkv, Nk, D), dtype, seed + 2)
    q = q * torch.linspace(0.01, 2.0, N, device="cuda")[:, None].to(dtype)          # 32-row groups of different magnitude
    q[:, :, N // 2:N // 2 + 130] = (q[:, :, :1] + 0.05 * q[:, :, N // 2:N // 2 + 130]).to(dtype)      # similar blocks
    if H > 3 and N > 300:
        q[:, 1, 5] = 0.0
        q[:, 2, 140, 3] = float("nan")
        q[:, 3, 270, 7] = float("inf")
    return [t.transpose(1, 2).contiguous() if nhd else t for t in (q, k, v)]


# D = 128, more than 576 rows of Q blocks; the first has exactly as many and is quantised in front
@pytest.mark.parametrize("H,N,Nk,D", [(36, 2048, 700, 128), (48, 1537, 64, 128), (34, 2049, 1000, 128), (74, 1024, 4096, 128), (54, 1313, 4097, 128),
                                      (64, 2049, 300, 64)])
@pytest.mark.parametrize("dtype,gran,nhd", [(torch.bfloat16, 1, False), (torch.float16, 2, True)])
def test_selection_in_place(H, N, Nk, D, dtype, gran, nhd):
    q, k, v = _qkv(H, H // 2, N, Nk, D, dtype, nhd, N)
    kw = dict(qk_quant_gran=gran, tensor_layout="NHD" if nhd else "HND", return_sparsity=True)
    sim = torch.tensor([0.3, -0.1], device="cuda").repeat_interleave(2).repeat((H + 3) // 4)[:H].contiguous()
    for fn in (lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=0.4, **kw),
               lambda: sa.spas_sage2_attn_meansim_cuda(q, k, v, cdfthreshd=0.8, simthreshd1=0.4, attention_sink=True, **kw),
               lambda: sa.spas_sage2_attn_meansim_cuda(q, k, v, cdfthreshd=0.9, simthreshd1=sim, **kw),
               lambda: sa.spas_sage_attn_meansim_topk_cuda(q, k, v, topk=0.3, **kw)):
        (o, s), (o2, s2) = _both(fn)
        assert torch.equal(_bits(o), _bits(o2)) and s == s2


@pytest.mark.parametrize("H,N,Nk,D", [(11, 4096, 700, 128), (11, 4097, 700, 128), (45, 1024, 9000, 128), (3, 16400, 64, 128)])     # 352 rows and more
@pytest.mark.parametrize("dtype,gran,nhd", [(torch.bfloat16, 2, False), (torch.float16, 1, True)])
def test_own_mask(H, N, Nk, D, dtype, gran, nhd):
    q, k, v = _qkv(H, H, N, Nk, D, dtype, nhd, N)
    nq, nk = -(-N // 128), -(-Nk // 64)
    mask = (torch.rand((1, H, nq, nk), generator=torch.Generator().manual_seed(N)) < 0.4).cuda()
    mask[..., 0] = True
    o, o2 = _both(lambda: sa.block_sparse_sage2_attn_cuda(q, k, v, mask_id=mask, qk_quant_gran=gran, tensor_layout="NHD" if nhd else "HND"))
    assert torch.equal(_bits(o), _bits(o2))


# B, H, Hkv, N, Nk, causal: two batch entries and grouped heads, one and two columns per lane of the selection, partial last blocks on both sides
BATCHED = [(2, 24, 8, 1600, 1600, True), (2, 5, 5, 8000, 8000, True), (2, 10, 2, 4200, 4200, True), (2, 26, 13, 1537, 2500, False), (2, 9, 3, 4225, 6000, False)]


@pytest.mark.parametrize("B,H,Hkv,N,Nk,causal", BATCHED)
@pytest.mark.parametrize("dtype,gran,nhd", [(torch.bfloat16, 1, True), (torch.float16, 2, False)])
def test_batched_and_causal(B, H, Hkv, N, Nk, causal, dtype, gran, nhd):
    parts = [_qkv(H, Hkv, N, Nk, 128, dtype, nhd, 17 * b + N) for b in range(B)]
    q, k, v = (torch.cat(t) for t in zip(*parts))
    kw = dict(qk_quant_gran=gran, tensor_layout="NHD" if nhd else "HND", return_sparsity=True, is_causal=causal)
    for kernel_causal in ((False, True) if causal else (False,)):
        for fn in (lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=0.4, kernel_causal=kernel_causal, **kw),
                   lambda: sa.spas_sage2_attn_meansim_cuda(q, k, v, cdfthreshd=0.8, simthreshd1=0.4, kernel_causal=kernel_causal, **kw)):
            (o, s), (o2, s2) = _both(fn)
            assert torch.equal(_bits(o), _bits(o2)) and s == s2
    (o, s), (o2, s2) = _both(lambda: sa.spas_sage_attn_meansim_topk_cuda(q, k, v, topk=0.3, **kw))
    assert torch.equal(_bits(o), _bits(o2)) and s == s2


# B, H, Hkv, N, Nk: few heads of K, and many of them
MASKS = [(1, 11, 11, 4097, 1100), (2, 4, 4, 6017, 2000), (1, 3, 3, 16400, 1300), (2, 32, 16, 1537, 2000), (1, 62, 62, 1024, 9000)]


@pytest.mark.parametrize("B,H,Hkv,N,Nk", MASKS)
@pytest.mark.parametrize("dtype,gran,nhd", [(torch.bfloat16, 2, False), (torch.float16, 1, True)])
def test_batched_masks(B, H, Hkv, N, Nk, dtype, gran, nhd):
    parts = [_qkv(H, Hkv, N, Nk, 128, dtype, nhd, 19 * b + N) for b in range(B)]
    q, k, v = (torch.cat(t) for t in zip(*parts))
    mask = torch.rand((B, H, -(-N // 128), -(-Nk // 64)), generator=torch.Generator().manual_seed(N)) < 0.4
    mask[..., 0] = True
    mask = mask.cuda()
    o, o2 = _both(lambda: sa.block_sparse_sage2_attn_cuda(q, k, v, mask_id=mask, qk_quant_gran=gran, tensor_layout="NHD" if nhd else "HND"))
    assert torch.equal(_bits(o), _bits(o2))


def test_in_place_under_capture():
    """The route has no state of its own: a captured call replays with other inputs in the same buffers."""
    H, N, Nk, D = 40, 2049, 1000, 128
    q, k, v = _qkv(H, H, N, Nk, D, torch.bfloat16, False, 1)
    call = lambda: sa.spas_sage2_attn_meansim_topk_cuda(q, k, v, topk=0.4)       # noqa: E731
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for seed in (1, 11, 21):
        for dst, src in zip((q, k, v), _qkv(H, H, N, Nk, D, torch.bfloat16, False, seed)):
            dst.copy_(src)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(_bits(out), _bits(call()))


def _output_over_q(alias, selection, N):
    H, Nk, D = 40, 512, 128
    buf = rand_T((H * N * D + 64 * D,), torch.bfloat16, 5)
    q = buf[:H * N * D].view(1, H, N, D)
    k, v = rand_T((1, H, Nk, D), torch.bfloat16, 6), rand_T((1, H, Nk, D), torch.bfloat16, 7)
    out = {"rows": q, "shifted": buf[64 * D:].view(1, H, N, D), "other_layout": q.view(1, N, H, D).transpose(1, 2)}[alias]
    mask = torch.ones((1, H, N // 128, Nk // 64), dtype=torch.int8, device="cuda") if selection == _lib.SELECT_MASK else None

    def call(q, out):
        plan = _lib.ForwardPlan(q, k, v, out, mask, selection, False, False, False, False, 1, D ** -0.5)
        plan.run(q, k, v, out, mask, 0.5, -0.1, 50.0)
        return out

    want = call(q.clone(), torch.empty_like(q))
    assert torch.equal(_bits(call(q, out).contiguous()), _bits(want))


@pytest.mark.parametrize("alias", ["rows", "shifted", "other_layout"])
@pytest.mark.parametrize("selection", [_lib.SELECT_TOPK, _lib.SELECT_MASK])
def test_output_over_q(alias, selection):
    """Every Q block is read before another's output lands on it: the output may lie over q in any way."""
    _output_over_q(alias, selection, 2048)


@pytest.mark.parametrize("alias", ["rows", "shifted", "other_layout"])
def test_output_over_q_with_a_mask_in_place(alias):
    _output_over_q(alias, _lib.SELECT_MASK, 4608)
