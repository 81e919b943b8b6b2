"""Selection of few rows: a workgroup to a row.  The same heads among many others take a wavefront to a row (and eight or sixteen rows to a
workgroup); both have to write the same lists, counts and maps, bit for bit."""
import pytest
import torch

from spargeattn_amd import _lib

pytestmark = pytest.mark.gpu


# around the widths of a wavefront's share and of a workgroup's row (256, 512, 1024, 2048 columns)
@pytest.mark.parametrize("nk", [1, 63, 64, 65, 129, 255, 256, 257, 278, 511, 512, 513, 1000, 1025, 1563, 2047, 2048])
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (64, torch.bfloat16), (128, torch.float16), (128, torch.bfloat16)])
def test_equal_the_rows_among_many(D, dtype, nk):
    g = torch.Generator().manual_seed(D + nk)
    H, Hkv, nq, times = 4, 2, 9, 16                    # 36 rows, and 576
    causal = nk % 2 == 1
    if causal:
        nq = (nk + 1) // 2                             # square masks: up to 512 rows, and more than 512
        H = max(1, min(4, 512 // nq))
        Hkv = 1
        times = 512 // (H * nq) + 1
    scale = torch.tensor([0.3, 1.0, 4.0, 12.0])[:H]    # even rows, and probabilities far below what binary64 holds beside 1
    pq = (torch.randn((1, H, nq, D), generator=g) * scale[:, None, None]).to(dtype)
    pk = torch.randn((1, Hkv, nk, D), generator=g).to(dtype)
    pk[:, :, nk // 2:] = pk[:, :, nk // 2:][:, :, :1]   # equal scores: the order of the columns decides
    sq = torch.rand((1, H, nq), generator=g) > 0.1
    sk = torch.rand((1, Hkv, nk), generator=g) > 0.1
    if nq > 3:
        pq[0, 0, 1, 3] = float("inf")
        pq[0, -1, 2, 5] = float("nan")
        pq[0, 0, 3] = 0.0
    few = [t.cuda() for t in (pq, sq, pk, sk)]
    many = [t.repeat((times,) + (1,) * (t.dim() - 1)).cuda() for t in (pq, sq, pk, sk)]
    for levels in ([0.5, 0.05, 0.9, 0.3], [0.0, 1.0, 1.5, 0.98]):
        for name in ("topk", "cdfthreshd"):
            kw = {name: torch.tensor(levels[:H], device="cuda"), "is_causal": causal, "attention_sink": nk % 4 == 1, "return_map": True}
            want, got = _lib.block_select(*many, **kw), _lib.block_select(*few, **kw)
            for w, o in zip(want, got):
                assert torch.equal(w, o.expand_as(w).contiguous() if o.shape[0] == 1 else o)
