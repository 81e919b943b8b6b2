"""INT8 codes by one rounding: where a * m, with m = RN(1 / s) or the float above it, rounds to the code of the division for the elements next
to the ties (n + 1/2) s, it does so for every element of the block.  Restates the kernels' rule (csrc/stage_bodies.h, code_multiplier) on
the CPU and holds the kernels to the oracle on blocks of every outcome of it, over all magnitudes."""
import numpy as np
import pytest
import torch

from oracle import maskpred as mp
from gpu_common import tag_of, to_np

F = np.float32
DTYPES = [torch.bfloat16, torch.float16]
TIES = np.arange(127, dtype=F) + F(0.5)
BY_R, BY_ABOVE, BY_DIVISION = 0, 1, 2


def _finite(dtype, lo, hi):
    """Every positive value of the type from lo to hi."""
    bits = torch.arange(1, 0x7f80 if dtype == torch.bfloat16 else 0x7c00, dtype=torch.int32).to(torch.int16)
    x = bits.view(dtype).float().numpy()
    return x[(x >= lo) & (x <= hi)]


def _scale(amax):
    return (amax / F(127.0)).astype(F) + F(1e-7)


def _above(r):
    return (r.view(np.int32) + np.int32(1)).view(F)


def _by_division(a, s):
    return np.trunc((a / s).astype(F) + F(0.5)).astype(np.int64)


def _by_product(a, m):
    exact = a.astype(np.longdouble) * m.astype(np.longdouble) + np.longdouble(12582912.0)     # 64-bit mantissa, rounded once below
    return np.rint(exact).astype(np.int64) - 12582912


def _next_to_ties(s, dtype):
    t = (TIES * s[..., None]).astype(F)
    return torch.from_numpy(t).to(dtype)


def _route(amax, dtype):
    """What code_multiplier decides for blocks with these maxima."""
    s = _scale(amax)
    a, r = _next_to_ties(s, dtype).float().numpy(), F(1.0) / s
    want = _by_division(a, s[..., None])
    by_r = (_by_product(a, r[..., None]) == want).all(-1)
    by_above = (_by_product(a, _above(r)[..., None]) == want).all(-1)
    return np.where(by_r, BY_R, np.where(by_above, BY_ABOVE, BY_DIVISION))


def _maxima(dtype):
    """Every maximum whose scale is far enough from the ends of binary32 for the rule to be asked (2^-60 to 2^60)."""
    return _finite(dtype, 0.0, 2.0 ** 60 * 126)


@pytest.mark.parametrize("dtype", DTYPES)
def test_the_products_give_the_codes_of_the_division(dtype):
    """Every block maximum, at the elements next to the ties and two on either side of them."""
    for amax in np.array_split(_maxima(dtype), 32):
        s, route = _scale(amax), _route(amax, dtype)
        m = np.where(route == BY_R, F(1.0) / s, _above(F(1.0) / s))
        near = _next_to_ties(s, dtype).view(torch.int16)
        for off in range(-2, 3):
            a = torch.clamp(near + off, min=0).view(dtype).float().numpy()
            ok = (_by_product(a, m[:, None]) == _by_division(a, s[:, None])) | (a > amax[:, None])
            assert ok[route != BY_DIVISION].all()


@pytest.mark.parametrize("dtype", DTYPES)
def test_every_element_of_some_blocks(dtype):
    rng = np.random.default_rng(1)
    amax = rng.choice(_maxima(dtype), 200, replace=False)
    for a, s, route in zip(amax, _scale(amax), _route(amax, dtype)):
        x, r = _finite(dtype, 0.0, a), F(1.0) / s
        if route != BY_DIVISION:
            assert np.array_equal(_by_product(x, r if route == BY_R else _above(r)), _by_division(x, s)), float(a)


@pytest.mark.parametrize("dtype", DTYPES)
def test_few_blocks_of_any_magnitude_need_the_division(dtype):
    """Above 64 half of every maximum lies at a tie; that alone must not send a block to the division."""
    top = 65504.0 if dtype == torch.float16 else 1e9
    edges = 10.0 ** np.arange(-3.0, np.log10(top), 0.5)
    for lo, hi in zip(edges, np.append(edges[1:], top)):
        route = _route(_finite(dtype, lo, hi), dtype)
        assert (route == BY_DIVISION).mean() < 0.03, (lo, hi)
        assert (route == BY_R).mean() > (0.98 if hi < 100 else 0.5), (lo, hi)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", DTYPES)
def test_codes_of_blocks_of_every_route(dtype, D):
    """A block holds its maximum, the elements next to the ties of its scale and their neighbours, both signs, and some of them a NaN."""
    from spargeattn_amd import _lib
    rng = np.random.default_rng(2)
    all_max = _finite(dtype, 1e-3, 6e4)
    routes = _route(all_max, dtype)
    large = all_max >= 48
    picks = [all_max[large & (routes == BY_R)], all_max[~large & (routes == BY_R)], all_max[large & (routes == BY_ABOVE)],
             all_max[large & (routes == BY_DIVISION)]]
    if dtype == torch.float16:
        picks += [all_max[~large & (routes == BY_ABOVE)], all_max[~large & (routes == BY_DIVISION)]]
    amax = np.concatenate([rng.choice(p, 12, replace=len(p) < 12) for p in picks])
    H = len(amax)
    near = _next_to_ties(_scale(amax), dtype)
    x = np.zeros((1, H, 128, D), F)
    for h in range(H):
        rows = np.concatenate([(near[h].view(torch.int16) + d).view(dtype).float().numpy() for d in (0, 1, -1)])
        rows = np.minimum(rows, amax[h])
        x[0, h].flat[:3 * 127] = rows
        x[0, h].flat[3 * 127:6 * 127] = -rows
        x[0, h, 30::32, :] = amax[h]                      # in every 32-row group
        if h % 3 == 0:
            x[0, h, 63, 5] = np.nan
            x[0, h, 0, 7] = -np.nan
    t = torch.from_numpy(x).to(dtype).cuda()
    thr = torch.zeros(H, device="cuda")
    for bs, rows in ((128, 128), (64, 64), (128, 32)):
        kw = {} if rows == bs else {"quant_rows": rows}
        got = _lib.pool_sim_quant(t, None, bs, thr, **kw)
        want = mp.pool_sim_quant(to_np(t), None, bs, np.zeros(H, F), tag_of(dtype), **kw)
        assert np.array_equal(got[2].cpu().numpy(), want["q"])
        assert np.array_equal(got[3].cpu().numpy().view(np.uint32), want["scale"].view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", DTYPES)
def test_groups_of_different_routes_in_one_block(dtype, D):
    """The four 32-row groups of a block have routes and scales of their own, in every order; the last block has 40 rows."""
    from spargeattn_amd import _lib
    rng = np.random.default_rng(3)
    all_max = _finite(dtype, 48.0, 6e4)
    routes = _route(all_max, dtype)
    H, N = 6, 128 * 4 + 40
    x = np.zeros((1, H, N, D), F)
    for h in range(H):
        for g in range(0, N, 32):
            amax = rng.choice(all_max[routes == rng.integers(3)])
            near = _next_to_ties(_scale(amax), dtype).view(torch.int16)
            rows = np.minimum(np.concatenate([(near + d).view(dtype).float().numpy() for d in (0, 1, -1)]), amax)
            part = np.concatenate([[amax], rows, -rows]).astype(F)
            n = min(32, N - g) * D
            x[0, h, g:g + 32].flat[:min(n, part.size)] = part[:n]
    t = torch.from_numpy(x).to(dtype).cuda()
    got = _lib.pool_sim_quant(t, None, 128, torch.zeros(H, device="cuda"), quant_rows=32)
    want = mp.pool_sim_quant(to_np(t), None, 128, np.zeros(H, F), tag_of(dtype), quant_rows=32)
    assert np.array_equal(got[2].cpu().numpy(), want["q"])
    assert np.array_equal(got[3].cpu().numpy().view(np.uint32), want["scale"].view(np.uint32))
