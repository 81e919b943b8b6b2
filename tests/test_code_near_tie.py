"""INT8 codes by one rounding: where no 16-bit float lies near a tie (n + 1/2) s, rounding a * RN(1 / s) once to an integer gives the
code of the division.  Restates the kernels' rule (csrc/stage_bodies.h, no_code_near_tie) on the CPU and holds the kernels to the
oracle on blocks at both sides of it."""
import numpy as np
import pytest
import torch

from oracle import maskpred as mp
from gpu_common import tag_of, to_np

F = np.float32


def _elements(dtype, top):
    """Every finite value of the type up to `top`."""
    bits = torch.arange(0, 0x7f80 if dtype == torch.bfloat16 else 0x7c00, dtype=torch.int32).to(torch.int16)
    x = bits.view(dtype).float().numpy()
    return x[x <= top]


def _near_tie(s, dtype):
    t = ((np.arange(128, dtype=F) + F(0.5)) * s).astype(F)
    a = torch.from_numpy(t).to(dtype).float().numpy()
    return bool((np.abs(a - t) <= t * F(float.fromhex("0x1.04p-22"))).any())


def _by_division(a, s):
    return np.trunc((a / s).astype(F) + F(0.5)).astype(np.int64)


def _by_product(a, s):
    r = F(1.0) / s
    exact = a.astype(np.longdouble) * np.longdouble(r) + np.longdouble(12582912.0)     # 64-bit mantissa, rounded once below
    return np.rint(exact).astype(np.int64) - 12582912


def _scales(dtype, n, seed):
    """Random scales, and scales that put an element within a few ulp of a tie."""
    rng = np.random.default_rng(seed)
    amax = torch.from_numpy((rng.random(n) * 4 + 0.01).astype(F)).to(dtype).float().numpy()
    s = list((amax / F(127.0)).astype(F) + F(1e-7))
    for a in amax[:n // 2]:
        q = F(float(a) / (rng.integers(0, 127) + 0.5))
        for ulps in range(-6, 7):
            s.append((q.view(np.int32) + np.int32(ulps)).view(F))
    return s


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_one_rounding_gives_the_code_of_the_division(dtype):
    fast = 0
    for s in _scales(dtype, 120, 1):
        a = _elements(dtype, float(s) * 127)
        if _near_tie(s, dtype):
            continue
        fast += 1
        assert np.array_equal(_by_product(a, s), _by_division(a, s)), float(s)
    assert fast >= 80                                   # nearly all of the 120 random ones


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_codes_of_blocks_with_and_without_near_ties(dtype, D):
    """The first block row by row holds the block maximum and, where the scale has one, the element at the tie and its neighbours."""
    from spargeattn_amd import _lib
    rng, H = np.random.default_rng(2), 64
    x = np.zeros((1, H, 128, D), F)
    hit = 0
    for h in range(H):
        amax = torch.tensor(rng.random() * 4 + 0.1).to(dtype).float().numpy()
        s = (amax / F(127.0)).astype(F) + F(1e-7)
        t = ((np.arange(127, dtype=F) + F(0.5)) * s).astype(F)
        near = torch.from_numpy(t).to(dtype)
        up, down = ((near.view(torch.int16) + d).view(dtype).float().numpy() for d in (1, -1))
        rows = np.concatenate([near.float().numpy(), up, down])
        hit += _near_tie(s, dtype)
        x[0, h].flat[:3 * 127] = np.minimum(rows, amax)
        x[0, h].flat[3 * 127:6 * 127] = -np.minimum(rows, amax)
        x[0, h, 127, :] = amax
    assert dtype == torch.bfloat16 or 0 < hit < H
    t = torch.from_numpy(x).to(dtype).cuda()
    thr = torch.zeros(H, device="cuda")
    for bs, rows in ((128, 128), (64, 64), (128, 32)):
        kw = {} if rows == bs else {"quant_rows": rows}
        got = _lib.pool_sim_quant(t, None, bs, thr, **kw)
        want = mp.pool_sim_quant(to_np(t), None, bs, np.zeros(H, F), tag_of(dtype), **kw)
        assert np.array_equal(got[2].cpu().numpy(), want["q"])
        assert np.array_equal(got[3].cpu().numpy().view(np.uint32), want["scale"].view(np.uint32))
