"""The work a user of the operators has them do, as cases that can be timed.

Every case is one call of a public operator of ``spargeattn_amd`` on tensors that are already on the GPU, as a model's
attention layer makes it: five entry points (top-k and CDF selection and a mask of the caller's own in front of the FP8-PV
kernel, top-k and CDF selection in front of the FP16-PV kernel), both head sizes, fp16 and bf16, both tensor layouts, block-
and token-level causality, fewer K/V heads than query heads, key/value lengths of their own, per-head parameters from a
tuner.  Sequence lengths run from 128 tokens (the shortest the operators take) to 118 800, the longest of the benchmark
configurations; the work of a call spans more than five decades.

Fields of a case: ``op`` (entry point), ``B H Hkv N Nk D`` (sizes), ``dtype``, ``field`` (how q and k are distributed),
``layout`` ("HND" / "NHD"), ``causal``, ``token_causal`` (the FP8-PV operators' ``kernel_causal``), ``gran`` (INT8
granularity of Q), ``level`` (top-k fraction, CDF threshold, or density of the mask), ``sim`` (similarity threshold),
``pv`` (PV threshold), ``sink`` (attention sink), ``tuned`` (per-head tensors instead of scalars), ``report`` (the call
returns the sparsity as well, which waits for the GPU).
"""
import math

import torch

import spargeattn_amd as sa
from spargeattn_amd import workloads as W

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}

BASE = dict(op="topk", B=1, H=8, Hkv=0, N=4096, Nk=0, D=128, dtype="bf16", field="rank", layout="HND", causal=False,
            token_causal=False, gran=1, level=0.5, sim=-0.1, pv=50.0, sink=False, tuned=False, report=False)


def _case(name=None, **kw):
    c = dict(BASE, **kw)
    c["Hkv"] = c["Hkv"] or c["H"]
    c["Nk"] = c["Nk"] or c["N"]
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest configuration of the benchmark set: a short prompt, two heads.  Nothing but latency and launches.
        _case("short_fp16_d64", H=2, N=1024, D=64, dtype="fp16"),
        # A short ragged sequence with the default operator (CDF selection with a similarity test), causal.
        _case("ragged_cdf_causal", op="cdf", B=2, H=3, N=1025, level=0.98, sim=0.6, causal=True),
        # What the per-head tuner asks for thousands of times: one head of a video model, with the sparsity read back.
        _case("tuner_one_head", op="cdf", H=1, N=17776, D=64, field="smooth", level=0.9, sim=0.3, report=True),
        # Prefill of a grouped-query model in the (B, N, H, D) layout its projections produce, masked token by token.
        _case("gqa_prefill_nhd", H=32, Hkv=8, N=4096, layout="NHD", causal=True, token_causal=True),
        # Cross attention: 16 heads of video tokens over a shorter key/value sequence, finer scales of Q.
        _case("cross_per_warp", H=16, N=8190, Nk=2500, D=128, dtype="fp16", gran=2),
        # The FP16-PV operator on a causal prefill.
        _case("fp16pv_causal", op="topk16", H=24, N=8192, dtype="fp16", causal=True),
        # A tuned layer of a 30-head video model: per-head CDF / similarity / PV thresholds and the attention sink.
        _case("tuned_video_d64", op="cdf", H=30, N=17776, D=64, field="smooth", level=0.97, sim=-0.5, pv=10.0, sink=True,
              tuned=True),
        # The same layer with top-k selection (cfg3 of the benchmark set).
        _case("video_topk_d64", H=30, N=17776, D=64, field="smooth"),
        # A block mask that the caller brings (cfg2 of the benchmark set).
        _case("own_mask", op="mask", B=2, H=24, N=16384, field="noise", level=0.3),
        # The headline configuration (cfg4): long causal prefill.
        _case("long_causal_topk", H=32, N=32768, causal=True),
        # The longest (cfg5): a video model's full sequence.
        _case("longest_video", H=24, N=118800, field="smooth", level=0.3),
    ]


def _pairs(c):
    """(query, key) pairs of the full score matrix, times the channels: what the cost of a call grows with."""
    return c["B"] * c["H"] * c["N"] * c["Nk"] * c["D"]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges.  A call costs at most what the second largest listed one does."""
    op = rng.choice(["topk", "topk", "topk", "cdf", "cdf", "mask", "topk16", "cdf16"])
    D = rng.choice([64, 128])
    dtype = rng.choice(["fp16", "bf16", "bf16"])
    N = _log_int(rng, 128, 118800)
    if rng.random() < 0.5:                       # half of them at a whole number of blocks, as padded sequences are
        N = max(128, (N + 64) // 128 * 128)
    cap = 32 * 32768 * 32768 * 128
    most = max(1, min(48, cap // (N * N * D)))
    H = rng.randint(1, most)
    B = 2 if 2 * H <= most and rng.random() < 0.3 else 1
    Hkv = H
    if rng.random() < 0.25 and op != "mask":
        Hkv = rng.choice([h for h in range(1, H + 1) if H % h == 0])
    causal = op != "mask" and rng.random() < 0.4
    Nk = N
    if not causal and op != "mask" and rng.random() < 0.2:
        Nk = max(128, _log_int(rng, max(128, N / 8), N))
    level = {"topk": rng.uniform(0.15, 0.7), "topk16": rng.uniform(0.15, 0.7), "cdf": rng.uniform(0.8, 0.98),
             "cdf16": rng.uniform(0.8, 0.98), "mask": rng.uniform(0.1, 0.6)}[op]
    return _case(op=op, B=B, H=H, Hkv=Hkv, N=N, Nk=Nk, D=D, dtype=dtype, field=rng.choice(["rank", "smooth", "noise"]),
                 layout=rng.choice(["HND", "HND", "NHD"]), causal=causal,
                 token_causal=causal and op in ("topk", "cdf") and rng.random() < 0.5,
                 gran=rng.choice([1, 1, 1, 2]), level=round(level, 3),
                 sim=-0.1 if op.startswith("topk") else rng.choice([-0.1, 0.3, 0.6]),
                 pv=rng.choice([50.0, 50.0, 15.0]), sink=rng.random() < 0.2)


def _grid_of(n):
    """(frames, rows, columns) of a latent video with at most n tokens, in the proportions of the video configurations."""
    w = max(1, int(round((n * 3.0) ** (1.0 / 3.0))))
    h = max(1, w * 2 // 3)
    return max(1, n // (h * w)), h, w


def _qk(c, heads, n, g):
    """(B, heads, n, D) float32 queries or keys.

    "rank":   a rotated rank-16 signal with noise, as queries and keys behind rotary embeddings are (long causal prefill)
    "smooth": a field that varies slowly over a latent video, with text tokens behind it (video models)
    "noise":  N(0, 1)
    """
    B, D, dev = c["B"], c["D"], "cuda"
    randn = lambda *s: torch.randn(s, generator=g, device=dev)                       # noqa: E731
    if c["field"] == "noise":
        return randn(B, heads, n, D)
    if c["field"] == "rank":
        return W.rope(randn(B, heads, n, 16) @ (randn(B, heads, 16, D) / 4.0)) + randn(B, heads, n, D)
    grid = _grid_of(n)
    tokens = grid[0] * grid[1] * grid[2]
    x = W.smooth_field_3d(B, heads, grid, D, 2.0, g, dev) + 0.2 * randn(B, heads, tokens, D)
    return torch.cat([x, randn(B, heads, n - tokens, D)], dim=2) if tokens < n else x


def prepare(case, seed):
    c = case
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    dtype = DTYPES[c["dtype"]]

    def laid_out(x):
        x = x.to(dtype)
        return x.transpose(1, 2).contiguous() if c["layout"] == "NHD" else x.contiguous()

    q = laid_out(_qk(c, c["H"], c["N"], g))
    k = laid_out(_qk(c, c["Hkv"], c["Nk"], g))
    v = laid_out(torch.randn((c["B"], c["Hkv"], c["Nk"], c["D"]), generator=g, device="cuda"))
    kw = dict(tensor_layout=c["layout"], pvthreshd=c["pv"], qk_quant_gran=c["gran"])
    op = c["op"]
    if op == "mask":
        nq, nk = (c["N"] + 127) // 128, (c["Nk"] + 63) // 64
        mask = torch.rand((c["B"], c["H"], nq, nk), generator=g, device="cuda") < c["level"]
        i = torch.arange(nq, device="cuda")
        for off in (0, 1):                       # the diagonal is always kept
            mask[:, :, i, (2 * i + off).clamp(max=nk - 1)] = True
        kw["mask_id"] = mask.to(torch.int32)
        return {"fn": sa.block_sparse_sage2_attn_cuda, "args": (q, k, v), "kw": kw}
    kw.update(is_causal=c["causal"], simthreshd1=c["sim"], attention_sink=c["sink"], return_sparsity=c["report"])
    level_name = "topk" if op.startswith("topk") else "cdfthreshd"
    kw[level_name] = c["level"]
    if c["tuned"]:
        # what the tuner stores: one value per head, around the case's own
        def per_head(lo, hi):
            return lo + (hi - lo) * torch.rand((c["H"],), generator=g, device="cuda")
        kw[level_name] = per_head(c["level"] - 0.03, min(1.0, c["level"] + 0.03))
        kw["simthreshd1"] = per_head(c["sim"] - 0.4, c["sim"] + 0.9)
        kw["pvthreshd"] = per_head(0.5 * c["pv"], 2.0 * c["pv"])
    if op in ("topk", "cdf"):
        kw["kernel_causal"] = c["token_causal"]
    fn = {"topk": sa.spas_sage2_attn_meansim_topk_cuda, "cdf": sa.spas_sage2_attn_meansim_cuda,
          "topk16": sa.spas_sage_attn_meansim_topk_cuda, "cdf16": sa.spas_sage_attn_meansim_cuda}[op]
    return {"fn": fn, "args": (q, k, v), "kw": kw}


def run(state):
    return state["fn"](*state["args"], **state["kw"])


def work(case):
    """q, k, v (and a mask) read once, the output written once; both products over the blocks that are kept: exactly
    known for top-k selection and a mask, at most the threshold's share of the blocks for CDF selection."""
    c = case
    nq, nk = (c["N"] + 127) // 128, (c["Nk"] + 63) // 64
    heads = c["B"] * c["H"]
    data = 2 * c["D"] * c["B"] * (2 * c["H"] * c["N"] + 2 * c["Hkv"] * c["Nk"])
    if c["op"] == "mask":
        data += 4 * heads * nq * nk
    kept = c["level"] * nk
    if c["causal"]:
        blocks = sum(min(kept, 2 * (i + 1), nk) for i in range(nq))
    else:
        blocks = kept * nq
    return {"bytes": data, "flops": heads * blocks * 2 * (2 * 128 * 64 * c["D"])}


def tolerance(case):
    """Outputs are fp16 or bf16.  The codes of Q, K, V and P (INT8, e4m3) and the selected blocks follow from the
    arithmetic the operators prescribe, so what is free is the order of binary32 sums and the rounding of the result."""
    return {"rel": 1e-2}
