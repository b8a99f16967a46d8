"""Bamanex decoder: the framework (model registry -> LLMEngine -> native scheduler -> ops) against the slow float64 oracle
in tests/bamanex_oracle.py. Small made-up configurations and random weights with sizeable biases, sinks, gates and layer
scales, so that a wrong key, a window off by one, a sink left out, a swapped norm, a wrong pass of the loop or a wrong expert
moves the logits far beyond the tolerance. CPU runs use the reference ops, GPU runs the HIP kernels (fp32: tight tolerance;
bf16: rounding level).
"""
import json
import math
import os
import subprocess
import sys

import pytest
import torch

from generativeaiexamples_amd import ops
from generativeaiexamples_amd.engine import EngineConfig, LLMEngine, SamplingParams
from generativeaiexamples_amd.models.bamanex import BamanexConfig, BamanexModel
from generativeaiexamples_amd.models.registry import build_llm

from . import bamanex_oracle as O

_GPU = pytest.mark.gpu
TARGETS = [pytest.param("cpu", torch.float32, id="cpu-fp32"),
           pytest.param("cuda", torch.float32, id="gpu-fp32", marks=_GPU),
           pytest.param("cuda", torch.bfloat16, id="gpu-bf16", marks=_GPU)]
FP32_TARGETS = TARGETS[:2]
B = ops.BLOCK


def row_err(got, want):
    """RMS of the difference (mean over the vocabulary taken off) over the RMS of the centred reference, per row."""
    centre = lambda x: x.double() - x.double().mean(-1, keepdim=True)  # noqa: E731
    w = centre(want)
    return (centre(got) - w).pow(2).mean(-1).sqrt() / w.pow(2).mean(-1).sqrt().clamp_min(1e-9)


def close(got, want, dtype):
    """fp32: every row within 1e-4. bf16: rounding level - rows within 3 % on average, none beyond 15 %; a wrong mechanism is
    off by tens of percent on most rows it touches."""
    assert got.shape == want.shape
    e = row_err(got, want)
    if dtype == torch.float32:
        return e.max().item() < 1e-4
    return e.mean().item() < 3e-2 and e.max().item() < 0.15


def make_engine(cfg, sd, device, dtype, max_tokens=512, max_seqs=4):
    from generativeaiexamples_amd.engine.tokenizer import load_tokenizer
    model = BamanexModel(BamanexConfig.from_json(cfg), device=device, dtype=dtype).load_state(sd)
    return LLMEngine(model, load_tokenizer(None, "llama3", cfg["vocab"]), EngineConfig(
        max_num_seqs=max_seqs, num_blocks=max_tokens // B, max_model_len=max_tokens, max_batched_tokens=1 << 20,
        use_graphs=device != "cpu", graph_batch_sizes=(1, 2, 4), decode_steps=1))


def run_schedule(eng, prompts, schedule):
    """schedule: list of steps, each a list of (request name, count). Returns {name: logits of every position}; a request
    ends when its tokens are used up."""
    at = {n: 0 for n in prompts}
    got = {n: [] for n in prompts}
    for step in schedule:
        entries, end = [], []
        for name, count in step:
            entries.append((name, prompts[name][at[name]:at[name] + count], list(range(count))))
            at[name] += count
            if at[name] == len(prompts[name]):
                end.append(name)
        out, r = eng.replay_step(entries, end), 0
        for name, count in step:
            got[name].append(out[r:r + count])
            r += count
    return {n: torch.cat(v) for n, v in got.items() if v}


def tokens(n, vocab, seed):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


def config_for(dtype, layers, **kw):
    """An expert choice is a discrete decision, and with random weights some position always has two router logits closer
    than bf16 rounding of the router's input: bf16 runs take every expert (the same kernels, no decision), and the choice
    itself is tested in fp32 on prompts without a near-tie (clear_tokens)."""
    if dtype == torch.bfloat16:
        layers = [l if (l["mlp"] or {}).get("kind") != "moe" else
                  dict(l, mlp=dict(l["mlp"], router=dict(l["mlp"]["router"], top=l["mlp"]["router"]["experts"])))
                  for l in layers]
    return O.make_config(layers, **kw)


def clear_tokens(n, cfg, sd, seed, gap=1e-4):
    """Random tokens whose router has no near-tie between the last chosen and the first rejected expert."""
    for s in range(seed, seed + 60):
        t, margins = tokens(n, cfg["vocab"], s), []
        O.forward(cfg, sd, t, margins=margins)
        if min(margins + [math.inf]) > gap:
            return t
    raise AssertionError("no clear-cut prompt found")


def cuts(n, sizes):
    out, i = [], 0
    while n > 0:
        out.append(min(n, sizes[i % len(sizes)]))
        n -= out[-1]
        i += 1
    return out


FULL = [O.dense(O.att()), O.experts(O.att(window=7, kv_heads=6)),
        O.no_ff(O.att(heads=3, kv_heads=1, dim=10, vdim=5, window=23, rot=4, scaling=None, scale=0.9)), O.experts(O.att(), n=4, top=1, shared=0)]
LOOP = (1, 3, 2)


# ------------------------------------------------------------------------------------------------ each mechanism alone
MECHANISMS = {
    "attention": ([O.no_ff(O.att())], {}),
    "attention-1head-1dim": ([O.no_ff(O.att(heads=1, kv_heads=1, dim=1, vdim=1, rot=0, scale=2.0))], {}),
    "attention-mha-wide-values": ([O.no_ff(O.att(heads=5, kv_heads=5, dim=6, vdim=40, rot=2, window=3))], {}),
    "attention-one-kv-head": ([O.no_ff(O.att(heads=7, kv_heads=1, dim=16, vdim=16, rot=16, window=16))], {}),
    "attention-window-1": ([O.no_ff(O.att(window=1))], {}),
    "attention-wide-window-plain-rotation": ([O.no_ff(O.att(window=1000, scaling=None, base=10000.0))], {}),
    "attention-no-rotation": ([O.no_ff(O.att(rot=0, scaling=None))], {}),
    "attention-all-stretched": ([O.no_ff(O.att(scaling=(5.0, 1.0, 4.0, 2)))], {}),
    "attention-all-kept": ([O.no_ff(O.att(scaling=(5.0, 1.0, 4.0, 10 ** 7)))], {}),
    "dense": ([O.dense(O.att())], {}),
    "dense-narrow": ([O.dense(O.att(), ff=7)], {}),
    "experts": ([O.experts(O.att())], {}),
    "experts-top1-no-shared": ([O.experts(O.att(), n=3, top=1, shared=0)], {}),
    "experts-12-top5-tight": ([O.experts(O.att(), ff=40, n=12, top=5, limit=0.3, shared=8, shared_limit=0.2)], {}),
    "experts-all": ([O.experts(O.att(), n=4, top=4, limit=50.0)], {}),
    "experts-70": ([O.experts(O.att(), ff=4, n=70, top=16)], {}),
    "loop-whole-stack": ([O.dense(O.att()), O.no_ff(O.att(window=4))], dict(loop=(0, 2, 4))),
    "loop-once": ([O.dense(O.att()), O.no_ff(O.att(window=4))], dict(loop=(1, 2, 1))),
    "large-eps-unit-scale": ([O.dense(O.att(scale=1.0))], dict(eps=0.3, logit_scale=1.0)),
}


@pytest.mark.parametrize("device,dtype", TARGETS)
@pytest.mark.parametrize("name", [n for n in MECHANISMS if n != "experts-70"])
def test_single_mechanism(name, device, dtype):
    check_mechanism(name, device, dtype)


@pytest.mark.parametrize("device,dtype", FP32_TARGETS)
def test_more_experts_than_lanes(device, dtype):
    check_mechanism("experts-70", device, dtype)   # 16 of 70 chosen: more than bf16 runs could take at once


def check_mechanism(name, device, dtype):
    layers, kw = MECHANISMS[name]
    cfg = config_for(dtype, layers, width=40, **kw)
    sd = O.random_checkpoint(cfg, 1)
    toks = clear_tokens(37, cfg, sd, 2, gap=2e-5 if name == "experts-70" else 1e-4)
    want = O.forward(cfg, sd, toks)
    got = run_schedule(make_engine(cfg, sd, device, dtype), {"a": toks}, [[("a", 20)], [("a", 1)], [("a", 1)], [("a", 15)]])["a"]
    assert close(got, want, dtype)


@pytest.mark.parametrize("device", [pytest.param("cpu"), pytest.param("cuda", marks=_GPU)])
def test_parallel_add_norm_against_equations(device):
    """Every combination of branch outputs, scales and norms; widths on and off the vector grid, wider than the registers
    of one workgroup; branch outputs as column slices; rows so small that the epsilon inside the root matters."""
    g = torch.Generator().manual_seed(0)
    rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    for T, D in ((3, 256), (70, 64), (5, 70), (2, 4100), (1, 17000), (4, 1), (2, 8192)):
        for dt in (torch.float32, torch.bfloat16):
            res, a, b = rn(T, D), rn(T, D + 8).to(dt)[:, 4:D + 4], rn(T, D).to(dt)
            res[0], a[0], b[0] = res[0] * 1e-3, a[0] * 1e-3, b[0] * 1e-3
            sa, sb, w1, w2 = rn(D), rn(D), rn(D), rn(D)
            for use in ("", "a", "ab", "aA", "aAbB", "bB"):
                for norms in ("", "1", "12", "2"):
                    if not use and not norms:
                        continue
                    want = res.double()
                    kw = {}
                    for n, y, s in (("a", a, sa), ("b", b, sb)):
                        if n in use:
                            kw[n] = y.to(device)
                            sc = s.double() if n.upper() in use else 1.0
                            if n.upper() in use:
                                kw["s" + n] = s.to(device)
                            want = want + y.double() * sc
                    r = res.clone().to(device)
                    h = ops.parallel_add_norm_f32(r, **kw, w1=w1.to(device) if "1" in norms else None,
                                                  w2=w2.to(device) if "2" in norms else None, eps=1e-5, out_dtype=dt)
                    assert torch.allclose(r.cpu().double(), want, atol=1e-5, rtol=1e-5)
                    for got, w, n in ((h[0], w1, "1"), (h[1], w2, "2")):
                        assert (got is not None) == (n in norms)
                        if got is not None:
                            ref = O.unit_rms(want, 1e-5) * w.double()
                            tol = 1e-4 if dt == torch.float32 else 1e-2
                            assert torch.allclose(got.cpu().double(), ref, atol=tol, rtol=tol), (T, D, dt, use, norms)


@_GPU
@pytest.mark.parametrize("D", [2044, 2048, 2052, 4096, 4100, 511, 513, 1025])
def test_parallel_add_norm_kept_groups(D):
    """Rows that fill the kept groups of each form, and one group more or fewer: against float64 (bf16 results, eight
    significant bits: 2^-8; and the
    fp32 sum of up to 4100 squares)."""
    g = torch.Generator(device="cuda").manual_seed(D)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    res, a, b, w1, w2 = rn(5, D), rn(5, D).bfloat16(), rn(5, D).bfloat16(), rn(D), rn(D)
    want = res.double() + a.double() + b.double()
    h1, h2 = ops.parallel_add_norm_f32(res, a=a, b=b, w1=w1, w2=w2, eps=1e-5, out_dtype=torch.bfloat16)
    assert torch.allclose(res.double(), want, atol=1e-6, rtol=1e-6)
    for h, w in ((h1, w1), (h2, w2)):
        ref = O.unit_rms(want, 1e-5) * w.double()
        assert ((h.double() - ref).abs() <= (2.0 ** -8 + 2e-6) * ref.abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T,D,K,form", [(1, 512, 512, "rows"), (24, 2048, 5632, "split"), (24, 2048, 2048, "cut"), (64, 2048, 11264, "split"),
                                        (17, 1040, 4096, "cut"), (3, 16, 1024, "cut"), (33, 1024, 5120, "split"), (65, 2048, 2048, "rows"),
                                        (5, 2064, 5632, "rows"), (1, 2048, 4608, "split"), (16, 1024, 5632, "split"), (32, 1040, 5120, "split"),
                                        (9, 2048, 6656, "split")])
def test_branches_as_k_slices(cuda, T, D, K, form):
    """A branch handed over as its product's K slices: the rows that adding them in order and rounding once gives (the stream's bits),
    normed alike up to the order of the squares' sum, in either branch, beside rows or alone, with and without bias and scale. "split": the
    product has these slices by itself, and gives these bits; "cut": it is one pass over K, which is cut here; "rows" (more than 64, or 2048
    channels, or too little K): the product."""
    g = torch.Generator(device=cuda).manual_seed(T + D + K)
    rn = lambda *s: torch.randn(*s, device=cuda, generator=g)  # noqa: E731
    x, w, bias = rn(T, K).bfloat16(), (rn(D, K) * K ** -0.5).bfloat16(), rn(D).bfloat16()
    other, res, sa, sb, w1, w2 = rn(T, D).bfloat16(), rn(T, D), rn(D), rn(D), rn(D), rn(D)
    for frag in (False, True):
        wt = w.clone()
        if frag and not ops.to_fragment_layout_(wt):
            continue
        for b in (None, bias):
            p = ops.linear_partial(x, wt, b)
            want = ops.linear(x, wt, b)
            assert isinstance(p, ops.Partial) == (form != "rows")
            if form == "rows":
                assert torch.equal(p, want)
                continue
            rows = torch.zeros(T, D, device=cuda)
            for s in p.slabs:
                rows = rows + s
            rows = (rows if b is None else rows + b.float()).bfloat16()
            assert len(p.slabs) > 1 and (form == "cut" or torch.equal(rows, want))
            exact = x.double() @ w.double().t() + (0 if b is None else b.double())
            # K products of unit normals and weights of K^-1/2: fp32 sums, then one rounding to bf16
            assert ((rows.double() - exact).abs() <= 2.0 ** -8 * exact.abs() + 2.0 ** -18 * K ** 0.5).all()
            for kw, kr in ((dict(a=p, sa=sa), dict(a=rows, sa=sa)), (dict(a=other, sa=sa, b=p, sb=sb), dict(a=other, sa=sa, b=rows, sb=sb)),
                           (dict(a=p, b=ops.Partial(p.slabs.flip(0).contiguous()[:1])), dict(a=rows, b=p.slabs[-1].bfloat16()))):
                r1, r2 = res.clone(), res.clone()
                h = ops.parallel_add_norm_f32(r1, **kw, w1=w1, w2=w2, eps=1e-5, out_dtype=torch.bfloat16)
                k = ops.parallel_add_norm_f32(r2, **kr, w1=w1, w2=w2, eps=1e-5, out_dtype=torch.bfloat16)
                assert torch.equal(r1, r2)
                for y, z in zip(h, k):    # one bf16 step where the two sums of squares round apart
                    assert ((y.float() - z.float()).abs() <= 2.0 ** -7 * z.float().abs()).all()
                r1 = res.clone()
                assert ops.parallel_add_norm_f32(r1, **kw) == (None, None) and torch.equal(r1, r2)
            few = p.index_select(0, torch.tensor([T - 1, 0], device=cuda))
            assert torch.equal(few.slabs, p.slabs[:, [T - 1, 0]])


@_GPU
@pytest.mark.parametrize("D", [64, 513, 1000, 2048, 2050, 4096, 8196])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_parallel_add_norm_rows_alike(D, dt):
    """A row has the same sums and norms whether it comes with few rows or with more than the form for few rows takes."""
    g = torch.Generator(device="cuda").manual_seed(D)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    res, a, b, w1, w2, sa = rn(257, D), rn(257, D).to(dt), rn(257, D).to(dt), rn(D), rn(D), rn(D)
    kw = dict(w1=w1, w2=w2, sa=sa, eps=1e-5, out_dtype=dt)
    few = res.clone()
    parts = [ops.parallel_add_norm_f32(few[s:e], a=a[s:e], b=b[s:e], **kw) for s, e in ((0, 256), (256, 257))]
    h = ops.parallel_add_norm_f32(res, a=a, b=b, **kw)
    assert torch.equal(res, few)
    for i in range(2):
        assert torch.equal(h[i], torch.cat([p[i] for p in parts]))


@pytest.mark.parametrize("device,dtype", TARGETS)
def test_rotation_unit_norm_and_cache_write(device, dtype):
    """Rotated halves at positions up to 10^5 with and without the unit norm, tokens in scattered slots and tokens that fill
    whole pages, one and many tokens, head sizes on and off the 16-byte grid; no other cache entry is touched."""
    g = torch.Generator().manual_seed(1)
    rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    dev = torch.device(device)
    for T, H, G, dk, dv, rot in ((300, 4, 2, 64, 48, 32), (1, 2, 1, 64, 64, 32), (5, 3, 3, 7, 9, 4), (6, 4, 2, 128, 32, 128), (150, 5, 1, 48, 20, 16),
                                 (100, 2, 2, 16, 130, 16), (70, 1, 1, 256, 8, 64), (9, 2, 1, 200, 3, 0), (64, 6, 2, 8, 8, 6)):
        lens = (H * dk, G * dk, G * dv)
        x = rn(T, sum(lens) + 3).to(dtype)
        x[0] *= 1e-3
        parts = [x[:, sum(lens[:i]):sum(lens[:i + 1])] for i in range(3)]
        pos = torch.randint(0, 100000, (T,), generator=g)
        if T >= 64:   # consecutive slots from a page's start, then from a page's middle
            slots = torch.cat([torch.arange(T // 2) + 2 * B, torch.arange(T - T // 2) + 12 * B + 5])
        else:
            slots = torch.randperm(20 * B, generator=g)[:T]
        rd = dict(base=10000.0, dims=rot, scaling=dict(factor=4.0, low=1.0, high=4.0, original=300))
        freqs = O.frequencies(rd)
        inv = ops.rope_inv_freq(rot, 10000.0, rd["scaling"])
        assert torch.allclose(inv, torch.tensor(freqs, dtype=torch.float64), rtol=1e-12, atol=0)
        for eps in (None, 1e-5):
            kc, vc = torch.zeros(24, G, B, dk, dtype=dtype, device=dev), torch.zeros(24, G, dv, B, dtype=dtype, device=dev)
            xd = x.to(dev)
            q = ops.rotary_half_kv_write(*[xd[:, sum(lens[:i]):sum(lens[:i + 1])] for i in range(3)], pos.int().to(dev),
                                         slots.int().to(dev), kc, vc, H, G, dk, dv, inv.to(dev), eps)
            turn = lambda p, n: O.rotate_halves(p.double().reshape(T, n, dk), freqs, pos)  # noqa: E731
            wq, wk = turn(parts[0], H), turn(parts[1], G)
            if eps is not None:
                wq, wk = O.unit_rms(wq, eps), O.unit_rms(wk, eps)
            tol = dict(atol=2e-5, rtol=2e-5) if dtype == torch.float32 else dict(atol=1e-2, rtol=1e-2)
            assert torch.allclose(q.cpu().double(), wq.reshape(T, -1), **tol), (T, dk, eps)
            kcc, vcc = kc.cpu().double(), vc.cpu().double()
            assert torch.allclose(kcc[slots // B, :, slots % B], wk, **tol), (T, dk, eps)
            assert torch.equal(vcc[slots // B, :, :, slots % B], parts[2].double().reshape(T, G, dv)), (T, dv)
            kcc[slots // B, :, slots % B] = 0
            vcc[slots // B, :, :, slots % B] = 0
            assert not kcc.any() and not vcc.any()


@pytest.mark.parametrize("device,dtype", TARGETS)
def test_router_against_equations(device, dtype):
    """Router product, softmax and choice for few tokens (one launch) and many (GEMM, then the choice), expert counts below,
    at and above a wave and off the GEMM's grid, top-k of 1, of 16 and of all; large logits; strided logits."""
    g = torch.Generator().manual_seed(2)
    for T, D, E, k in ((1, 64, 6, 2), (5, 48, 16, 4), (64, 72, 70, 16), (7, 33, 3, 3), (100, 64, 20, 5), (3, 256, 130, 1)):
        x, W = torch.randn(T, D, generator=g).to(dtype), torch.randn(E, D, generator=g).to(dtype)
        Wp = torch.cat([W, torch.zeros((-E) % 16, D).to(dtype)])
        z = x.double() @ W.double().t()
        ids, w = ops.moe_router(x.to(device), Wp.to(device), E, k, 1e-20)
        wid, ww = O.route(z, k)
        assert torch.allclose(w.cpu().double().sum(-1), torch.ones(T, dtype=torch.float64), atol=1e-5)
        s = z.sort(-1, descending=True).values
        clear = (s[:, :-1] - s[:, 1:])[:, :k].min(-1).values > 1e-3 * s.abs().max() if E > 1 else torch.ones(T, dtype=torch.bool)
        assert clear.any()
        assert torch.equal(ids.cpu().long()[clear], wid[clear])
        assert torch.allclose(w.cpu().double()[clear], ww[clear], atol=2e-4)
        i2, w2 = ops.moe_route(torch.cat([z, z], 1).float().to(device)[:, E:], k, eps=1e-20)
        assert torch.equal(i2.cpu().long(), wid) and torch.allclose(w2.cpu().double(), ww, atol=1e-5)


@_GPU
@pytest.mark.parametrize("M", [1, 5, 17, 40, 64, 100, 300, 1500])
def test_geglu_epilogue(M):
    """Gated tanh-GELU in the epilogue of every GEMM family (decode streams, split-K, skinny, tiles, 256-wide walks)
    against the fp32 product of the same bf16 values; shapes off the fused grid take the separate kernel."""
    g = torch.Generator().manual_seed(3)
    for K, F_ in ((512, 1024), (2048, 4096), (192, 48), (64, 16), (256, 320), (40, 32)):
        x = torch.randn(M, K, generator=g).to(torch.bfloat16)
        gate, up = ((torch.randn(F_, K, generator=g) * 2 * K ** -0.5).to(torch.bfloat16) for _ in range(2))
        w = ops.interleave_gate_up(gate, up)
        got = ops.linear(x.cuda(), w.cuda(), act="geglu").float().cpu()
        a = O.gelu_tanh(x.double() @ gate.double().t()) * (x.double() @ up.double().t())
        assert got.shape == a.shape
        assert (got - a).norm() < 8e-3 * a.norm() and (got - a).abs().max() < 0.03 * a.abs().max(), (M, K, F_)


# ------------------------------------------------------------------------------------ whole model, schedules, batches
@pytest.mark.parametrize("device,dtype", TARGETS)
def test_prefill_decode_portions(device, dtype):
    """Whole prompt, token-by-token decoding from the first token on, and portions of 2 / 3 / 5 / 17 / 1 tokens: every
    position's logits equal the oracle's, so they do not depend on how the prompt was cut. The stream after every layer run
    (a looped layer counts each time) equals the oracle's."""
    cfg = config_for(dtype, FULL, loop=LOOP)
    sd = O.random_checkpoint(cfg, 3)
    toks = clear_tokens(61, cfg, sd, 4)
    res = []
    want = O.forward(cfg, sd, toks, res)
    eng = make_engine(cfg, sd, device, dtype)
    for name, sizes in (("whole", [61]), ("decode", [1]), ("prefill+decode", [30] + [1] * 31), ("small", [2, 3, 5, 17, 1]),
                        ("twos", [2])):
        got = run_schedule(eng, {name: toks}, [[(name, c)] for c in cuts(61, sizes)])[name]
        assert close(got, want, dtype), name
    eng.model.capture_residuals = []
    run_schedule(eng, {"r": toks}, [[("r", 61)]])
    got_res, eng.model.capture_residuals = eng.model.capture_residuals, None
    assert len(got_res) == len(res) == 6
    for i, (gr, wr) in enumerate(zip(got_res, res)):
        e = (gr.cpu().double() - wr).norm() / wr.norm()
        assert e < (1e-5 if dtype == torch.float32 else 3e-2), (i, float(e))


@pytest.mark.parametrize("device,dtype", TARGETS)
def test_mixed_batches_and_reuse(device, dtype):
    """Unequal requests in one batch (portions beside single tokens, requests sitting out steps) against each alone; a pool of
    six pages, so pages of finished requests are used again by later ones."""
    cfg = config_for(dtype, FULL, loop=LOOP)
    sd = O.random_checkpoint(cfg, 5)
    lens = dict(a=45, b=18, c=33, d=1, e=26)
    prompts = {n: clear_tokens(L, cfg, sd, 10 + 60 * i) for i, (n, L) in enumerate(lens.items())}
    want = {n: O.forward(cfg, sd, t) for n, t in prompts.items()}
    eng = make_engine(cfg, sd, device, dtype, max_tokens=96, max_seqs=2)
    sched = [[("a", 20), ("b", 3)], [("a", 1), ("b", 15)],          # b ends: its pages go back
             [("a", 1), ("c", 2)], [("c", 17), ("a", 5)], [("a", 1), ("c", 1)], [("a", 17), ("c", 13)],  # a, c end
             [("d", 1), ("e", 7)], [("e", 2)], [("e", 1)], [("e", 16)]]
    got = run_schedule(eng, prompts, sched)
    for n in prompts:
        assert close(got[n], want[n], dtype), n
    assert eng.sched.num_free_blocks() == 96 // B


@pytest.mark.parametrize("device,dtype", TARGETS)
def test_first_tokens_and_long_decode(device, dtype):
    """The first five tokens (a few keys beside the sink) and 150 single-token steps across many page borders and windows."""
    cfg = config_for(dtype, [O.experts(O.att(window=20)), O.no_ff(O.att(window=64)), O.dense(O.att(heads=2, window=3))])
    sd = O.random_checkpoint(cfg, 7)
    toks = clear_tokens(155, cfg, sd, 8, gap=3e-5)
    want = O.forward(cfg, sd, toks)
    got = run_schedule(make_engine(cfg, sd, device, dtype), {"a": toks}, [[("a", 1)] for _ in toks])["a"]
    assert close(got[:5], want[:5], dtype)
    assert close(got, want, dtype)


@pytest.mark.parametrize("device,dtype", TARGETS)
@pytest.mark.parametrize("shape", ["wide-odd", "tiny", "unit"])
def test_other_shapes(shape, device, dtype):
    kw = {}
    if shape == "wide-odd":
        layers = [O.experts(O.att(heads=9, kv_heads=3, dim=12, vdim=20, window=13, rot=10), ff=48, n=9, top=3, shared=40),
                  O.no_ff(O.att(heads=2, kv_heads=2, dim=30, vdim=2, rot=2)), O.dense(O.att(heads=4, kv_heads=1), ff=100)]
        kw = dict(width=72, vocab=201, eps=1e-3, loop=(0, 1, 4))
    elif shape == "tiny":
        layers = [O.experts(O.att(heads=1, kv_heads=1, dim=2, vdim=1, rot=2), ff=4, n=2, top=1, shared=2), O.dense(O.att(), ff=1)]
        kw = dict(width=8, vocab=20, logit_scale=3.0)
    else:
        layers = [O.experts(O.att(heads=1, kv_heads=1, scale=1.0, window=1), n=1, top=1, limit=1.0, shared=16, shared_limit=1.0)]
        kw = dict(width=24, logit_scale=1.0, loop=(0, 1, 1))
    cfg = config_for(dtype, layers, **kw)
    sd = O.random_checkpoint(cfg, 23)
    toks = clear_tokens(50, cfg, sd, 22)
    want = O.forward(cfg, sd, toks)
    got = run_schedule(make_engine(cfg, sd, device, dtype), {"a": toks}, [[("a", c)] for c in cuts(50, [19, 1, 1, 6])])["a"]
    assert close(got, want, dtype)


@_GPU
def test_matrix_core_kernels_in_model():
    """bf16 model with sizes on the matrix-core grids: portions take the matrix-core kernels, single tokens the decode
    kernels; both against the oracle, alone and in a mixed batch."""
    layers = [O.experts(O.att(heads=8, kv_heads=2, dim=64, vdim=64, window=50, rot=32), ff=64, n=4, shared=64),
              O.dense(O.att(heads=4, kv_heads=4, dim=32, vdim=32, window=20, rot=32), ff=192),
              O.experts(O.att(heads=6, kv_heads=1, dim=64, vdim=128, window=100, rot=16), ff=128, n=4, shared=0)]
    cfg = config_for(torch.bfloat16, layers, width=192, vocab=128, loop=(0, 2, 2))
    sd = O.random_checkpoint(cfg, 61)
    prompts = {"a": tokens(150, 128, 62), "b": tokens(90, 128, 163)}
    want = {n: O.forward(cfg, sd, t) for n, t in prompts.items()}
    eng = make_engine(cfg, sd, "cuda", torch.bfloat16)
    for sched in ([[("a", 150)], [("b", 40)], [("b", 3)], [("b", 47)]],
                  [[("a", 100), ("b", 5)], [("a", 1), ("b", 60)], [("a", 1), ("b", 1)], [("a", 48), ("b", 24)]]):
        got = run_schedule(eng, prompts, sched)
        for n in prompts:
            assert close(got[n], want[n], torch.bfloat16), n


# ------------------------------------------------------------------------------ keys that stand out: windows, pages, sinks
def _probe(device, dtype, n_ctx, hot, portion, window, query=-1, H=2, G=1, dk=16, dv=8, rot=8, score=30.0, sink=None, gate=None):
    """ops-level: n_ctx positions through the paged cache (pages deliberately scattered). Keys are orthogonal to a probing
    direction - inside the channels that are not rotated - except the one at position `hot`; the query at `query` lies along
    it, so that after the unit norms the hot key's score is `score` and every other 0. The hot value is 1 in every channel, the
    others 0. Returns that query's output per head: the weight of the hot key (times the gate)."""
    dev = torch.device(device)
    nb = (n_ctx + B - 1) // B
    pages = list(range(nb + 3))[::-1][:nb]  # not the identity
    kc = torch.zeros(nb + 4, G, B, dk, dtype=dtype, device=dev)
    vc = torch.zeros(nb + 4, G, dv, B, dtype=dtype, device=dev)
    g = torch.Generator().manual_seed(0)
    qi = query % n_ctx
    d = torch.zeros(dk)
    d[rot:] = torch.randn(dk - rot, generator=g)
    d = d / d.norm()
    k = torch.randn(n_ctx, dk, generator=g)
    k = k - (k @ d)[:, None] * d
    k[hot] = d
    v = torch.zeros(n_ctx, dv)
    v[hot] = 1.0
    q = torch.randn(n_ctx, H, dk, generator=g)
    q[qi] = d
    x = torch.cat([q.reshape(n_ctx, -1), k.repeat(1, G), v.repeat(1, G)], 1).to(dev, dtype)
    sinks = (torch.full((H,), -1e4) if sink is None else torch.tensor(sink, dtype=torch.float32)).to(dev)
    gates = (torch.full((H,), 30.0) if gate is None else torch.tensor(gate)).expand(n_ctx, H).contiguous().to(dev, dtype)
    inv = ops.rope_inv_freq(rot, 100.0, None).to(dev)
    bt = torch.tensor([pages], dtype=torch.int32, device=dev)
    done, res = 0, None
    for c in cuts(n_ctx, portion):
        pos = torch.arange(done, done + c)
        slots = torch.tensor([pages[p // B] * B + p % B for p in pos.tolist()], dtype=torch.int32, device=dev)
        xs = x[done:done + c]
        a, b = H * dk, (H + G) * dk
        qs = ops.rotary_half_kv_write(xs[:, :a], xs[:, a:b], xs[:, b:], pos.int().to(dev), slots, kc, vc, H, G, dk, dv, inv,
                                      1e-6)
        out = ops.window_attention(qs, kc, vc, bt, torch.tensor([0, c], dtype=torch.int32, device=dev),
                                   torch.tensor([done + c], dtype=torch.int32, device=dev), H, G, dk, dv, score / dk,
                                   window=window, sink=sinks, gate=gates[done:done + c])
        if done <= qi < done + c:
            res = out[qi - done].float().cpu().view(H, dv)
        done += c
    assert (res - res[:, :1]).abs().max() < 0.02   # every value channel alike
    return res[:, 0].tolist()


PORTIONS = {"prompt": [1000], "decode": [1], "portions": [7, 2, 30]}


@pytest.mark.parametrize("device,dtype", FP32_TARGETS)
@pytest.mark.parametrize("portion", PORTIONS.values(), ids=PORTIONS.keys())
def test_window_edges_far_keys_and_sinks(device, dtype, portion):
    """One key carries the output: just inside and just outside windows of 1, 2, 15, 16, 17, 33 and 100 at queries around
    page borders, in prompts, portions and single-token steps; far keys among hundreds without a window edge near; the
    query's own position (seen) and the next one (not seen). Sinks and gates differ by head: a visible hot key of score x
    against a sink of score s gets the weight 1 / (1 + e^(s - x)); a gate logit of 0 halves the output."""
    for window in (1, 2, 15, 16, 17, 33, 100):
        for qi in (111, 112, 116):
            near = lambda hot: _probe(device, dtype, 118, hot, portion, window, query=qi)  # noqa: B023, E731
            inside, outside = near(qi - window + 1), near(qi - window)
            assert all(abs(o - 1.0) < 2e-3 for o in inside), (window, qi, inside)
            assert all(abs(o) < 2e-3 for o in outside), (window, qi, outside)
    n = 340
    por = portion if portion != [1] else [300, 1]
    for hot in (0, 1, 15, 16, 17, 63, 64, 200, n - 2, n - 1):
        out = _probe(device, dtype, n, hot, por, 0)
        assert all(abs(o - 1.0) < 2e-3 for o in out), (hot, out)
    for qi in (0, 5, 15, 16, 31, 32, 63, 64):
        assert all(abs(o - 1.0) < 2e-3 for o in _probe(device, dtype, 70, qi, portion, 9, query=qi)), qi
        assert all(abs(o) < 2e-3 for o in _probe(device, dtype, 70, qi + 1, portion, 9, query=qi)), qi
    out = _probe(device, dtype, 1, 0, [1], 4, score=1.0, sink=[1.0, 1.0 + math.log(3.0)])
    assert abs(out[0] - 0.5) < 2e-3 and abs(out[1] - 0.25) < 2e-3, out
    out = _probe(device, dtype, n, n - 33, por, 40, sink=[30.0, -50.0], gate=[0.0, math.log(3.0)])
    assert abs(out[0] - 0.25) < 2e-3 and abs(out[1] - 0.75) < 2e-3, out
    out = _probe(device, dtype, n, n - 33, por, 40, sink=[80.0, 30.0 + math.log(3.0)])
    assert abs(out[0]) < 2e-3 and abs(out[1] - 0.25) < 2e-3, out


@_GPU
@pytest.mark.parametrize("dk,dv,H,G", [(128, 128, 8, 2), (64, 64, 4, 4), (64, 128, 12, 2), (128, 64, 5, 1), (96, 64, 6, 3),
                                       (32, 32, 33, 1), (256, 256, 4, 2), (48, 80, 6, 2), (128, 128, 130, 1)])
def test_window_edges_bf16_kernels(dk, dv, H, G):
    """The same stand-out keys in bf16: head sizes and group sizes that take the matrix-core kernels (one, few and more than
    a hundred heads per kv head) beside sizes off their grid, windows on and off the kernels' key blocks, in prompts, portions
    and single-token steps."""
    dt = torch.bfloat16
    sink = [30.0 if h % 2 else -50.0 for h in range(H)]
    gate = [0.0 if h % 3 == 0 else 30.0 for h in range(H)]
    for portion in ([1000], [170, 140, 9, 11], [219, 3, 107], [329, 1]):
        for window in (16, 33, 64, 100):
            kw = dict(H=H, G=G, dk=dk, dv=dv)
            for qi in (329, 310, 303):
                inside = _probe("cuda", dt, 330, qi - window + 1, portion, window, query=qi, **kw)
                outside = _probe("cuda", dt, 330, qi - window, portion, window, query=qi, **kw)
                assert all(abs(o - 1.0) < 0.03 for o in inside), (portion, window, qi, inside)
                assert all(abs(o) < 0.03 for o in outside), (portion, window, qi, outside)
        out = _probe("cuda", dt, 330, 300, portion, 50, sink=sink, gate=gate, **kw)
        for h, o in enumerate(out):
            assert abs(o - (0.5 if h % 2 else 1.0) * (0.5 if h % 3 == 0 else 1.0)) < 0.04, (portion, h, o)


@_GPU
@pytest.mark.parametrize("dk,dv,H,G", [(128, 128, 8, 2), (64, 64, 6, 6), (64, 128, 12, 3), (128, 64, 4, 1), (96, 96, 10, 2),
                                       (40, 24, 6, 2), (64, 64, 128, 1)])
@pytest.mark.parametrize("window", [0, 1, 40, 200])
def test_grouped_attention_bf16_against_reference(dk, dv, H, G, window):
    """Unequal requests in one step - prompts, a continued portion, single tokens - with sinks and head gates through the
    bf16 kernels against the fp32 reference of the same op on the same (bf16-rounded) values; then steps of single tokens."""
    g = torch.Generator().manual_seed(1)
    rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    for ctx, qlen in (([300, 77, 513, 40], [300, 20, 1, 1]), ([300, 77, 1, 705], [1, 1, 1, 1]), ([90], [64]), ([33, 5], [2, 5])):
        S = len(ctx)
        nb = [(c + B - 1) // B for c in ctx]
        perm = torch.randperm(sum(nb) + 2, generator=g).tolist()
        bt = torch.zeros(S, max(nb), dtype=torch.int32)
        for s in range(S):
            bt[s, :nb[s]] = torch.tensor(perm[sum(nb[:s]):sum(nb[:s + 1])], dtype=torch.int32)
        kc, vc = rn(sum(nb) + 2, G, B, dk).to(torch.bfloat16), rn(sum(nb) + 2, G, dv, B).to(torch.bfloat16)
        T = sum(qlen)
        q = (rn(T, H * dk) * 2 * dk ** -0.5).to(torch.bfloat16)
        proj = rn(T, H + 5).to(torch.bfloat16)           # the gates are a column slice of a wider projection
        sink = rn(H) * 2
        cu = torch.tensor([sum(qlen[:s]) for s in range(S + 1)], dtype=torch.int32)
        args = (bt, cu, torch.tensor(ctx, dtype=torch.int32))
        want = ops.window_attention(q.float(), kc.float(), vc.float(), *args, H, G, dk, dv, 0.9, window=window, sink=sink,
                                    gate=proj[:, 3:3 + H].float())
        got = ops.window_attention(q.cuda(), kc.cuda(), vc.cuda(), *[a.cuda() for a in args], H, G, dk, dv, 0.9, window=window,
                                   sink=sink.cuda(), gate=proj.cuda()[:, 3:3 + H]).float().cpu()
        e = (got - want).norm(dim=-1) / want.norm(dim=-1)
        assert e.max() < 1e-2, (ctx, float(e.max()), int(e.argmax()))


@_GPU
@pytest.mark.parametrize("dk,dv,H,G", [(128, 128, 8, 2), (32, 32, 4, 1), (160, 160, 4, 2), (192, 128, 3, 1), (192, 192, 2, 1), (256, 256, 4, 2)])
@pytest.mark.parametrize("window", [0, 2500])
def test_grouped_attention_long_shares(dk, dv, H, G, window):
    """Single-token steps whose waves walk shares of one to five key blocks, the last of them partly past the sequence, against the fp32
    reference of the same op (the tolerance of the test above)."""
    g = torch.Generator().manual_seed(dk)
    rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    ctx = [4097, 3100, 2049, 33, 1, 4640]
    S, nb = len(ctx), [(c + B - 1) // B for c in ctx]
    perm = torch.randperm(sum(nb), generator=g).tolist()
    bt = torch.zeros(S, max(nb), dtype=torch.int32)
    for s in range(S):
        bt[s, :nb[s]] = torch.tensor(perm[sum(nb[:s]):sum(nb[:s + 1])], dtype=torch.int32)
    kc, vc = rn(sum(nb), G, B, dk).to(torch.bfloat16), rn(sum(nb), G, dv, B).to(torch.bfloat16)
    q, sink = (rn(S, H * dk) * 2 * dk ** -0.5).to(torch.bfloat16), rn(H) * 2
    args = (bt, torch.arange(S + 1, dtype=torch.int32), torch.tensor(ctx, dtype=torch.int32))
    want = ops.window_attention(q.float(), kc.float(), vc.float(), *args, H, G, dk, dv, 0.9, window=window, sink=sink)
    got = ops.window_attention(q.cuda(), kc.cuda(), vc.cuda(), *[a.cuda() for a in args], H, G, dk, dv, 0.9, window=window,
                               sink=sink.cuda()).float().cpu()
    e = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert e.max() < 1e-2, (float(e.max()), int(e.argmax()))


@pytest.mark.parametrize("device,dtype", FP32_TARGETS)
def test_window_edge_in_model(device, dtype):
    """One attention layer with nearly even weights: changing the token at the window's last position moves the logits,
    changing the one before it leaves them as they were - oracle and framework, in a prompt and decoded."""
    w = 21
    cfg = O.make_config([O.no_ff(O.att(heads=2, kv_heads=2, dim=8, vdim=8, window=w, scale=0.2))])
    sd = O.random_checkpoint(cfg, 71)
    a = tokens(60, 96, 72)
    eng = make_engine(cfg, sd, device, dtype)
    for j, moves in ((59 - w + 1, True), (59 - w, False)):
        b = list(a)
        b[j] = (b[j] + 31) % 96
        wa, wb = O.forward(cfg, sd, a), O.forward(cfg, sd, b)
        assert (row_err(wb[-1:], wa[-1:]).item() > 1e-3) == moves
        for i, sizes in enumerate(([60], [59, 1], [40, 2, 7, 1])):
            got = run_schedule(eng, {f"a{j}{i}": a, f"b{j}{i}": b}, [[(n, c)] for n in (f"a{j}{i}", f"b{j}{i}") for c in cuts(60, sizes)])
            assert close(got[f"a{j}{i}"], wa, dtype) and close(got[f"b{j}{i}"], wb, dtype)


# -------------------------------------------------------------------------- entry points: registry, generation, runner
def _write_checkpoint(path, cfg, sd):
    from safetensors.torch import save_file
    os.makedirs(path, exist_ok=True)
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(cfg, f)
    save_file({k: v.to(torch.bfloat16).contiguous() for k, v in sd.items()}, os.path.join(path, "model.safetensors"))


def _is_greedy(cfg, sd, prompt, out):
    """out continues prompt by the oracle's argmax, up to a near-tie of its top logits."""
    seq = list(prompt) + [int(t) for t in out]
    rows = O.forward(cfg, sd, seq)[len(prompt) - 1:-1]
    for row, t in zip(rows, out):
        assert row[t] >= row.max() - 1e-3 * (row.max() - row.min()), (int(t), int(row.argmax()))


@pytest.mark.parametrize("device,dtype", FP32_TARGETS)
def test_greedy_generation_through_engine(tmp_path, device, dtype):
    """A checkpoint directory -> registry -> LLMEngine.generate (its scheduler with chunked prefill, cache, sampling): greedy
    continuations of three prompts served together equal the oracle's. Nothing but KV pages is carried from step to step,
    so a second round whose prompts share a cached prefix reuses those pages and gives the same continuations."""
    cfg = O.make_config(FULL, width=32, vocab=96, loop=LOOP)
    sd = O.random_checkpoint(cfg, 31)
    _write_checkpoint(str(tmp_path / "m"), cfg, sd)
    model, tok, _ = build_llm(weights=str(tmp_path / "m"), device=device, dtype=dtype)
    assert isinstance(model, BamanexModel)
    eng = LLMEngine(model, tok, EngineConfig(max_num_seqs=4, num_blocks=32, max_model_len=256, prefill_chunk=16,
                                             max_batched_tokens=24, prefix_cache=True, use_graphs=device != "cpu",
                                             graph_batch_sizes=(1, 2, 4), decode_steps=1))
    prompts = [tokens(n, 96, 40 + n) for n in (9, 43, 2)]
    greedy = SamplingParams(max_tokens=12, temperature=0.0, ignore_eos=True)
    for p, o in zip(prompts, eng.generate(prompts, greedy)):
        assert len(o.output_ids) == 12
        _is_greedy(cfg, sd, p, o.output_ids)
    before = eng.stats["prefill_tokens"]
    again = [prompts[1][:36] + [7, 8], prompts[1]]
    for p, o in zip(again, eng.generate(again, greedy)):
        _is_greedy(cfg, sd, p, o.output_ids)
    assert eng.stats["prefill_tokens"] - before < len(again[0]) + len(again[1])   # cached pages were not computed again


def test_preset_and_generation_cpu():
    model, tok, name = build_llm("tiny-bamanex", device="cpu", dtype=torch.float32)
    assert name == "tiny-bamanex" and isinstance(model, BamanexModel) and len(model.runs) == 6
    eng = LLMEngine(model, tok, EngineConfig(max_num_seqs=2, num_blocks=16, max_model_len=128, use_graphs=False))
    outs = eng.generate([[1, 2, 3], [4, 5]], SamplingParams(max_tokens=5, temperature=0.0, ignore_eos=True))
    assert [len(o.output_ids) for o in outs] == [5, 5]


@pytest.mark.parametrize("device", [pytest.param("cpu", id="cpu"), pytest.param("cuda:0", id="gpu", marks=_GPU)])
def test_runner_script(tmp_path, device):
    """The replay script: steps on stdin, logits files out, pages reused within a pool made for the live requests only."""
    cfg = O.make_config(FULL, width=32, vocab=96, loop=LOOP)
    sd = O.random_checkpoint(cfg, 33)
    _write_checkpoint(str(tmp_path / "m"), cfg, sd)
    a, b = clear_tokens(40, cfg, sd, 1), clear_tokens(21, cfg, sd, 70)
    wa, wb = O.forward(cfg, sd, a), O.forward(cfg, sd, b)
    steps = [dict(step=0, entries=[dict(id="a", tokens=a[:30], want=[0, 29])], end=[]),
             dict(step=1, entries=[dict(id="a", tokens=a[30:31], want=[0]), dict(id="b", tokens=b[:20], want=[19])], end=[]),
             dict(step=2, entries=[dict(id="b", tokens=b[20:], want=[])], end=["b"]),
             dict(step=3, entries=[dict(id="a", tokens=a[31:], want=[8])], end=["a"]),
             dict(step=4, entries=[dict(id="c", tokens=b, want=[20])], end=["c"])]
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = tmp_path / "out"
    p = subprocess.run([sys.executable, os.path.join(root, "bin", "trace_run"), "--model", str(tmp_path / "m"), "--dtype",
                        "float32", "--out", str(out), "--max-tokens", "128", "--device", device],
                       input="\n".join(json.dumps(s) for s in steps) + "\n", capture_output=True, text=True, timeout=600)
    assert p.returncode == 0, p.stderr[-2000:]
    assert [l for l in p.stdout.splitlines() if l.startswith("done")] == [f"done {i}" for i in range(5)]
    import numpy as np
    rd = lambda i: torch.from_numpy(np.fromfile(str(out / f"{i}.f32"), dtype="<f4").reshape(-1, 96))  # noqa: E731
    err = lambda got, want: row_err(got, want).max().item()  # noqa: E731
    assert err(rd(0), wa[[0, 29]]) < 1e-4 and err(rd(1), torch.stack([wa[30], wb[19]])) < 1e-4
    assert not (out / "2.f32").exists()
    assert err(rd(3), wa[39:40]) < 1e-4 and err(rd(4), wb[20:21]) < 1e-4


def test_config_errors():
    base = O.make_config(FULL, loop=LOOP)

    def bad(edit):
        c = json.loads(json.dumps(base))
        edit(c)
        with pytest.raises(ValueError):
            BamanexConfig.from_json(c)

    BamanexConfig.from_json(base)
    bad(lambda c: c["layers"][0].update(type="conv"))
    bad(lambda c: c["layers"][0]["mlp"].update(kind="sparse"))
    bad(lambda c: c["layers"][1]["mlp"]["router"].update(top=7))      # more than there are experts
    bad(lambda c: c["layers"][0]["mixer"].update(kv_heads=4))         # six heads do not share four kv heads
    bad(lambda c: c["layers"][0]["mixer"]["rot"].update(dims=5))      # odd
    bad(lambda c: c["layers"][0]["mixer"]["rot"].update(dims=10))     # more than a head has
    bad(lambda c: c["loop"].update(stop=9))
    bad(lambda c: c["loop"].update(start=3))
    with pytest.raises(ValueError):
        ops.rotary_half_kv_write(*[torch.zeros(1, 4)] * 3, torch.zeros(1), torch.zeros(1), None, None, 1, 1, 4, 4,
                                 torch.zeros(3, dtype=torch.float64))


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,G,D,n", [(1, 16, 4, 128, 32), (16, 16, 4, 128, 32), (17, 8, 8, 64, 32), (33, 4, 2, 256, 40), (64, 16, 4, 128, 0)])
@pytest.mark.parametrize("N,K", [(2048, 5632), (1040, 6144)])
def test_rotation_beside_a_product(cuda, T, H, G, D, n, N, K):
    """The rotation and cache write in the launch of a product's K slices: the bits of both by themselves. A head size that the shared
    launch does not take (96) and a row-major weight run one after the other."""
    torch.manual_seed(T + D)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    for d in (D, 96):
        qkv, x, w = bf(T, (H + 2 * G) * d), bf(T, K), bf(N, K)
        pos = torch.randint(0, 4000, (T,), device=cuda, dtype=torch.int32)
        slots = torch.randperm(8 * 16, device=cuda)[:T].to(torch.int32)
        freq = ops.rope_inv_freq(2 * n, 10000.0, None).to(cuda) if n else torch.zeros(0, dtype=torch.float64, device=cuda)
        want = ops.linear_partial(x, w)
        assert ops.linear_partial_later(x, w) is None   # row-major
        assert ops.to_fragment_layout_(w)
        outs = []
        for beside in (None, ops.linear_partial_later(x, w)):
            kc, vc = torch.zeros(8, G, 16, d, device=cuda, dtype=torch.bfloat16), torch.zeros(8, G, d, 16, device=cuda, dtype=torch.bfloat16)
            q = ops.rotary_half_kv_write(qkv[:, :H * d], qkv[:, H * d:(H + G) * d], qkv[:, (H + G) * d:], pos, slots, kc, vc, H, G, d, d,
                                         freq, 1e-6, beside=beside)
            outs.append((q, kc, vc))
        assert all(torch.equal(a, b) for a, b in zip(*outs))
        assert torch.equal(beside.slabs, want.slabs)


def test_slices_still_to_be_made():
    """A product whose slices a later launch makes: nothing reads them before, nothing makes them twice."""
    t = torch.zeros(2, 3, 8)
    later, there = ops.Partial(t, None, (t, t)), ops.Partial(t)
    assert there.index_select(0, torch.tensor([1])).slabs.shape == (2, 1, 8)
    with pytest.raises(RuntimeError):
        later.index_select(0, torch.tensor([1]))
    for a, b in ((later, None), (None, later), (there, later)):
        with pytest.raises(RuntimeError):
            ops.parallel_add_norm_f32(torch.zeros(3, 8), a, None, b)
    with pytest.raises(RuntimeError):
        ops.rotary_half_kv_write(*[torch.zeros(1, 4)] * 3, torch.zeros(1), torch.zeros(1), None, None, 1, 1, 4, 4,
                                 torch.zeros(2, dtype=torch.float64), beside=there)


@pytest.mark.gpu
def test_slices_made_beside_the_rotation(cuda):
    x, w = torch.zeros(3, 5632, device=cuda).bfloat16(), torch.zeros(2048, 5632, device=cuda).bfloat16()
    assert ops.to_fragment_layout_(w)
    p, qkv = ops.linear_partial_later(x, w), torch.zeros(3, 3 * 64, device=cuda).bfloat16()
    at = torch.arange(3, device=cuda, dtype=torch.int32)
    kc, vc = torch.zeros(1, 1, 16, 64, device=cuda).bfloat16(), torch.zeros(1, 1, 64, 16, device=cuda).bfloat16()
    freq, q = torch.ones(32, dtype=torch.float64, device=cuda), torch.empty(3, 64, device=cuda).bfloat16()
    rows = (qkv[:, :64], qkv[:, 64:128], qkv[:, 128:], at, at)
    ops.rotary_half_kv_write(*rows, kc, vc, 1, 1, 64, 64, freq, beside=p)
    assert p.made() is p and not p.slabs.any()
    for w_, ws in ((None, p.slabs), (w, None)):
        with pytest.raises(RuntimeError, match="without its weight or slices"):
            ops.native().rotary_half_kv_write(*rows, q, kc, vc, 1, 1, 64, 64, freq, -1.0, x, w_, ws)
