"""Weight-streaming split-K decode GEMM (M <= 64) vs the fp32 reference of the same op."""
import math

import pytest
import torch

from generativeaiexamples_amd import ops
from generativeaiexamples_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


def _run(x, w, bias, res, epi, out_dtype):
    M, K = x.shape
    N = w.shape[0]
    ncol = N // 2 if epi == 4 else N
    out = torch.empty(M, ncol, device="cuda", dtype=out_dtype)
    nat = ops.native()
    ws = torch.empty(nat.gemm_splitk_ws_floats(M, N, K), device="cuda", dtype=torch.float32)
    nat.gemm_splitk(x, w, out, bias, res, epi, ws)
    return out


@pytest.mark.parametrize("M", [1, 7, 16, 17, 33, 64])
@pytest.mark.parametrize("N,K", [(1000, 512), (6144, 4096), (4096, 14336)])
def test_splitk_plain(cuda, M, N, K):
    torch.manual_seed(M * 7 + N)
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    y = _run(x, w, None, None, 0, torch.float32)
    r = ref.linear(x.cpu(), w.cpu(), out_dtype=torch.float32)
    torch.testing.assert_close(y.cpu(), r, rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("act", ["bias", "gelu", "relu", "quick_gelu", "residual", "bias_residual", "swiglu"])
def test_splitk_epilogues(cuda, act):
    M, N, K = 24, 2048, 4096
    torch.manual_seed(3)
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    bias = torch.randn(N, device="cuda", dtype=torch.bfloat16) if "bias" in act or act in ("gelu", "relu", "quick_gelu") else None
    res = torch.randn(M, N, device="cuda", dtype=torch.bfloat16) if "residual" in act else None
    y = _run(x, w, bias, res, ops.EPI[act], torch.bfloat16)
    a = act if act in ("gelu", "relu", "quick_gelu", "swiglu") else None
    r = ref.linear(x.cpu(), w.cpu(), None if bias is None else bias.cpu(), None if res is None else res.cpu(), a,
                   torch.float32)
    torch.testing.assert_close(y.float().cpu(), r, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("M,N,K,epi", [
    (1, 16, 512, "bias"), (16, 1040, 1024, "gelu"), (17, 64, 1536, "residual"), (31, 96, 2560, "swiglu"),
    (32, 1024, 4096, "bias_residual"), (33, 2064, 512, None), (64, 4096, 2560, "relu"), (64, 2048, 2048, "quick_gelu"),
    (49, 3104, 1024, "geglu"), (5, 6160, 1024, None), (24, 5136, 1536, "bias"), (64, 3264, 2560, "bias"), (33, 3232, 2560, "swiglu"),
    (9, 2048, 4096, "gelu")])
@pytest.mark.parametrize("frag,f32", [(False, False), (True, False), (False, True)])
def test_one_launch_gemm(cuda, M, N, K, epi, frag, f32):
    """Narrow decode projections in one launch (all of K in a workgroup): row tiles 16 / 32 / 64 with ragged M, one and
    two column fragments with a half-empty last pair, 1 to 5 activation stages with a short last one; weights past 16 MiB
    (64 x 4096 x 2560) keep the split kernels. Bound per element: K fp32 products in any order, K 2^-24 sum |x w|, then what the epilogue's own steps can move, and one bf16 rounding."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(torch.bfloat16)
    bias = torch.randn(N, generator=g).to(torch.bfloat16) if epi in ("bias", "gelu", "relu", "quick_gelu", "bias_residual") \
        else None
    res = torch.randn(M, N, generator=g).to(torch.bfloat16) if epi in ("residual", "bias_residual") else None
    dev = [None if t is None else t.cuda() for t in (x, ops.shuffle_fragments(w) if frag else w, bias, res)]
    ncol = N // 2 if epi in ("swiglu", "geglu") else N
    out = torch.full((M, ncol), float("nan"), device="cuda", dtype=torch.float32 if f32 else torch.bfloat16)
    nat = ops.native()
    assert (nat.gemm_slim_nf(M, N, K, epi in ("swiglu", "geglu")) > 0) == (N * K <= 8 << 20)
    ws = torch.empty(nat.gemm_splitk_ws_floats(M, N, K), device="cuda", dtype=torch.float32)
    nat.gemm_splitk(dev[0], dev[1], out, dev[2], dev[3], ops.EPI[epi] if epi else 0, ws, frag)
    y = x.double() @ w.double().t()
    if bias is not None:
        y = y + bias.double()
    e = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    if epi in ("swiglu", "geglu"):
        y, e = (t.view(M, N // 32, 2, 16) for t in (y, e))
        a, u = y[:, :, 0], y[:, :, 1]
        act = torch.nn.functional.silu(a) if epi == "swiglu" else torch.nn.functional.gelu(a, approximate="tanh")
        # both gates have slopes below 1.13; the hardware exp / tanh forms stay within 2^-18 of the value
        e = 1.13 * e[:, :, 0] * u.abs() + act.abs() * e[:, :, 1] + 2.0 ** -18 * (act * u).abs() + 1e-6
        y, e = (act * u).reshape(M, ncol), e.reshape(M, ncol)
    elif epi in ("gelu", "quick_gelu", "relu"):
        y = {"gelu": torch.nn.functional.gelu, "relu": torch.relu, "quick_gelu": lambda t: t * torch.sigmoid(1.702 * t)}[epi](y)
        e = 1.13 * e + 2.0 ** -18 * y.abs() + 1e-6
    if res is not None:
        e = e + (0 if f32 else 2.0 ** -8 * y.abs())  # bf16 product, then the sum rounded again
        y = y + res.double()
    e = e + (2.0 ** -23 if f32 else 2.0 ** -8) * y.abs()
    d = (out.double().cpu() - y).abs()
    assert (d <= e).all(), (d / e).max()


def test_linear_routes_decode_to_splitk(cuda):
    """ops.linear for M <= 64 uses the decode kernels and matches the reference."""
    x = torch.randn(64, 4096, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(28672, 4096, device="cuda") / 64).to(torch.bfloat16)
    y = ops.linear(x, w, act="swiglu")
    r = ref.linear(x.cpu(), w.cpu(), act="swiglu", out_dtype=torch.float32)
    torch.testing.assert_close(y.float().cpu(), r, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("M", [5, 16, 40, 64])
@pytest.mark.parametrize("act", [None, "bias", "gelu", "residual", "swiglu"])
def test_splitk_wide_single_pass_epilogue(cuda, M, act):
    """N >= 256 column tiles -> one workgroup pass over K (KS = 1): the epilogue runs inside the GEMM kernel
    (4-wave in-workgroup K reduction through LDS), including a partial last column tile."""
    N, K = (16448 if act == "swiglu" else 16400), 1024
    torch.manual_seed(M + 11)
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(torch.bfloat16)
    bias = torch.randn(N, device="cuda", dtype=torch.bfloat16) if act in ("bias", "gelu") else None
    res = torch.randn(M, N, device="cuda", dtype=torch.bfloat16) if act == "residual" else None
    assert ops.native().gemm_splitk_ws_floats(M, N, K) == M * N  # KS == 1
    out_dtype = torch.float32 if act is None else torch.bfloat16
    y = _run(x, w, bias, res, ops.EPI[act] if act else 0, out_dtype)
    a = act if act in ("gelu", "swiglu") else None
    r = ref.linear(x.cpu(), w.cpu(), None if bias is None else bias.cpu(), None if res is None else res.cpu(), a,
                   torch.float32)
    tol = 2e-3 if out_dtype == torch.float32 else 2e-2
    torch.testing.assert_close(y.float().cpu(), r, rtol=tol, atol=tol)


@pytest.mark.parametrize("M", [1, 17, 64])
@pytest.mark.parametrize("act", [None, "swiglu", "residual", "bias"])
@pytest.mark.parametrize("N,K", [(4096, 14336), (6144, 4096), (2048, 1024)])
def test_preshuffled_weights_match(cuda, M, act, N, K):
    """Decode GEMM on fragment-shuffled weights (both split-K kernel variants) == plain layout."""
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=cuda).bfloat16()
    w = (torch.randn(N, K, device=cuda) * 0.02).bfloat16()
    b = (torch.randn(N, device=cuda) * 0.1).bfloat16() if act in ("bias", "gelu") else None
    r = torch.randn(M, N, device=cuda).bfloat16() if act == "residual" else None
    a = act if act == "swiglu" else None
    want = ops.linear(x, w, bias=b, residual=r, act=a).float()
    w2 = w.clone()
    assert ops.preshuffle_weight(w2)
    # the fragment copy is a permutation of the weight
    assert torch.equal(ops.shuffle_fragments(w2).view(-1).sort().values, w2.view(-1).sort().values)
    got = ops.linear(x, w2, bias=b, residual=r, act=a).float()
    assert (got - want).abs().max() <= 2e-2 * (want.abs().max() + 1)


def test_engine_preshuffles_projections(cuda):
    from generativeaiexamples_amd.models import LlamaConfig, LlamaModel

    m = LlamaModel(LlamaConfig.tiny(), device=cuda).random_init(0)
    added = m.preshuffle_decode_weights()
    assert added > 0 and ops.decode_operand(m.w["l0.down"]) is not None  # K=512 qualifies
    assert ops.decode_operand(m.w["l0.attn_norm"]) is None


def test_preshuffle_budget_takes_whole_kinds_by_priority(cuda):
    """A budget that holds gate_up + down but nothing else copies exactly those kinds (every layer)."""
    from generativeaiexamples_amd.models import LlamaConfig, LlamaModel

    m = LlamaModel(LlamaConfig.tiny(hidden_size=512, intermediate_size=1024, num_heads=8), device=cuda).random_init(0)
    size = lambda kind: sum(v.numel() * v.element_size() for k, v in m.w.items()  # noqa: E731
                            if k.rsplit(".", 1)[-1] == kind)
    for kind in ("gate_up", "down", "o"):
        assert all(ops.psw_qualifies(v) for k, v in m.w.items() if k.rsplit(".", 1)[-1] == kind), kind
    budget = size("gate_up") + size("down") + 1  # nothing after them fits
    assert m.preshuffle_decode_weights(budget_bytes=budget) == size("gate_up") + size("down")
    for i in range(m.cfg.num_layers):
        assert ops.decode_operand(m.w[f"l{i}.gate_up"]) is not None
        assert ops.decode_operand(m.w[f"l{i}.down"]) is not None
        assert ops.decode_operand(m.w[f"l{i}.qkv"]) is None and ops.decode_operand(m.w[f"l{i}.o"]) is None
    assert ops.decode_operand(m.w["lm_head"]) is None


@pytest.mark.parametrize("M", [1, 17, 64])
@pytest.mark.parametrize("K", [4096, 14336])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("psw", [False, True])
def test_linear_add_rmsnorm_decode_tail(cuda, M, K, bias, psw):
    """Decode tail residual += x.W^T (+ b); out = rmsnorm(residual) * g: natural layout (LDS-staged decode
    GEMM + residual-add norm) and fragment-shuffled layout (split-K + fused reduce/norm) vs fp32 reference
    with the same bf16 roundings."""
    N = 4096
    torch.manual_seed(M + K + bias)
    x = torch.randn(M, K, device=cuda).bfloat16()
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).bfloat16()
    b = (torch.randn(N, device=cuda) * 0.1).bfloat16() if bias else None
    res = torch.randn(M, N, device=cuda).bfloat16()
    g = (1 + 0.1 * torch.randn(N, device=cuda)).bfloat16()
    if psw:
        assert ops.preshuffle_weight(w)
    res_ref = res.clone()
    h = ref.linear(x.cpu(), w.cpu(), None if b is None else b.cpu(), out_dtype=torch.float32).bfloat16()
    r_ref = (h.float() + res_ref.cpu().float()).bfloat16()
    o_ref = r_ref.float() * torch.rsqrt(r_ref.float().pow(2).mean(-1, keepdim=True) + 1e-5) * g.cpu().float()
    out = ops.linear_add_rmsnorm(x, w, res, g, 1e-5, bias=b)
    torch.testing.assert_close(res.float().cpu(), r_ref.float(), rtol=1e-2, atol=2e-2)
    torch.testing.assert_close(out.float().cpu(), o_ref, rtol=2e-2, atol=3e-2)


@pytest.mark.parametrize("M", [1, 2, 16, 31, 64])
@pytest.mark.parametrize("N,K,act", [(28672, 4096, "swiglu"), (32000, 4096, None), (16384, 14336, "residual"),
                                     (18432, 4096, "bias"), (16384, 2048, "gelu")])
@pytest.mark.parametrize("psw", [False, True])
def test_decode_gemm_natural_layout(cuda, M, N, K, act, psw):
    """The LDS-staged decode GEMM (gemm_decode.hip, wide projections) vs the fp32 reference: Llama-3-8B
    gate_up+SwiGLU, a 32K-vocab LM head (fp32 logits), deep K + residual, bias, bias+GELU; on the natural
    [N, K] layout and on the fragment-shuffled copy (full-line non-temporal weight stream)."""
    torch.manual_seed(M * 3 + N)
    x = torch.randn(M, K, device=cuda).bfloat16()
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).bfloat16()
    b = (torch.randn(N, device=cuda) * 0.1).bfloat16() if act in ("bias", "gelu") else None
    r = torch.randn(M, N, device=cuda).bfloat16() if act == "residual" else None
    epi = ops.EPI[act]
    assert ops.native().gemm_dec2_ok(M, N, K, epi), "shape should take the LDS-staged decode kernel"
    out_dtype = torch.float32 if act is None else torch.bfloat16
    if psw:
        assert ops.preshuffle_weight(w)
        y = ops.linear(x, w, bias=b, residual=r, act=act if act in ("swiglu", "gelu") else None,
                       out_dtype=out_dtype)
    else:
        y = _run(x, w, b, r, epi, out_dtype)
    want = ref.linear(x.cpu(), w.cpu(), None if b is None else b.cpu(), None if r is None else r.cpu(),
                      act if act in ("swiglu", "gelu") else None, torch.float32)
    tol = 2e-3 if out_dtype == torch.float32 else 2e-2
    torch.testing.assert_close(y.float().cpu(), want, rtol=tol, atol=tol)


@pytest.mark.parametrize("M", [1, 17, 64])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("kv_fp8", [False, True])
@pytest.mark.parametrize("psw", [False, True])
@pytest.mark.parametrize("tail", [True, False])
def test_linear_rope_kv_fused_matches_unfused(cuda, monkeypatch, M, bias, kv_fp8, psw, tail):
    """Decode QKV tail fused into the split-K reduce (partials -> bias -> bf16 -> RoPE -> q / paged K, V^T)
    matches linear + rope_kv_write to the last bit on all but a handful of elements, bf16 and fp8 caches;
    tail: the reduce runs in the GEMM launch (last-arriving K-slice), else in the splitk_rope_kv launch."""
    monkeypatch.setattr(ops, "_QKV_TAIL", tail)
    Hq, Hkv, D, K = 32, 8, 128, 4096
    N = (Hq + 2 * Hkv) * D
    torch.manual_seed(M * 5 + bias + 2 * kv_fp8)
    x = torch.randn(M, K, device=cuda).bfloat16()
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).bfloat16()
    b = (torch.randn(N, device=cuda) * 0.1).bfloat16() if bias else None
    if psw:
        assert ops.preshuffle_weight(w)
    cs = ops.rope_cos_sin(4096, D, 500000.0, device=cuda)
    pos = torch.randint(0, 4000, (M,), device=cuda, dtype=torch.int32)
    nblk = 64
    slots = torch.randperm(nblk * 16, device=cuda)[:M].to(torch.int32)
    slots[0] = -1  # a padded row: no cache write
    kvd = torch.float8_e4m3fn if kv_fp8 else torch.bfloat16
    ks, vs = (0.05, 0.04) if kv_fp8 else (1.0, 1.0)
    outs = []
    for fused in (True, False):
        q = torch.zeros(M, Hq, D, device=cuda, dtype=torch.bfloat16)
        kc = torch.zeros(nblk, Hkv, 16, D, device=cuda, dtype=kvd)
        vc = torch.zeros(nblk, Hkv, D, 16, device=cuda, dtype=kvd)
        if fused:
            ops.linear_rope_kv(x, w, b, pos, cs, slots, q, kc, vc, Hq, Hkv, D, ks, vs)
        else:
            qkv = ops.linear(x, w, bias=b)
            ops.rope_kv_write(qkv, pos, cs, slots, q, kc, vc, Hq, Hkv, D, True, ks, vs)
        outs.append((q, kc.view(torch.uint8) if kv_fp8 else kc, vc.view(torch.uint8) if kv_fp8 else vc))
    # same partials, summation order and roundings; hipcc may contract the rotation's mul-sub into an FMA
    # differently at the two call sites, so a value that cancels to ~0 can differ in its last bit
    for a, r in zip(outs[0], outs[1]):
        if a.dtype == torch.uint8:  # fp8 codes: at most a handful one code apart
            assert (a != r).sum().item() <= max(2, a.numel() // 10000)
        else:
            torch.testing.assert_close(a.float(), r.float(), rtol=1e-2, atol=1e-5)
            assert (a != r).sum().item() <= max(2, a.numel() // 10000)
    if M > 1:  # row 0 is padded (no cache write)
        assert outs[0][1].float().abs().sum() > 0  # the cache was written
    if tail:
        assert int(ops.tail_counters(cuda).abs().sum()) == 0  # every ticket counter reset by its last arriver


def test_qkv_tail_graph_replays(cuda):
    """In-launch QKV tail under graph replay: counters reset themselves, every replay equals the eager result."""
    Hq, Hkv, D, K, M = 32, 8, 128, 4096, 64
    N = (Hq + 2 * Hkv) * D
    torch.manual_seed(3)
    x = torch.randn(M, K, device=cuda).bfloat16()
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).bfloat16()
    assert ops.preshuffle_weight(w)
    cs = ops.rope_cos_sin(4096, D, 500000.0, device=cuda)
    pos = torch.randint(0, 4000, (M,), device=cuda, dtype=torch.int32)
    slots = torch.randperm(64 * 16, device=cuda)[:M].to(torch.int32)
    kc = torch.zeros(64, Hkv, 16, D, device=cuda, dtype=torch.bfloat16)
    vc = torch.zeros(64, Hkv, D, 16, device=cuda, dtype=torch.bfloat16)
    q = torch.zeros(M, Hq, D, device=cuda, dtype=torch.bfloat16)
    ops.linear_rope_kv(x, w, None, pos, cs, slots, q, kc, vc, Hq, Hkv, D)
    want = (q.clone(), kc.clone(), vc.clone())
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops.linear_rope_kv(x, w, None, pos, cs, slots, q, kc, vc, Hq, Hkv, D)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ops.linear_rope_kv(x, w, None, pos, cs, slots, q, kc, vc, Hq, Hkv, D)
    for _ in range(10):
        q.zero_(); kc.zero_(); vc.zero_()  # noqa: E702
        g.replay()
        torch.cuda.synchronize()
        for a, b in zip((q, kc, vc), want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("M,N,K,ks", [(1, 1024, 4096, 4), (27, 1024, 4096, 4), (33, 1024, 1024, 2), (64, 2048, 4096, 2),
                                      (17, 384, 1536, 3), (16, 768, 3072, 3), (5, 16, 4096, 8), (31, 512, 2560, 5),
                                      (40, 2048, 1536, 0), (65, 1024, 4096, 0)])
@pytest.mark.parametrize("frag", [False, True])
def test_product_in_slices_and_norm(cuda, M, N, K, ks, frag):
    """LayerNorm(product + bias + residual) with K in slices, against float64; shapes without slices take the two ops. Error:
    bf16 roundings of the product, of its sum with the residual and of the result (2^-9 each, the first two of values up to
    ~6, divided by the row's deviation of ~1.4 and scaled by gains up to ~4)."""
    torch.manual_seed(M + N)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    x, w, bias, r, g, b = bf(M, K), bf(N, K) * K ** -0.5, bf(N), bf(M, N), bf(N), bf(N)
    assert (ops.native().gemm_slim_ks(M, N, K) if M <= 64 else 0) == ks
    wn = w.clone()
    if frag and ops.psw_qualifies(w):
        assert ops.to_fragment_layout_(w)
    y = ops.linear_layer_norm(x, w, bias, r, g, b, 1e-5)
    v = x.double() @ wn.double().t() + bias.double() + r.double()
    want = torch.nn.functional.layer_norm(v, (N,), g.double(), b.double(), 1e-5)
    assert ((y.double() - want).abs() <= 2.0 ** -8 * (want.abs() + 8 * g.double().abs())).all()
    odd = torch.empty(M * N + 1, device=cuda, dtype=torch.bfloat16)[1:].view(M, N).copy_(r)  # not on 16 bytes: the two ops
    z = ops.layer_norm(ops.linear(x, w, bias=bias, residual=odd), g, b, 1e-5)
    assert torch.equal(ops.linear_layer_norm(x, w, bias, odd, g, b, 1e-5), z)


@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N1,N2,K,one", [(11264, 3088, 2048, 64), (1120, 1040, 2048, 64), (1056, 1072, 6144, 0), (4128, 1072, 6144, 64), (1024, 1024, 1088, 0),
                                       (14336, 3088, 2048, 0), (18432, 4112, 2048, 64), (18432, 6144, 4096, 32), (28672, 6144, 3072, 0)])
def test_pair_of_products(cuda, M, N1, N2, K, one):
    """A gated product and one with a bias in one launch (up to ``one`` rows) or two, against float64: bf16 roundings of the result (2^-8 of it) and fp32 sums,
    the gate by approximate exponential and reciprocal (2^-20)."""
    torch.manual_seed(M + N1)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    x1, x2, w1, w2, b = bf(M, K), bf(M, K), bf(N1, K) * K ** -0.5, bf(N2, K) * K ** -0.5, bf(N2)
    gu = (x1.double() @ w1.double().t()).view(M, N1 // 32, 2, 16)
    want1 = (torch.nn.functional.gelu(gu[:, :, 0], approximate="tanh") * gu[:, :, 1]).reshape(M, -1)
    want2 = x2.double() @ w2.double().t() + b.double()
    assert (ops.to_fragment_layout_(w1) and ops.to_fragment_layout_(w2)) or K % 256
    assert ops.native().gemm_dec2_pair_ok(M, N1, N2, K) == (M <= one)
    y1, y2 = ops.linear_pair(x1, w1, x2, w2, b)
    for y, want in ((y1, want1), (y2, want2)):
        assert ((y.double() - want).abs() <= 2.0 ** -8 * 1.01 * want.abs() + 2e-5).all()


@pytest.mark.parametrize("M,N,K,parts", [(65, 2048, 1536, True), (96, 4096, 4096, True), (187, 4096, 14336, True), (193, 3088, 4096, True),
                                         (640, 4096, 4096, True), (640, 8192, 2048, False), (641, 4096, 4096, False), (200, 2032, 4096, False)])
@pytest.mark.parametrize("bias", [False, True])
def test_parts_added_by_the_rms_norm(cuda, M, N, K, parts, bias):
    """residual += product; rms norm, the parts of K added in the norm's launch, in both layouts of the weight and for a residual off
    16 bytes, against float64. Error: half a unit of bf16, at most 2^-8 of the value, for the product p, for its sum v with the
    residual and for the result; 2^-10 of it for the root mean square of thousands of such v and the fp32 sums."""
    torch.manual_seed(M + N)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    x, w, b, r, g = bf(M, K), bf(N, K) * K ** -0.5, bf(N) if bias else None, bf(M, N), bf(N)
    assert (ops.native().gemm_slabs_parts(M, N, K, False) > 1) == parts
    p = x.double() @ w.double().t() + (b.double() if bias else 0)
    v = p + r.double()
    inv = torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-5)
    want, off = v * inv * g.double(), 2.0 ** -8 * 1.01 * (p.abs() + v.abs()) + 1e-4
    odd = torch.empty(M * N + 1, device=cuda, dtype=torch.bfloat16)[1:].view(M, N).copy_(r)
    wf = w.clone()
    assert ops.to_fragment_layout_(wf)
    seen = []
    for wt, res in ((w, r.clone()), (wf, r.clone()), (wf, odd)):
        y = ops.linear_add_rmsnorm(x, wt, res, g, 1e-5, bias=b)
        assert ((res.double() - v).abs() <= off).all()
        assert ((y.double() - want).abs() <= 1.01 * off * inv * g.double().abs() + (2.0 ** -8 + 2.0 ** -10) * want.abs()).all()
        seen.append((res, y))
    assert torch.equal(seen[0][0], seen[1][0]) and torch.equal(seen[0][1], seen[1][1])


@pytest.mark.parametrize("M,N,K,layer,taken", [(385, 2048, 1024, False, False), (513, 4096, 3072, False, False), (400, 2048, 2048, False, True),
                                               (500, 2048, 3072, False, True), (513, 4096, 4096, False, True), (385, 1536, 768, True, False),
                                               (513, 1536, 1024, True, False), (65, 2048, 3072, True, False), (65, 2048, 1024, True, True),
                                               (385, 768, 1536, True, True), (212, 1088, 1920, True, False), (364, 1040, 4352, True, False)])
def test_slabs_where_they_are_the_faster_way(cuda, M, N, K, layer, taken):
    """Both sides of the line (timed at gai_gemm_mid_slabs_plan): products whose own sums and a norm after them take less are left to those."""
    assert (ops.native().gemm_slabs_parts(M, N, K, layer) > 1) == taken


@pytest.mark.parametrize("M,N,K", [(65, 1024, 1024), (187, 1024, 4096), (320, 768, 3072), (500, 384, 1536), (300, 2048, 4096), (640, 1024, 4096)])
def test_parts_added_by_the_layer_norm(cuda, M, N, K):
    """The same before a layer norm (error as in test_product_in_slices_and_norm), and rows with nothing beside them."""
    torch.manual_seed(M + N)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    x, w, bias, r, g, b = bf(M, K), bf(N, K) * K ** -0.5, bf(N), bf(M, N), bf(N), bf(N)
    assert ops.native().gemm_slabs_parts(M, N, K, True) > 1
    wf = w.clone()
    assert ops.to_fragment_layout_(wf)
    for bi, lb in ((bias, b), (None, None)):
        y = ops.linear_layer_norm(x, wf, bi, r, g, lb, 1e-5)
        v = x.double() @ w.double().t() + (bias.double() if bi is not None else 0) + r.double()
        want = torch.nn.functional.layer_norm(v, (N,), g.double(), None if lb is None else lb.double(), 1e-5)
        assert ((y.double() - want).abs() <= 2.0 ** -8 * (want.abs() + 8 * g.double().abs())).all()
        assert torch.equal(y, ops.linear_layer_norm(x, w, bi, r, g, lb, 1e-5))


@pytest.mark.parametrize("M", [1, 27, 64, 65, 300, 640, 641])
def test_linear_layer_norm_without_a_residual(cuda, M):
    """Nothing to add: the product's norm, as from the two operations."""
    torch.manual_seed(M)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    x, w, b, g = bf(M, 1024), bf(1024, 1024) / 32, bf(1024), bf(1024)
    want = ops.layer_norm(ops.linear(x, w, b), g, b, 1e-5)
    assert torch.equal(ops.linear_layer_norm(x, w, b, None, g, b, 1e-5), want)


@pytest.mark.parametrize("M,N,K,apart", [(2100, 1024, 1024, True), (4100, 512, 1024, True), (1300, 4096, 1024, True), (128, 1024, 1024, True), (8192, 1024, 1024, False),
                                         (2048, 4096, 1024, False), (641, 2048, 2048, False)])
def test_residual_in_the_product_or_the_norm(cuda, M, N, K, apart):
    """Both sides of the line between a residual added by the product's epilogue and by the norm (apart: the bits of the two operations)."""
    torch.manual_seed(M + N)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    x, w, r, g = bf(M, K), bf(N, K) * K ** -0.5, bf(M, N), bf(N)
    assert ops.native().gemm_residual_apart(M, N, K) == apart and ops._residual_in_product(x, w, M, N, K) != apart
    res, want_res = r.clone(), r.clone()
    want = ops.rms_norm(ops.linear(x, w), g, 1e-5, residual=want_res)
    y = ops.linear_add_rmsnorm(x, w, res, g, 1e-5)
    if apart:
        assert torch.equal(res, want_res) and torch.equal(y, want)
    # the product, its sum with the residual and the result may each be a bf16 step apart
    assert ((res.float() - want_res.float()).abs() <= 2.0 ** -7 * ((want_res - r).float().abs() + want_res.float().abs()) + 1e-4).all()
    assert (y.float() - want.float()).norm() <= 2.0 ** -7 * want.float().norm()


@pytest.mark.parametrize("N,K", [(2048, 2048), (1024, 1024), (2048, 1000), (2056, 2048)])
def test_residual_of_another_shape(cuda, N, K):
    """A stream [3, 100, N] beside rows [300, K]: the result has the rows' shape whatever kernels take the product (parts and norm; the
    product, then the norm; operands off the tile grid), the bits of the product and a norm that adds the residual where that ran."""
    torch.manual_seed(N + K)
    x, w = torch.randn(300, K, device=cuda).bfloat16(), (torch.randn(N, K, device=cuda) * K ** -0.5).bfloat16()
    g, r = torch.randn(N, device=cuda).bfloat16(), torch.randn(3, 100, N, device=cuda).bfloat16()
    res, want_res = r.clone(), r.clone()
    want = ops.rms_norm(ops.linear(x, w), g, 1e-5, residual=want_res)
    y = ops.linear_add_rmsnorm(x, w, res, g, 1e-5)
    assert y.shape == want.shape == (300, N) and res.shape == r.shape
    if ops.native().gemm_slabs_parts(300, N, K, False):  # sums in another order: a bf16 step of the product, and of the result
        assert ((res.float() - want_res.float()).abs() <= 2.0 ** -7 * ((want_res - r).float().abs() + want_res.float().abs()) + 1e-4).all()
        assert ((y.float() - want.float()).norm() <= 2.0 ** -7 * want.float().norm())
    else:
        assert torch.equal(res, want_res) and torch.equal(y, want)


@pytest.mark.parametrize("M", [1, 17, 64])
@pytest.mark.parametrize("N,K,slices", [(1024, 1024, False), (2048, 1024, False), (1536, 1536, False), (16, 1536, False), (2320, 1024, True), (1552, 1536, True),
                                        (1024, 2048, True), (1024, 1152, True)])
def test_small_products_before_a_norm(cuda, M, N, K, slices):
    """Both sides of the line below which the product is one launch and the norm another: there, the bits of those two."""
    torch.manual_seed(M + N)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    x, w, r, g = bf(M, K), bf(N, K) * K ** -0.5, bf(M, N), bf(N)
    assert ops.native().gemm_splitk_fusable_norm(M, N, K) == slices
    res, want_res = r.clone(), r.clone()
    want = ops.rms_norm(ops.linear(x, w), g, 1e-5, residual=want_res)
    y = ops.linear_add_rmsnorm(x, w, res, g, 1e-5)
    if not slices:
        assert torch.equal(res, want_res) and torch.equal(y, want)
    # sums in another order: the product, its sum with the residual and the result each a bf16 step apart
    assert ((res.float() - want_res.float()).abs() <= 2.0 ** -7 * ((want_res - r).float().abs() + want_res.float().abs()) + 1e-4).all()
    assert (y.float() - want.float()).norm() <= 2.0 ** -7 * want.float().norm()


@pytest.mark.parametrize("M,N,K,ks", [(1, 1024, 5632, 2), (9, 1024, 7168, 3), (32, 512, 17408, 6), (17, 256, 8704, 3), (16, 1280, 8192, 3), (5, 144, 18944, 7)])
def test_deep_products_in_uneven_slices(cuda, M, N, K, ks):
    """Up to 32 rows of a deep product in slices that differ by 512, the first ones longer, under every epilogue that adds them and before a
    rms norm, against float64: a bf16 rounding of each result (2^-8 of it; the activations as elsewhere by approximate functions, 2^-10 more)
    and fp32 sums of K products of unit normals and weights of K^-1/2."""
    torch.manual_seed(M + K)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    x, w, b, r, g = bf(M, K), bf(N, K) * K ** -0.5, bf(N), bf(M, N), bf(N)
    assert ops.native().gemm_partials_ks(M, N, K) == ks and (K // 512) % ks  # unequal
    wf = w.clone()
    assert ops.to_fragment_layout_(wf)
    p = x.double() @ w.double().t()
    gelu = torch.nn.functional.gelu
    cases = [(dict(out_dtype=torch.float32), p, 0), (dict(), p, 2.0 ** -8), (dict(bias=b), p + b.double(), 2.0 ** -8),
             (dict(bias=b, act="gelu"), gelu(p + b.double()), 2.0 ** -8 + 2.0 ** -10), (dict(bias=b, act="relu"), (p + b.double()).relu(), 2.0 ** -8)]
    if N % 32 == 0:
        gu = p.view(M, N // 32, 2, 16)
        cases.append((dict(act="swiglu"), (torch.nn.functional.silu(gu[:, :, 0]) * gu[:, :, 1]).reshape(M, -1), 2.0 ** -8 + 2.0 ** -10))
    sums = 2.0 ** -18 * K ** 0.5
    for kw, want, rel in cases:
        y = ops.linear(x, w, **kw)
        assert ((y.double() - want).abs() <= rel * want.abs() + sums).all()
        assert torch.equal(y, ops.linear(x, wf, **kw))
    # the product is rounded before the residual is added
    v, off = p + r.double(), 2.0 ** -8 * 1.01 * (p.abs() + (p + r.double()).abs()) + sums
    assert ((ops.linear(x, w, residual=r).double() - v).abs() <= off).all()
    inv = torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-5)
    want = v * inv * g.double()
    for wt in (w, wf):
        res = r.clone()
        y = ops.linear_add_rmsnorm(x, wt, res, g, 1e-5)
        assert ((res.double() - v).abs() <= off).all()
        assert ((y.double() - want).abs() <= 1.01 * off * inv * g.double().abs() + (2.0 ** -8 + 2.0 ** -8) * want.abs()).all()


@pytest.mark.parametrize("M,N,K", [(16, 1024, 5632), (9, 1024, 7168), (24, 1024, 1024), (24, 6144, 4096), (3, 18432, 2048), (24, 4096, 14336), (40, 1024, 5632)])
@pytest.mark.parametrize("off", [1, 4])
@pytest.mark.parametrize("frag", [False, True])
def test_rows_off_16_bytes(cuda, M, N, K, off, frag):
    """Decode products of rows 2 or 8 bytes past a multiple of 16, by every kernel of them: the bits of the same rows on 16 bytes."""
    torch.manual_seed(M + K)
    x, w = torch.randn(M, K, device=cuda).bfloat16(), (torch.randn(N, K, device=cuda) * K ** -0.5).bfloat16()
    odd = torch.empty(M * K + off, device=cuda, dtype=torch.bfloat16)[off:].view(M, K).copy_(x)
    assert odd.data_ptr() & 15 and odd.is_contiguous() and (not frag or ops.to_fragment_layout_(w))
    assert torch.equal(ops.linear(odd, w), ops.linear(x, w))
    if N <= 8192:
        g, r = torch.randn(N, device=cuda).bfloat16(), torch.randn(M, N, device=cuda).bfloat16()
        a, b = r.clone(), r.clone()
        assert torch.equal(ops.linear_add_rmsnorm(odd, w, a, g, 1e-5), ops.linear_add_rmsnorm(x, w, b, g, 1e-5)) and torch.equal(a, b)


@pytest.mark.parametrize("M,N", [(70, 1024), (300, 2048), (1500, 1024)])
def test_rows_that_are_the_stream(cuda, M, N):
    """The stream itself as the product's rows: no product writes over rows that it still reads."""
    torch.manual_seed(M)
    w, g = (torch.randn(N, N, device=cuda) * N ** -0.5).bfloat16(), torch.randn(N, device=cuda).bfloat16()
    r = torch.randn(M, N, device=cuda).bfloat16()
    apart, res = r.clone(), r.clone()
    want = ops.linear_add_rmsnorm(r, w, apart, g, 1e-5)
    y = ops.linear_add_rmsnorm(res, w, res, g, 1e-5)
    assert torch.equal(res, apart) and torch.equal(y, want)


@pytest.mark.parametrize("layer", [False, True])
def test_longer_bias_before_a_norm(cuda, layer):
    """A bias padded past the product's columns: the first N are taken, as by the product alone."""
    torch.manual_seed(2)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    x, w, b, r, g = bf(200, 2048), bf(2048, 2048) / 45, bf(2064), bf(200, 2048), bf(2048)
    assert ops.native().gemm_slabs_parts(200, 2048, 2048, layer) > 1
    if layer:
        assert torch.equal(ops.linear_layer_norm(x, w, b, r, g, g, 1e-5), ops.layer_norm(ops.linear(x, w, b, residual=r), g, g, 1e-5))
    else:
        res, want_res = r.clone(), r.clone()
        want = ops.rms_norm(ops.linear(x, w, b), g, 1e-5, residual=want_res)
        assert torch.equal(ops.linear_add_rmsnorm(x, w, res, g, 1e-5, bias=b), want) and torch.equal(res, want_res)


@pytest.mark.parametrize("name,value", [("_SPLITK", False), ("_GEMM_FORCE", 2)])
def test_linear_layer_norm_under_the_gemm_switches(cuda, monkeypatch, name, value):
    """A forced GEMM kernel, or the decode GEMMs switched off, hold for the product before a layer norm too."""
    torch.manual_seed(0)
    x, r = torch.randn(20, 1024, device=cuda).bfloat16(), torch.randn(20, 1024, device=cuda).bfloat16()
    w = (torch.randn(1024, 1024, device=cuda) / 32).bfloat16()
    g, b = torch.randn(1024, device=cuda).bfloat16(), torch.randn(1024, device=cuda).bfloat16()
    monkeypatch.setattr(ops, name, value)
    want = ops.layer_norm(ops.linear(x, w, bias=b, residual=r), g, b, 1e-5)
    monkeypatch.setattr(ops.native(), "linear_layernorm", None)
    assert torch.equal(ops.linear_layer_norm(x, w, b, r, g, b, 1e-5), want)


@pytest.mark.parametrize("M", [20, 70])
def test_linear_layer_norm_has_the_rows_shape(cuda, M):
    """The result has the shape of the product's rows, whatever that of the residual's, on either side of the K slices' reach."""
    torch.manual_seed(1)
    x, r = torch.randn(2, M // 2, 1024, device=cuda).bfloat16(), torch.randn(M, 1024, device=cuda).bfloat16()
    w, g = (torch.randn(1024, 1024, device=cuda) / 32).bfloat16(), torch.randn(1024, device=cuda).bfloat16()
    assert ops.linear_layer_norm(x, w, None, r, g, None, 1e-5).shape == (2, M // 2, 1024)
