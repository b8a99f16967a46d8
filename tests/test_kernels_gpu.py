"""Numerics of every gfx950 HIP kernel against the plain-PyTorch fp32 reference of the same op."""
import math
import os

import pytest
import torch

from generativeaiexamples_amd import ops
from generativeaiexamples_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


def _close(a, b, atol, rtol=0.0, what=""):
    a, b = a.float().cpu(), b.float().cpu()
    err = (a - b).abs()
    tol = atol + rtol * b.abs()
    bad = err > tol
    assert not bad.any(), f"{what}: max err {err.max().item():.4g}, {bad.sum().item()} / {bad.numel()} bad"


@pytest.mark.parametrize("D", [768, 1024, 1280, 4096])
@pytest.mark.parametrize("resid", [False, True])
def test_rmsnorm(cuda, D, resid):
    torch.manual_seed(0)
    x = torch.randn(37, D, device=cuda, dtype=torch.bfloat16)
    w = torch.randn(D, device=cuda, dtype=torch.bfloat16)
    r = torch.randn(37, D, device=cuda, dtype=torch.bfloat16) if resid else None
    r_ref = r.clone().cpu() if resid else None
    y = ops.rms_norm(x, w, 1e-5, r)
    y_ref = ref.rms_norm(x.cpu(), w.cpu(), 1e-5, r_ref)
    _close(y, y_ref, 2e-2, 2e-2, "rmsnorm")
    if resid:
        _close(r, r_ref, 0, 0, "residual")


@pytest.mark.parametrize("D", [768, 1024, 1280])
@pytest.mark.parametrize("resid", [False, True])
def test_layernorm(cuda, D, resid):
    torch.manual_seed(1)
    x = torch.randn(29, D, device=cuda, dtype=torch.bfloat16)
    w = torch.randn(D, device=cuda, dtype=torch.bfloat16)
    b = torch.randn(D, device=cuda, dtype=torch.bfloat16)
    r = torch.randn(29, D, device=cuda, dtype=torch.bfloat16) if resid else None
    r_ref = r.clone().cpu() if resid else None
    y = ops.layer_norm(x, w, b, 1e-12, r)
    y_ref = ref.layer_norm(x.cpu(), w.cpu(), b.cpu(), 1e-12, r_ref)
    _close(y, y_ref, 3e-2, 2e-2, "layernorm")


GEMM_SHAPES = [(1, 256, 256), (7, 384, 512), (64, 1024, 1024), (128, 512, 768), (129, 384, 256),
               (200, 1024, 512), (513, 640, 1024), (1024, 1536, 4096)]


@pytest.mark.parametrize("M,N,K", GEMM_SHAPES)
@pytest.mark.parametrize("act", [None, "bias", "gelu", "relu", "residual", "swiglu"])
def test_gemm(cuda, M, N, K, act):
    torch.manual_seed(M * 7 + N)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    bias = torch.randn(N, device=cuda, dtype=torch.bfloat16) if act in ("bias", "gelu", "relu") else None
    res = torch.randn(M, N, device=cuda, dtype=torch.bfloat16) if act == "residual" else None
    a = act if act in ("gelu", "relu", "swiglu") else None
    y = ops.linear(x, w, bias=bias, residual=res, act=a)
    y_ref = ref.linear(x.cpu(), w.cpu(), None if bias is None else bias.cpu(), None if res is None else res.cpu(), a)
    _close(y, y_ref, 3e-2, 2e-2, f"gemm {M}x{N}x{K} {act}")


@pytest.mark.parametrize("M", [3, 64, 300])
def test_gemm_fp32_out(cuda, M):
    torch.manual_seed(3)
    x = torch.randn(M, 512, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(1000, 512, device=cuda) / 20).to(torch.bfloat16)
    y = ops.linear(x, w, out_dtype=torch.float32)
    assert y.dtype == torch.float32
    _close(y, x.float().cpu() @ w.float().cpu().t(), 2e-3, 2e-3, "gemm fp32 out")


def _make_cache(nb, Hkv, D, device):
    k = torch.zeros(nb, Hkv, 16, D, device=device, dtype=torch.bfloat16)
    v = torch.zeros(nb, Hkv, D, 16, device=device, dtype=torch.bfloat16)
    return k, v


@pytest.mark.parametrize("D", [64, 96, 128])
def test_rope_kv_write(cuda, D):
    torch.manual_seed(4)
    Hq, Hkv, T = 8, 2, 45
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, device=cuda, dtype=torch.bfloat16)
    pos = torch.randint(0, 1000, (T,), device=cuda, dtype=torch.int32)
    cs = ops.rope_cos_sin(2048, D, 500000.0, device=cuda)
    slots = torch.randperm(10 * 16, device=cuda)[:T].int()
    slots[3] = -1
    kc, vc = _make_cache(10, Hkv, D, cuda)
    q = torch.empty(T, Hq, D, device=cuda, dtype=torch.bfloat16)
    ops.rope_kv_write(qkv, pos, cs, slots, q, kc, vc, Hq, Hkv, D)
    kr, vr = _make_cache(10, Hkv, D, "cpu")
    qr = torch.empty(T, Hq, D, dtype=torch.bfloat16)
    ref.rope_kv_write(qkv.cpu(), pos.cpu(), cs.cpu(), slots.cpu(), qr, kr, vr, Hq, Hkv, D)
    _close(q, qr, 2e-2, 1e-2, "q")
    _close(kc, kr, 2e-2, 1e-2, "k cache")
    _close(vc, vr, 0, 0, "v cache")


def _paged_setup(seq_lens, Hkv, D, device, seed=0):
    g = torch.Generator().manual_seed(seed)
    nb_total = sum((n + 15) // 16 for n in seq_lens) + 3
    kc = torch.randn(nb_total, Hkv, 16, D, generator=g).to(torch.bfloat16)
    vc = torch.randn(nb_total, Hkv, D, 16, generator=g).to(torch.bfloat16)
    perm = torch.randperm(nb_total, generator=g)
    maxb = max((n + 15) // 16 for n in seq_lens)
    bt = torch.zeros(len(seq_lens), maxb, dtype=torch.int32)
    i = 0
    for b, n in enumerate(seq_lens):
        nb = (n + 15) // 16
        bt[b, :nb] = perm[i:i + nb]
        i += nb
    return kc.to(device), vc.to(device), bt.to(device)


@pytest.mark.parametrize("D,Hq,Hkv", [(128, 8, 2), (128, 32, 8), (64, 4, 4), (128, 8, 1), (64, 16, 8), (96, 16, 16),
                                      (96, 8, 2)])
@pytest.mark.parametrize("causal", [True, False])
def test_attention_prefill(cuda, D, Hq, Hkv, causal):
    torch.manual_seed(5)
    ctx = [1, 77, 130, 300]
    qlen = [1, 77, 33, 300] if causal else ctx  # chunked prefill: q is a suffix of ctx
    kc, vc, bt = _paged_setup(ctx, Hkv, D, cuda)
    cu = torch.tensor([0] + list(torch.tensor(qlen).cumsum(0)), dtype=torch.int32)
    q = torch.randn(int(cu[-1]), Hq, D, device=cuda, dtype=torch.bfloat16)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    o = ops.attention_prefill(q, kc, vc, bt, cu.to(cuda), ctx_t.to(cuda), scale, causal, q_lens=qlen)
    o_ref = ref.attention_prefill(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), cu, ctx_t, scale, causal)
    _close(o, o_ref, 2e-2, 2e-2, "prefill")


@pytest.mark.parametrize("D,Hq,Hkv", [(128, 32, 8), (64, 16, 2), (128, 16, 1)])
def test_attention_prefill_half_tiles(cuda, D, Hq, Hkv):
    """Few tiles go to the 4-wave kernel in halves of 32 rows, many whole to the 8-wave one: sequences of one short half, one
    row into the second, whole tiles, chunks over a prefix. A row's sums are the same in both, so the bits are."""
    torch.manual_seed(19)
    ctx = [1, 32, 33, 64, 65, 200, 131]
    qlen = [1, 32, 33, 64, 65, 17, 64]
    times = 3 * 256 // (2 * Hkv * (Hq // Hkv // 4)) // len(ctx) + 1  # sequences enough for whole tiles
    kc, vc, bt = _paged_setup(ctx, Hkv, D, cuda, seed=7)
    q = torch.randn(sum(qlen), Hq, D, device=cuda, dtype=torch.bfloat16)
    out = []
    for n in (1, times):
        cu = torch.tensor([0] + list(torch.tensor(qlen * n).cumsum(0)), dtype=torch.int32)
        out.append(ops.attention_prefill(q.repeat(n, 1, 1), kc, vc, bt.repeat(n, 1), cu.to(cuda), torch.tensor(ctx * n, dtype=torch.int32, device=cuda),
                                         D ** -0.5, True, q_lens=qlen * n))
    assert torch.equal(out[0], out[1][:len(q)]) and torch.equal(out[0], out[1][-len(q):])
    cu = torch.tensor([0] + list(torch.tensor(qlen).cumsum(0)), dtype=torch.int32)
    want = ref.attention_prefill(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), cu, torch.tensor(ctx, dtype=torch.int32), D ** -0.5, True)
    _close(out[0], want, 2e-2, 2e-2, "half tiles")


@pytest.mark.parametrize("lens", [[1, 64, 65, 63], [128, 129, 200], [512, 17]])
def test_attention_rows_many(cuda, lens):
    """Past three workgroups a CU the form in fewer registers: the bits of the other one, whose rows fp32 attention bounds (P and
    the result are rounded to bf16: 2^-8 of the largest value, as the other attention tests). The last sequence ends the buffer."""
    torch.manual_seed(23)
    H, out = 16, []
    qkv = torch.randn(sum(lens), 3 * H * 64, device=cuda, dtype=torch.bfloat16)
    for n in (1, 3 * 256 // (H * len(lens)) + 2):
        cu = torch.tensor([0] + list(torch.tensor(lens * n).cumsum(0)), dtype=torch.int32, device=cuda)
        o = torch.empty(sum(lens) * n, H, 64, device=cuda, dtype=torch.bfloat16)
        ops.native().attn_rows(qkv.repeat(n, 1), ops.build_prefill_tiles(lens * n, H, H, cuda, head_dim=64), cu,
                               torch.tensor(lens * n, dtype=torch.int32, device=cuda), o, H, 0.125, False)
        out.append(o)
    assert torch.equal(out[0], out[1][:len(qkv)]) and torch.equal(out[0], out[1][-len(qkv):])
    q, k, v = qkv.float().cpu().view(-1, 3, H, 64).unbind(1)
    want = torch.cat([torch.nn.functional.scaled_dot_product_attention(*(x[a:a + n].transpose(0, 1) for x in (q, k, v)), scale=0.125).transpose(0, 1)
                      for a, n in zip([0] + list(torch.tensor(lens).cumsum(0)), lens)])
    _close(out[0], want, 2e-2, 2e-2, "rows")


@pytest.mark.parametrize("D", [256, 4096, 8192])
def test_norm_one_wave_rows(cuda, D):
    """A wave a workgroup up to 512 rows, four beyond: the same row, the same bits."""
    torch.manual_seed(20)
    x, w, b = torch.randn(513, D, device=cuda).bfloat16(), torch.randn(D, device=cuda).bfloat16(), torch.randn(D, device=cuda).bfloat16()
    four, one = ops.layer_norm(x, w, b, 1e-5), torch.cat([ops.layer_norm(x[:512].clone(), w, b, 1e-5), ops.layer_norm(x[512:].clone(), w, b, 1e-5)])
    assert torch.equal(four, one)
    assert torch.equal(ops.rms_norm(x, w, 1e-5)[:512], ops.rms_norm(x[:512].clone(), w, 1e-5))


@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (16, 16)])
def test_attention_prefill_running_max_jumps(cuda, Hq, Hkv):
    """Score scales that jump by far more than the deferred-max threshold between key tiles (keys 64-255 scaled x8,
    keys from 448 on x24, so the running max moves by ~2^10 and more mid-row), and a chunked prefill over that prefix:
    the kernel's deferred running max (rescale only past 2^8) still matches the fp32 reference, with the 8-wave GQA
    workgroups and the 4-wave MHA ones."""
    torch.manual_seed(17)
    D = 128
    ctx = [700, 333]
    qlen = [700, 100]
    kc, vc, bt = _paged_setup(ctx, Hkv, D, cuda, seed=5)
    kcf = kc.float()
    for s, n in enumerate(ctx):
        for pos in range(n):
            f = 8.0 if 64 <= pos < 256 else 24.0 if pos >= 448 else 1.0
            b, o = int(bt[s, pos // 16]), pos % 16
            kcf[b, :, o] *= f
    kc = kcf.to(torch.bfloat16)
    cu = torch.tensor([0] + list(torch.tensor(qlen).cumsum(0)), dtype=torch.int32)
    q = torch.randn(int(cu[-1]), Hq, D, device=cuda, dtype=torch.bfloat16)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    for causal in (True, False):
        ql = qlen if causal else ctx
        cu_c = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32)
        qq = q if causal else torch.randn(int(cu_c[-1]), Hq, D, device=cuda, dtype=torch.bfloat16)
        o = ops.attention_prefill(qq, kc, vc, bt, cu_c.to(cuda), ctx_t.to(cuda), scale, causal, q_lens=ql)
        o_ref = ref.attention_prefill(qq.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), cu_c, ctx_t, scale, causal)
        _close(o, o_ref, 3e-2, 3e-2, f"prefill with running-max jumps, causal={causal}")


@pytest.mark.parametrize("L,D,Hq,Hkv", [(2048, 128, 32, 8), (4096, 128, 32, 8), (8192, 128, 32, 8),
                                         (2048, 256, 16, 8), (4096, 256, 8, 4), (8192, 256, 8, 1)])
def test_attention_prefill_long(cuda, L, D, Hq, Hkv):
    """Long-context causal GQA prefill (one 2K-8K sequence plus a short one, D 128 / 256) against an
    fp32 dense reference computed per head on the GPU (the CPU reference would need GBs of scores)."""
    torch.manual_seed(L + D)
    ctx = [L, 300]
    kc, vc, bt = _paged_setup(ctx, Hkv, D, cuda, seed=L)
    cu = torch.tensor([0, L, L + 300], dtype=torch.int32, device=cuda)
    q = torch.randn(L + 300, Hq, D, device=cuda, dtype=torch.bfloat16)
    scale = 1 / math.sqrt(D)
    o = ops.attention_prefill(q, kc, vc, bt, cu, torch.tensor(ctx, dtype=torch.int32, device=cuda), scale, True,
                              q_lens=ctx)
    for s, n in enumerate(ctx):
        blocks = bt[s, :(n + 15) // 16].long()
        k = kc[blocks].permute(1, 0, 2, 3).reshape(Hkv, -1, D)[:, :n].float()  # [Hkv, n, D]
        v = vc[blocks].permute(1, 0, 3, 2).reshape(Hkv, -1, D)[:, :n].float()
        qs = q[int(cu[s]):int(cu[s]) + n].float()
        mask = torch.ones(n, n, device=cuda, dtype=torch.bool).tril()
        for h in range(Hq):
            kv = h // (Hq // Hkv)
            sc = (qs[:, h] @ k[kv].t()) * scale
            ref_o = sc.masked_fill(~mask, float("-inf")).softmax(-1) @ v[kv]
            _close(o[int(cu[s]):int(cu[s]) + n, h], ref_o, 2e-2, 2e-2, f"prefill L={n} h={h}")


@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (8, 1), (64, 8)])
@pytest.mark.parametrize("causal", [True, False])
def test_attention_prefill_two_heads_per_wave(cuda, Hq, Hkv, causal):
    """The head_dim-128 prefill kernel with two q heads per wave (64 query rows per tile, Q fragments staged in LDS)
    against the fp32 reference and against the one-head kernel: varlen, chunked prefill over a cached prefix, and a
    long sequence (multi-tile walks, diagonal and interior key tiles)."""
    torch.manual_seed(11)
    D = 128
    ctx = [1, 77, 130, 300, 1500]
    qlen = [1, 77, 33, 300, 1500] if causal else ctx
    kc, vc, bt = _paged_setup(ctx, Hkv, D, cuda, seed=3)
    cu = torch.tensor([0] + list(torch.tensor(qlen).cumsum(0)), dtype=torch.int32)
    q = torch.randn(int(cu[-1]), Hq, D, device=cuda, dtype=torch.bfloat16)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    outs = []
    try:
        for hl in (2, 1):
            ops.set_prefill_heads_per_wave(hl)
            # one head per wave: 8-wave workgroups (2 row groups) at >= 4 q heads per kv head
            waves = 8 if hl == 1 and Hq // Hkv >= 4 and os.environ.get("GAI_ATTN_WAVES", "8") == "8" else 4
            assert ops.prefill_rows_per_tile(Hq, Hkv, D) == (64 if hl == 2 else 32 * waves // min(4, Hq // Hkv))
            outs.append(ops.attention_prefill(q, kc, vc, bt, cu.to(cuda), ctx_t.to(cuda), scale, causal, q_lens=qlen))
    finally:
        ops.set_prefill_heads_per_wave(1)
    o_ref = ref.attention_prefill(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), cu, ctx_t, scale, causal)
    _close(outs[0], o_ref, 2e-2, 2e-2, "prefill, two heads per wave")
    # same math per head (the k-step loop order of QK^T differs: fp32 sums in another order)
    assert (outs[0].float() - outs[1].float()).abs().max().item() < 2e-2


@pytest.mark.parametrize("D,Hq,Hkv", [(128, 32, 8), (128, 64, 8), (64, 8, 8), (128, 4, 4)])
def test_attention_decode(cuda, D, Hq, Hkv):
    torch.manual_seed(6)
    ctx = [1, 16, 17, 100, 513, 2000, 4097]
    kc, vc, bt = _paged_setup(ctx, Hkv, D, cuda, seed=1)
    q = torch.randn(len(ctx), Hq, D, device=cuda, dtype=torch.bfloat16)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    for split in (128, 512, None):
        ws = ops.DecodeWorkspace(len(ctx), Hq, D, max(ctx), cuda, split_keys=split)
        o = ops.attention_decode(q, kc, vc, bt, ctx_t.to(cuda), scale, ws=ws)
        o_ref = ref.attention_decode(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), ctx_t, scale)
        _close(o, o_ref, 2e-2, 2e-2, f"decode split={ws.split_keys}")


@pytest.mark.parametrize("nsplit", [1, 2, 3, 7])
def test_attention_decode_adaptive_splits(cuda, nsplit):
    """split_keys = 0: every sequence's actual context is cut into nsplit equal 128-key-aligned parts inside the
    kernel (graphs captured for max_model_len stay balanced at every replay); fused in-launch merge == separate
    reduce launch == the fp32 reference, on ragged contexts from 1 key to far past one split."""
    torch.manual_seed(8)
    D, Hq, Hkv = 128, 32, 8
    ctx = [1, 100, 129, 700, 2535, 2663, 4097, 300]
    kc, vc, bt = _paged_setup(ctx, Hkv, D, cuda, seed=3)
    q = torch.randn(len(ctx), Hq, D, device=cuda, dtype=torch.bfloat16)
    scale = 1 / math.sqrt(D)
    ws = ops.DecodeWorkspace(len(ctx), Hq, D, 8192, cuda)
    nat = ops.native()
    c = torch.tensor(ctx, dtype=torch.int32, device=cuda)
    o_f, o_u = torch.empty_like(q), torch.empty_like(q)
    nat.attn_decode(q, kc, vc, bt, c, o_f, ws.o, ws.ml, scale, 0, nsplit, 1.0, 1.0, ws.cnt)
    nat.attn_decode(q, kc, vc, bt, c, o_u, ws.o, ws.ml, scale, 0, nsplit, 1.0, 1.0, None)
    assert int(ws.cnt.abs().sum()) == 0
    o_ref = ref.attention_decode(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), c.cpu(), scale)
    _close(o_f, o_ref, 2e-2, 2e-2, "adaptive fused")
    _close(o_u, o_ref, 2e-2, 2e-2, "adaptive reduce")


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("Hq,Hkv,nsplit,ctx", [
    (32, 8, 2, [1]), (4, 4, 3, [257, 0, 128]), (16, 1, 2, [1, 127, 128, 129, 0, 0, 2049]),
    (32, 8, 7, [2663, 31, 4097, 640, 1, 300, 2048, 255, 33, 96, 97, 1500]),
    (64, 8, 33, [4200, 4096, 700, 700, 129]),             # a part per unit
    (16, 4, 4, [(37 * i * i) % 701 for i in range(131)]),  # more parts than workgroups; equal lengths, empty sequences
    (8, 8, 9, [8000, 1] * 100), (32, 8, 2, [0, 0, 0]),
    (32, 8, 8, [2663 - 97 * i for i in range(24)]), (8, 4, 4, [513] * 63 + [0]), (8, 4, 4, [513] * 64 + [0]),  # ranked, one wave's worth or more
    (8, 4, 2, [(91 * i) % 300 for i in range(256)]), (8, 4, 3, [0] * 60 + [300] * 4), (4, 4, 3, [60] * 70)])  # all resident
def test_attention_decode_queue(cuda, Hq, Hkv, nsplit, ctx, fp8):
    """Parts handed out by the launch: the bits of the launch with a workgroup per part, whatever their number and order; rows of
    sequences without keys are left alone; tickets and counters back at zero; graph replays the same."""
    torch.manual_seed(len(ctx))
    D, B = 128, len(ctx)
    kc, vc, bt = _paged_setup([max(1, n) for n in ctx], Hkv, D, cuda, seed=4)
    if fp8:
        kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    q = torch.randn(B, Hq, D, device=cuda, dtype=torch.bfloat16)
    c, scale = torch.tensor(ctx, dtype=torch.int32, device=cuda), 1 / math.sqrt(D)
    ws = ops.DecodeWorkspace(B, Hq, D, max(bt.shape[1] * 16, 128 * nsplit), cuda)
    sk, sv = (0.5, 2.0) if fp8 else (1.0, 1.0)

    def run(out, queue):
        ops.native().attn_decode(q, kc, vc, bt, c, out, ws.o, ws.ml, scale, 0, nsplit, sk, sv, ws.cnt, queue=queue)

    want, out = torch.full_like(q, 7.0), torch.full_like(q, 7.0)
    run(want, False)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        run(out, True)
    for i in range(6):
        out.fill_(7.0)
        run(out, True) if i % 2 else g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and int(ws.cnt.abs().sum()) == 0
    live = c.cpu() > 0
    assert (out.cpu()[~live] == 7.0).all()
    if live.any() and B < 100:
        k, v = (kc.float() * sk, vc.float() * sv) if fp8 else (kc, vc)
        o_ref = ref.attention_decode(q.cpu()[live], k.cpu(), v.cpu(), bt.cpu()[live], c.cpu()[live], scale)
        _close(out.cpu()[live], o_ref, 2e-2, 2e-2, "queue")     # test_attention_decode's bound: probabilities and result in bf16
    with pytest.raises(RuntimeError):
        ops.native().attn_decode(q, kc, vc, bt, c, out, ws.o, ws.ml, scale, 0, nsplit, sk, sv, ws.cnt[: B * Hkv], queue=True)


def test_decode_workspace_holds_the_queues(cuda, monkeypatch):
    """A workspace has room for whatever the launch asks for its queues, also behind a ticket for every sequence and q head."""
    nat = ops.native()

    class Larger:
        DECODE_QUEUE_INTS = nat.DECODE_QUEUE_INTS + 64

        def __getattr__(self, name):
            return getattr(nat, name)

    monkeypatch.setattr(ops, "native", Larger)
    B, H, D = 70, 8, 128
    kc, vc, bt = _paged_setup([600] * B, H, D, cuda, seed=1)
    ws, took = ops.DecodeWorkspace(B, H, D, 1024, cuda), []
    attn = nat.attn_decode
    monkeypatch.setattr(Larger, "attn_decode", lambda self, *a: took.append(a[-1]) or attn(*a), raising=False)
    q = torch.randn(B, H, D, device=cuda, dtype=torch.bfloat16)
    ops.attention_decode(q, kc, vc, bt, torch.full((B,), 600, dtype=torch.int32, device=cuda), 0.1, ws=ws, max_ctx=1024)
    assert took == [True] and ops.DecodeWorkspace(B, H, D, 1024, "cpu").cnt.numel() == B * H


def test_attention_decode_fused_merge_reuse(cuda):
    """In-launch split merge (ticket counters, last split combines): equal to the separate reduce launch, and
    the counters reset themselves - many back-to-back launches and graph replays on one workspace, with the
    number of splits changing between calls, stay exact."""
    torch.manual_seed(7)
    D, Hq, Hkv = 128, 32, 8
    ctx = [5, 130, 700, 1500, 2600, 33, 4000, 257]
    kc, vc, bt = _paged_setup(ctx, Hkv, D, cuda, seed=2)
    q = torch.randn(len(ctx), Hq, D, device=cuda, dtype=torch.bfloat16)
    scale = 1 / math.sqrt(D)
    ws = ops.DecodeWorkspace(len(ctx), Hq, D, max(ctx), cuda, split_keys=128)
    nat = ops.native()
    for trial in range(6):
        c = torch.tensor([max(1, x - 97 * trial) for x in ctx], dtype=torch.int32, device=cuda)
        o_f = torch.empty_like(q)
        o_u = torch.empty_like(q)
        nsplit = (int(c.max()) + 127) // 128
        nat.attn_decode(q, kc, vc, bt, c, o_f, ws.o, ws.ml, scale, 128, nsplit, 1.0, 1.0, ws.cnt)
        nat.attn_decode(q, kc, vc, bt, c, o_u, ws.o, ws.ml, scale, 128, nsplit, 1.0, 1.0, None)
        assert torch.equal(o_f, o_u), f"trial {trial}"
        assert int(ws.cnt.abs().sum()) == 0
    o_ref = ref.attention_decode(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), c.cpu(), scale)
    _close(o_f, o_ref, 2e-2, 2e-2, "fused merge")
    # graph replays
    c = torch.tensor(ctx, dtype=torch.int32, device=cuda)
    out = torch.empty_like(q)
    nsplit = (max(ctx) + 127) // 128
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        nat.attn_decode(q, kc, vc, bt, c, out, ws.o, ws.ml, scale, 128, nsplit, 1.0, 1.0, ws.cnt)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        nat.attn_decode(q, kc, vc, bt, c, out, ws.o, ws.ml, scale, 128, nsplit, 1.0, 1.0, ws.cnt)
    want = torch.empty_like(q)
    nat.attn_decode(q, kc, vc, bt, c, want, ws.o, ws.ml, scale, 128, nsplit, 1.0, 1.0, None)
    for _ in range(20):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    assert int(ws.cnt.abs().sum()) == 0


F8 = torch.float8_e4m3fn


@pytest.mark.parametrize("D", [64, 96, 128, 256])
def test_rope_kv_write_fp8(cuda, D):
    torch.manual_seed(14)
    Hq, Hkv, T = 8, 2, 45
    qkv = (torch.randn(T, (Hq + 2 * Hkv) * D, device=cuda) * 4).to(torch.bfloat16)
    pos = torch.randint(0, 1000, (T,), device=cuda, dtype=torch.int32)
    cs = ops.rope_cos_sin(2048, D, 500000.0, device=cuda)
    slots = torch.randperm(10 * 16, device=cuda)[:T].int()
    kc = torch.zeros(10, Hkv, 16, D, device=cuda, dtype=F8)
    vc = torch.zeros(10, Hkv, D, 16, device=cuda, dtype=F8)
    q = torch.empty(T, Hq, D, device=cuda, dtype=torch.bfloat16)
    ops.rope_kv_write(qkv, pos, cs, slots, q, kc, vc, Hq, Hkv, D, True, 0.5, 2.0)
    kr = torch.zeros(10, Hkv, 16, D, dtype=F8)
    vr = torch.zeros(10, Hkv, D, 16, dtype=F8)
    qr = torch.empty(T, Hq, D, dtype=torch.bfloat16)
    ref.rope_kv_write(qkv.cpu(), pos.cpu(), cs.cpu(), slots.cpu(), qr, kr, vr, Hq, Hkv, D, True, 0.5, 2.0)
    # same bf16 inputs, both round-to-nearest into e4m3fn: at most one fp8 step apart (rope's fp32 math)
    _close(kc.float(), kr.float(), 1e-3, 0.13, "k cache fp8")
    _close(vc.float(), vr.float(), 0, 0, "v cache fp8")
    assert (kc.float() == kr.float().to(cuda)).float().mean() > 0.97


def _fp8_paged(ctx, Hkv, D, seed):
    kc, vc, bt = _paged_setup(ctx, Hkv, D, "cpu", seed=seed)
    return (kc.float() * 3).to(F8).to("cuda"), (vc.float() * 3).to(F8).to("cuda"), bt.to("cuda")


@pytest.mark.parametrize("D,Hq,Hkv", [(128, 32, 8), (64, 8, 8), (256, 8, 2)])
def test_attention_decode_fp8(cuda, D, Hq, Hkv):
    torch.manual_seed(15)
    ctx = [1, 17, 513, 2000, 4097]
    kc, vc, bt = _fp8_paged(ctx, Hkv, D, 3)
    q = torch.randn(len(ctx), Hq, D, device=cuda, dtype=torch.bfloat16)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    for split in (128, None):
        ws = ops.DecodeWorkspace(len(ctx), Hq, D, max(ctx), cuda, split_keys=split)
        o = ops.attention_decode(q, kc, vc, bt, ctx_t.to(cuda), scale, ws=ws, k_scale=0.25, v_scale=0.5)
        o_ref = ref.attention_decode(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), ctx_t, scale, 0.25, 0.5)
        _close(o, o_ref, 2e-2, 2e-2, f"fp8 decode split={ws.split_keys}")


@pytest.mark.parametrize("D,Hq,Hkv", [(128, 32, 8), (64, 16, 8), (256, 8, 4), (96, 16, 16)])
def test_attention_prefill_fp8(cuda, D, Hq, Hkv):
    torch.manual_seed(16)
    ctx, qlen = [77, 300, 1030], [77, 33, 1030]
    kc, vc, bt = _fp8_paged(ctx, Hkv, D, 4)
    cu = torch.tensor([0] + list(torch.tensor(qlen).cumsum(0)), dtype=torch.int32)
    q = torch.randn(int(cu[-1]), Hq, D, device=cuda, dtype=torch.bfloat16)
    ctx_t = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(D)
    o = ops.attention_prefill(q, kc, vc, bt, cu.to(cuda), ctx_t.to(cuda), scale, True, q_lens=qlen, k_scale=0.25,
                              v_scale=0.5)
    o_ref = ref.attention_prefill(q.cpu(), kc.cpu(), vc.cpu(), bt.cpu(), cu, ctx_t, scale, True, k_scale=0.25,
                                  v_scale=0.5)
    _close(o, o_ref, 2e-2, 2e-2, "fp8 prefill")


def test_sample_greedy_and_topk1(cuda):
    torch.manual_seed(7)
    B, V = 9, 128256
    logits = torch.randn(B, V, device=cuda)
    temp = torch.tensor([0.0] * 3 + [0.7] * 6, device=cuda)
    top_p = torch.ones(B, device=cuda)
    top_k = torch.tensor([0, 0, 0, 1, 1, 1, 0, 0, 0], dtype=torch.int32, device=cuda)
    seeds = torch.arange(B, dtype=torch.int64, device=cuda)
    t = ops.sample(logits, temp, top_p, top_k, seeds, 0)
    am = logits.argmax(-1).int()
    assert torch.equal(t[:6], am[:6])


def test_sample_top_p_membership(cuda):
    torch.manual_seed(8)
    B, V = 64, 32000
    logits = torch.randn(B, V, device=cuda) * 3
    temp = torch.full((B,), 0.8, device=cuda)
    top_p = torch.full((B,), 0.5, device=cuda)
    top_k = torch.zeros(B, dtype=torch.int32, device=cuda)
    seeds = torch.arange(B, dtype=torch.int64, device=cuda) + 11
    t = ops.sample(logits, temp, top_p, top_k, seeds, 3).long()
    probs = (logits / 0.8).softmax(-1)
    sp, si = probs.sort(-1, descending=True)
    cum = sp.cumsum(-1)
    for b in range(B):
        n_keep = int(((cum[b] - sp[b]) < 0.5).sum())
        allowed = set(si[b, : n_keep + 1].tolist())  # +1 tolerates threshold ties / fp rounding
        assert int(t[b]) in allowed
    # determinism for a fixed seed/step
    t2 = ops.sample(logits, temp, top_p, top_k, seeds, 3).long()
    assert torch.equal(t, t2)


@pytest.mark.parametrize("scale,T,p", [(1.28, 0.2, 0.7), (3.0, 1.0, 0.9), (0.01, 1.0, 0.9), (1.0, 0.05, 0.95)])
def test_sample_nucleus_exact(cuda, scale, T, p):
    """Every sampled token lies in the exact nucleus (largest logit cut with mass >= p), across the LDS
    fast path (peaked rows) and the full radix fallback (flat rows: > 4096 candidates)."""
    torch.manual_seed(12)
    B, V = 64, 128256
    logits = torch.randn(B, V, device=cuda) * scale
    logits[0, :100] = float("-inf")  # masked tokens (constrained decoding)
    temp = torch.full((B,), T, device=cuda)
    top_p = torch.full((B,), p, device=cuda)
    top_k = torch.zeros(B, dtype=torch.int32, device=cuda)
    seen = set()
    for step in range(4):
        t = ops.sample(logits, temp, top_p, top_k, torch.arange(B, dtype=torch.int64, device=cuda), step).long()
        x = (logits.double() / T)
        probs = x.softmax(-1)
        sp, si = probs.sort(-1, descending=True)
        cum = sp.cumsum(-1)
        n_keep = ((cum - sp) < p * (1 + 1e-5)).sum(-1)
        rank = (si == t[:, None]).float().argmax(-1)
        assert bool((rank <= n_keep).all()), (rank - n_keep).max()
        seen.update(t.tolist())
    assert len(seen) > 1


def test_sample_distribution(cuda):
    """Empirical frequencies of the Gumbel-max sampler match softmax(x/T) on a tiny vocab."""
    V, B = 8, 4096
    base = torch.tensor([2.0, 1.0, 0.5, 0.0, -0.5, -1.0, -2.0, -3.0], device=cuda)
    logits = base.repeat(B, 1).contiguous()
    temp = torch.full((B,), 1.0, device=cuda)
    t = ops.sample(logits, temp, torch.ones(B, device=cuda), torch.zeros(B, dtype=torch.int32, device=cuda),
                   torch.arange(B, dtype=torch.int64, device=cuda), 0).long()
    freq = torch.bincount(t, minlength=V).float() / B
    p = base.softmax(-1)
    assert (freq - p).abs().max().item() < 0.03


def test_penalties(cuda):
    logits = torch.randn(2, 100, device=cuda)
    l_ref = logits.clone().cpu()
    ids = torch.tensor([[1, 5, 0], [7, 0, 0]], dtype=torch.int32, device=cuda)
    cnt = torch.tensor([[2, 1, 0], [3, 0, 0]], dtype=torch.int32, device=cuda)
    n = torch.tensor([2, 1], dtype=torch.int32, device=cuda)
    f = torch.tensor([0.5, 0.1], device=cuda)
    p = torch.tensor([0.2, 0.3], device=cuda)
    r = torch.tensor([1.0, 1.2], device=cuda)
    ops.apply_penalties(logits, ids, cnt, n, f, p, r)
    ref.apply_penalties(l_ref, ids.cpu(), cnt.cpu(), n.cpu(), f.cpu(), p.cpu(), r.cpu())
    _close(logits, l_ref, 1e-5, 0, "penalties")


@pytest.mark.parametrize("nq,N,D,k", [(1, 1000, 1024, 4), (5, 70001, 768, 4), (33, 20000, 1024, 10),
                                      (64, 50000, 1024, 4), (100, 30000, 384, 40), (3, 5, 1024, 4)])
def test_sim_topk(cuda, nq, N, D, k):
    torch.manual_seed(9)
    X = torch.nn.functional.normalize(torch.randn(N, D, device=cuda), dim=-1).to(torch.bfloat16)
    Q = torch.nn.functional.normalize(torch.randn(nq, D, device=cuda), dim=-1).to(torch.bfloat16)
    bias = torch.zeros(N, device=cuda)
    bias[::7] = float("-inf")  # tombstones
    v, i = ops.sim_topk(Q, X, bias, N, k)
    vr, ir = ref.sim_topk(Q.cpu(), X.cpu(), bias.cpu(), N, k)
    _close(v, vr, 1e-3, 1e-3, "topk scores")
    # ids must match where scores are not tied
    s_true = (Q.float() @ X.float().t()).cpu() + bias.cpu()
    picked = torch.gather(s_true, 1, i.cpu())
    _close(picked, vr, 1e-3, 1e-3, "scores of returned ids")
    assert (i.cpu() % 7 != 0).all()


@pytest.mark.parametrize("nq", [1, 16, 40, 64])
def test_sim_topk_stream_large(cuda, nq):
    """Streaming k <= 8 path at index scale (1M rows, several workgroups per CU-range), vs fp32 torch."""
    torch.manual_seed(nq)
    N, D = 1_000_003, 1024
    X = torch.randn(N, D, device=cuda, dtype=torch.bfloat16)
    Q = torch.randn(nq, D, device=cuda, dtype=torch.bfloat16)
    bias = torch.zeros(N, device=cuda)
    bias[5::11] = float("-inf")
    for k in (4, 8):
        v, i = ops.sim_topk(Q, X, bias, N, k)
        s = Q.float() @ X.float().t() + bias
        vr, _ = torch.topk(s, k, dim=-1)
        _close(v, vr, 2e-2, 2e-3, f"stream topk k={k}")
        _close(torch.gather(s, 1, i), vr, 2e-2, 2e-3, "scores of returned ids")
        assert ((i % 11) != 5).all() and (i < N).all()


@pytest.mark.parametrize("nq,N,D,k,kind", [
    (1, 9, 64, 9, "plain"), (2, 40, 384, 33, "plain"), (300, 60, 1024, 16, "plain"), (3, 145, 64, 9, "plain"), (2, 640, 64, 40, "plain"), (17, 16 * 1024, 96, 64, "plain"), (3, 16 * 1024 + 1, 384, 17, "plain"),
    (130, 70_001, 128, 40, "plain"), (33, 300_000, 32, 64, "equal"), (70, 20_000, 64, 7, "plain"), (2, 400_003, 32, 64, "strided"), (5, 2000, 64, 12, "odd")])
def test_sim_topk_long_lists(cuda, nq, N, D, k, kind):
    """k > 8 (group maxima + second pass): small whole numbers, so every sum is exact and the order among equal scores
    (lowest row first) can be compared too. equal: every row the same; strided: the best rows share one thread of the
    selection; odd: NaN, infinite and deleted rows."""
    g = torch.Generator().manual_seed(N + k)
    X = torch.randint(-2, 3, (N, D), generator=g).float()
    Q = torch.randint(-2, 3, (nq, D), generator=g).float()
    bias = torch.zeros(N)
    if kind == "equal":
        X[:] = X[0]
    if kind == "strided":
        bias[7 * 16::16 * 1024] = 1000.0
        bias[7 * 16 + 1::16 * 1024] = 1000.0
        bias[3 * 16:20_000 * 16:16] = torch.arange(bias[3 * 16:20_000 * 16:16].numel()).flip(0) / 64
    if kind == "odd":
        bias[::3] = float("-inf")
        bias[10], bias[11], bias[13] = float("nan"), float("inf"), float("inf")
        bias[16:] = float("-inf")   # nine live rows
    s = Q @ X.t() + bias
    v, i = ops.sim_topk(Q.to(cuda, torch.bfloat16), X.to(cuda, torch.bfloat16), bias.to(cuda), N, k)
    s = torch.where(s.isnan(), torch.full_like(s, float("-inf")), s)
    vr, ir = torch.sort(s, dim=-1, descending=True, stable=True)
    vr, ir = vr[:, :k], ir[:, :k]
    assert torch.equal(v.cpu(), vr)
    assert torch.equal(i.cpu(), torch.where(vr == float("-inf"), torch.full_like(ir, -1), ir))


@pytest.mark.parametrize("nq,k", [(130, 40), (200, 7), (64, 9)])
def test_sim_topk_long_lists_in_slices(cuda, monkeypatch, nq, k):
    """More group maxima than the budget: 64 queries at a time, the last slice shorter; whole numbers, so exact."""
    g = torch.Generator().manual_seed(nq)
    X, Q = torch.randint(-2, 3, (5003, 64), generator=g).float(), torch.randint(-2, 3, (nq, 64), generator=g).float()
    monkeypatch.setattr(ops, "_TOPK_MAXIMA", 1000)
    v, i = ops.sim_topk(Q.to(cuda, torch.bfloat16), X.to(cuda, torch.bfloat16), torch.zeros(5003, device=cuda), 5003, k)
    vr, ir = torch.sort(Q @ X.t(), dim=-1, descending=True, stable=True)
    assert torch.equal(v.cpu(), vr[:, :k]) and torch.equal(i.cpu(), ir[:, :k])


@pytest.mark.parametrize("nq,N,D,k", [(65, 16400, 256, 9), (128, 1000, 320, 16), (129, 129, 1024, 3), (192, 5003, 384, 20),
                                      (193, 128, 256, 7), (257, 40001, 448, 4), (320, 2049, 1024, 40), (321, 33000, 256, 64),
                                      (700, 4097, 768, 10), (66, 300, 96, 10), (320, 20000, 2048, 4)])
def test_sim_topk_many_queries(cuda, nq, N, D, k):
    """More than 64 queries: partial tiles of rows and queries, several query blocks, fewer tiles of rows than CUs and more; the
    same lists, bit for bit, as the same queries 64 at a time. Scores of -inf, NaN and absent rows among them."""
    g = torch.Generator(device=cuda).manual_seed(nq + N)
    X = torch.randn(N, D, device=cuda, generator=g).to(torch.bfloat16)
    Q = torch.randn(nq, D, device=cuda, generator=g).to(torch.bfloat16)
    bias = torch.randn(N, device=cuda, generator=g)
    bias[::7] = float("-inf")
    bias[N - 1] = 5.0
    X[N // 2] = float("nan")
    X[N // 3, 0] = float("inf")
    Q[nq - 1] = 0.0
    v, i = ops.sim_topk(Q, X, bias, N, k)
    parts = [ops.sim_topk(Q[s:s + 64], X, bias, N, max(k, 9)) for s in range(0, nq, 64)]
    if k >= 9:
        assert torch.equal(v, torch.cat([p[0] for p in parts])) and torch.equal(i, torch.cat([p[1] for p in parts]))
    else:     # the best k of the longer lists: the same scores (equal ones may swap rows)
        assert torch.equal(v, torch.cat([p[0] for p in parts])[:, :k])
    if N > k:     # every query's rows are different ones, and have the scores that stand beside them
        got = v.isfinite()
        assert ((i[:, :, None] == i[:, None, :]) & got[:, :, None] & got[:, None, :]).sum() == got.sum()
        own = torch.gather(Q.double() @ X.double().t() + bias.double(), 1, i.clamp_min(0))
        assert ((v.double() - own).abs()[got] <= 1e-5 * D ** 0.5 * 8).all()
    s = Q.double() @ X.double().t() + bias.double()
    s[:, N // 2] = float("-inf")
    want = torch.topk(s.masked_fill(s.isnan(), float("-inf")), k, dim=-1)[0]
    fin = want.isfinite()
    assert ((v.double() - want).abs()[fin] <= 1e-5 * D ** 0.5 * 8).all()     # fp32 sums of D unit products
    assert torch.equal(v.isfinite(), fin)


@pytest.mark.parametrize("nq,N,D,k,off", [
    (1, 33, 64, 2, 0), (3, 641, 192, 40, 0), (2, 1025, 96, 64, 0), (17, 4100, 320, 9, 0), (5, 70_001, 64, 64, 0), (40, 12_345, 1024, 17, 4),
    (64, 262_165, 32, 33, 0), (65, 100, 256, 6, 0), (70, 20_003, 320, 40, 0), (130, 5_021, 384, 64, 0), (200, 9_999, 448, 12, 2),
    (300, 40_007, 256, 50, 0)])
def test_sim_topk_groups_of_four(cuda, monkeypatch, nq, N, D, k, off):
    """Maxima of 4 rows give the lists of maxima of 16 rows, bit for bit, in either first pass and with rows off 16 bytes: whole
    numbers with many equal scores (lowest rows first), then random rows with deleted, infinite and NaN ones among them."""
    g = torch.Generator(device=cuda).manual_seed(N)
    for whole in (True, False):
        make = (lambda *s: torch.randint(-2, 3, s, device=cuda, generator=g)) if whole else (
            lambda *s: torch.randn(*s, device=cuda, generator=g))
        base = make(N * D + off).bfloat16()
        X, Q = base[off:].view(N, D), make(nq, D).bfloat16()
        bias = torch.zeros(N, device=cuda)
        bias[::7] = float("-inf")
        if not whole:
            X[N // 2], X[N // 3, 0] = float("nan"), float("inf")
            bias[N - 1] = 50.0
        got = []
        for rows in (16, 4):
            monkeypatch.setattr(ops, "_topk_group_rows", lambda *a, r=rows: r)
            monkeypatch.setattr(ops, "_topk_lists", lambda *a: False)
            got.append(ops.sim_topk(Q, X, bias, N, k))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
        if whole:
            vr, ir = torch.sort(Q.float() @ X.float().t() + bias, dim=-1, descending=True, stable=True)
            vr, ir = vr[:, :k], ir[:, :k]
            assert torch.equal(got[1][0], vr)
            assert torch.equal(got[1][1], torch.where(vr == float("-inf"), torch.full_like(ir, -1), ir))


@pytest.mark.parametrize("nq,N,D,k", [(300, 33_001, 256, 5), (257, 49_152, 320, 40), (319, 33_000, 1024, 9), (190, 33_001, 256, 12),
                                      (256, 65_535, 320, 64), (193, 40_000, 768, 20)])
def test_sim_topk_tall_tiles(cuda, nq, N, D, k):
    """Tiles of 192 and of 256 rows (a round of them over the chip where two of 128 rows would go): the lists of the same queries 64 at
    a time, bit for bit, partial tiles of rows and queries, deleted and NaN rows among them."""
    g = torch.Generator(device=cuda).manual_seed(nq)
    X = torch.randn(N, D, device=cuda, generator=g).to(torch.bfloat16)
    Q = torch.randn(nq, D, device=cuda, generator=g).to(torch.bfloat16)
    bias = torch.randn(N, device=cuda, generator=g)
    bias[::7] = float("-inf")
    bias[N - 1] = 5.0 * D ** 0.5
    X[N // 2] = float("nan")
    v, i = ops.sim_topk(Q, X, bias, N, k)
    parts = [ops.sim_topk(Q[s:s + 64], X, bias, N, max(k, 9)) for s in range(0, nq, 64)]
    assert torch.equal(v, torch.cat([p[0] for p in parts])[:, :k])
    assert torch.equal(i, torch.cat([p[1] for p in parts])[:, :k])


@pytest.mark.parametrize("nq,D,k", [(1, 32, 1), (3, 100, 4), (70, 1024, 64), (300, 384, 65), (2, 8, 130), (4, 64, 0), (0, 64, 4)])
def test_l2_relevance(cuda, nq, D, k):
    """1 - |q - x| / sqrt(2) from the scores, against 64 bits: the kernel rounds |q|^2 at most D / 64 + 6 times on the way to a sum, so
    d^2 is off by e <= (D / 64 + 8) 2^-24 |q|^2 + 2^-22 |score| and the distance by at most min(e / d, sqrt(e)). Rows at the query itself,
    absent rows (-inf), NaN and strided queries among them."""
    g = torch.Generator(device=cuda).manual_seed(nq + D)
    q = torch.randn(nq, 2 * D, device=cuda, generator=g)[:, ::2]
    raw = torch.randn(nq, k, device=cuda, generator=g) - 0.3 * D
    if nq and k:
        raw[0, 0] = 0.5 * q[0].square().sum()
        raw[nq - 1, k - 1] = float("-inf")
        raw[nq // 2, k // 2] = float("nan")
    got = ops.l2_relevance(q, raw)
    qq = q.double().square().sum(-1, keepdim=True)
    d2 = (qq - 2 * raw.double()).clamp_min(0)
    want = 1 - d2.sqrt() / 2 ** 0.5
    e = (D / 64 + 8) * 2.0 ** -24 * qq + 2.0 ** -22 * raw.double().abs()
    tol = torch.minimum(e / d2.sqrt(), e.sqrt()) + 2.0 ** -22 * (1 + d2.sqrt())
    fin = want.isfinite()
    assert got.shape == (nq, k) and ((got.double() - want).abs() <= tol)[fin].all()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())


def test_sim_topk_group_rows():
    """Which groups, on either side of each line of the rule."""
    rows = ops._topk_group_rows
    assert rows(300, 250_007, 1024, 40) == 4 and rows(300, 250_007, 1024, 10) == 16      # long fetch
    assert rows(300, 640, 1024, 40) == 16 and rows(300, 641, 1024, 40) == 4              # every group is taken
    assert rows(65, 16384 * 16, 1024, 16) == 4 and rows(64, 16384 * 16, 1024, 16) == 16  # the stream's stores
    assert rows(300, 250_000, 1024, 40) == 4 and rows(1100, 250_000, 1024, 40) == 16     # all maxima at once


@pytest.mark.parametrize("nq,D,k", [(3, 64, 10), (70, 256, 10), (70, 256, 4), (2, 1024, 40)])
@pytest.mark.parametrize("off", [2, 4])
def test_sim_topk_rows_off_16_bytes(cuda, nq, D, k, off):
    """Rows (and queries) that begin off a 16-byte line give the bits of the same rows on one: no 16-byte copies to LDS there."""
    torch.manual_seed(nq)
    N = 3000
    base = torch.randn(N * D + off, device=cuda).bfloat16()
    bq = torch.randn(nq * D + off, device=cuda).bfloat16()
    X, Q = base[off:].view(N, D), bq[off:].view(nq, D)
    assert X.data_ptr() % 16 and Q.data_ptr() % 16
    bias = -0.5 * X.float().square().sum(-1)
    want = ops.sim_topk(Q.clone(), X.clone(), bias, N, k)
    for q, x in ((Q, X), (Q.clone(), X), (Q, X.clone())):
        v, i = ops.sim_topk(q, x, bias, N, k)
        assert torch.equal(v, want[0]) and torch.equal(i, want[1])


@pytest.mark.parametrize("nq,N,D,k,room,lists", [
    (65, 16384, 256, 4, 1 << 20, False), (300, 20000, 256, 4, 1250 * 320, False),
    (300, 20000, 256, 4, 1250 * 256, True),     # two slices would read the index twice
    (65, 20000, 256, 3, 1250 * 64, True),       # slices of one tile: the tiled product would not run
    (300, 16383, 256, 4, 1 << 20, True), (65, 20000, 192, 4, 1 << 20, True), (65, 20000, 256, 8, 1000, False)])
def test_sim_topk_form(cuda, monkeypatch, nq, N, D, k, room, lists):
    """Short lists of more queries than a tile: which form answers, with maxima for one slice and for less, and the answer."""
    torch.manual_seed(nq)
    monkeypatch.setattr(ops, "_TOPK_MAXIMA", room)
    X, Q = torch.randn(N, D, device=cuda).bfloat16(), torch.randn(nq, D, device=cuda).bfloat16()
    nat, forms = ops.native(), []

    class Spy:
        def sim_topk(self, *a):
            forms.append(a[6] is not None)
            return nat.sim_topk(*a)

    monkeypatch.setattr(ops, "native", Spy)
    v, i = ops.sim_topk(Q, X, torch.zeros(N, device=cuda), N, k)
    assert set(forms) == {lists}
    s = Q.double() @ X.double().t()
    # bf16 operands, fp32 sums of D products: D * 2^-24 of |q| |x| <= 2 D covers any order
    tol = 2 * D * D * 2.0 ** -24
    assert (v.double() - s.topk(k, dim=1).values).abs().max() <= tol
    assert (torch.gather(s, 1, i) - v.double()).abs().max() <= tol
    assert all(len(set(r)) == k for r in i.tolist())


def test_sim_topk_without_room_for_maxima(cuda, monkeypatch):
    """A card without memory for the group maxima answers k <= 4 from lists."""
    torch.manual_seed(5)
    X, Q = torch.randn(20000, 256, device=cuda).bfloat16(), torch.randn(70, 256, device=cuda).bfloat16()
    bias = torch.zeros(20000, device=cuda)
    want = ops.sim_topk(Q, X, bias, 20000, 4)
    empty = torch.empty

    def small(*a, **k):
        if a[0] == 70 * 1250:
            raise torch.OutOfMemoryError("no room")
        return empty(*a, **k)

    monkeypatch.setattr(torch, "empty", small)
    v, i = ops.sim_topk(Q, X, bias, 20000, 4)
    assert torch.equal(v, want[0]) and torch.equal(i, want[1])
    with pytest.raises(torch.OutOfMemoryError):
        ops.sim_topk(Q, X, bias, 20000, 9)


@pytest.mark.parametrize("nq,k", [(1, 4), (64, 40), (65, 4), (65, 40)])
def test_sim_topk_refuses_wide_rows(cuda, nq, k):
    """Rows too wide for an LDS image of sixteen queries are an error whatever the number of queries."""
    X = torch.zeros(20000, 5120 + 64, device=cuda, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="dimension too large"):
        ops.sim_topk(X[:nq].contiguous(), X, torch.zeros(20000, device=cuda), 20000, k)


def test_sim_topk_no_candidates(cuda):
    """k = 0 asks for nothing and gets empty lists, from the kernel's entry point and from the index."""
    from generativeaiexamples_amd.index.hbm_index import HBMIndex
    X = torch.randn(300, 64, device=cuda)
    v, i = ops.sim_topk(X[:3].bfloat16(), X.bfloat16(), torch.zeros(300, device=cuda), 300, 0)
    assert v.shape == (3, 0) and v.dtype == torch.float32 and i.shape == (3, 0) and i.dtype == torch.int64
    index = HBMIndex(64, "cosine", device=cuda, capacity=300)
    index.add(X)
    assert index.search_raw(X[:3], 0)[1].shape == (3, 0) and index.search(X[:3], 0) == [[], [], []]


@pytest.mark.parametrize("M,N,K", [(64, 6144, 4096), (23, 6080, 4096), (7, 6144, 4096), (33, 5120, 3072), (1, 3072, 2048), (16, 2064, 1024),
                                   (64, 4096, 4096)])
@pytest.mark.parametrize("frag", [True, False])
def test_splitk_slices(cuda, M, N, K, frag):
    """K slices of decode-sized products with six and with eight waves a workgroup, the last of them partly past the columns: every
    slice against 64 bits (sums of exact bf16 products in fp32: K / ks roundings of at most the absolute sum)."""
    g = torch.Generator(device=cuda).manual_seed(N + M)
    x, w = (torch.randn(n, K, device=cuda, generator=g).bfloat16() for n in (M, N))
    ws = torch.full((ops.native().gemm_splitk_ws_floats(M, N, K),), float("nan"), device=cuda)
    ks = ops.native().gemm_qkv_partials(x, ops.shuffle_fragments(w) if frag else w, ws, frag)
    assert ks >= 2
    for i, part in enumerate(ws[:ks * M * N].view(ks, M, N)):
        a, b = (t[:, i * K // ks:(i + 1) * K // ks].double() for t in (x, w))
        tol = K // ks * 2.0 ** -24 * (a.abs() @ b.abs().t())
        assert ((part.double() - a @ b.t()).abs() <= tol).all()


def _scattered(lens, g, skip=()):
    """Packed prompts' positions and slots on shuffled pages; tokens of `skip` have no slot."""
    pages = torch.randperm(sum(-(-n // 16) for n in lens), device="cuda", generator=g)
    pos, slots, at = [], [], 0
    for n in lens:
        p = torch.arange(n, device="cuda")
        pos.append(p)
        slots.append(pages[at:at + -(-n // 16)].repeat_interleave(16)[:n] * 16 + p % 16)
        at += -(-n // 16)
    slots = torch.cat(slots)
    slots[list(skip)] = -1
    return torch.cat(pos).int(), slots.int(), pages.numel()


@pytest.mark.parametrize("D,Hq,Hkv,lens,skip", [(128, 32, 8, [187], ()), (128, 16, 4, [100, 33, 7, 1, 300], (5, 150)), (64, 3, 2, [65], (64,)),
                                                (256, 5, 1, [16, 16, 40], ()), (96, 7, 3, [41, 90], (0,)), (128, 0, 3, [70], ()),
                                                (64, 9, 1, [1] * 80, (8, 9))])
def test_rope_kv_rows(cuda, D, Hq, Hkv, lens, skip):
    """Prompt-sized rotation and cache write: the bits of the same tokens 64 at a time (the kernel of decode-sized steps), nothing
    written for tokens without a slot, with and without the rotation; with head norms the separate norm's rows up to a bf16 step."""
    g = torch.Generator(device=cuda).manual_seed(sum(lens))
    pos, slots, n = _scattered(lens, g, skip)
    T = pos.numel()
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, device=cuda, generator=g).bfloat16()
    cs = torch.randn(512, D, device=cuda, generator=g)

    def run(step, rope=True, norm=None):
        q = torch.full((T, Hq, D), 7.0, device=cuda, dtype=torch.bfloat16)
        kc, vc = torch.full((n, Hkv, 16, D), 7.0, device=cuda).bfloat16(), torch.full((n, Hkv, D, 16), 7.0, device=cuda).bfloat16()
        for a in range(0, T, step):
            b = min(T, a + step)
            args = (pos[a:b].contiguous(), cs, slots[a:b].contiguous(), q[a:b], kc, vc, Hq, Hkv, D)
            if norm:
                ops.norm_rope_kv_write(qkv[a:b].clone(), *norm, 1e-6, *args)
            else:
                ops.rope_kv_write(qkv[a:b], *args, rope)
        return q, kc, vc

    for rope in (True, False):
        for got, want in zip(run(T, rope), run(64, rope)):
            assert torch.equal(got, want)
    if not ops.native().rope_kv_norm_ok(D) or Hq == 0:
        return
    w = [1 + 0.1 * torch.randn(D, device=cuda, generator=g).bfloat16() for _ in range(2)]
    q3 = qkv.view(T, -1, D).clone()
    q3[:, :Hq] = ops.rms_norm(q3[:, :Hq].reshape(-1, D).contiguous(), w[0], 1e-6).view(T, -1, D)
    q3[:, Hq:Hq + Hkv] = ops.rms_norm(q3[:, Hq:Hq + Hkv].reshape(-1, D).contiguous(), w[1], 1e-6).view(T, -1, D)
    got = run(T, norm=w)
    assert all(torch.equal(x, y) for x, y in zip(got, run(7, norm=w)))     # a token's rows do not depend on the others
    qkv = q3.view(T, -1)
    for x, y in zip(got, run(64)):      # a normed element may round the other way: a bf16 step of it, times |cos| + |sin|
        assert ((x.float() - y.float()).abs() <= 2.0 ** -7 * 2 * (cs.abs().max() * q3.float().abs().max())).all()
        assert ((x.float() - y.float()).norm() <= 2.0 ** -9 * y.float().norm())


@pytest.mark.parametrize("D,Hq,Hkv,lens,shift", [(128, 32, 8, [72], 0), (128, 32, 8, [5, 80, 1, 9, 40], 0), (128, 16, 4, [1] * 144, 0), (64, 3, 2, [838], 5),
                                                 (64, 12, 12, [17, 137], 0), (256, 5, 1, [253, 11], 0), (96, 7, 3, [204, 120], 0), (96, 0, 3, [512], 7)])
def test_rope_kv_rows_from(cuda, D, Hq, Hkv, lens, shift):
    """Steps at the line from which the kernel for many rows runs, and a token below it: the bits of 64 tokens at a time. Prompts that begin
    anywhere in the packed rows or in their pages, tokens in pages of their own or in none, a last eight that the rows end in."""
    g = torch.Generator(device=cuda).manual_seed(sum(lens) + D)
    pos, slots, n = _scattered([x + shift for x in lens], g, ())
    pos, slots = pos[shift:], slots[shift:]
    slots[40::211] = -1
    H = Hq + 2 * Hkv
    line = -(-(9 << 16) // ((Hq + 4 * Hkv) * D))
    cs = torch.randn(2048, D, device=cuda, generator=g)
    for T in sorted({min(line - 1, pos.numel()), min(line, pos.numel()), pos.numel()}):
        qkv = torch.randn(T, H * D, device=cuda, generator=g).bfloat16()

        def run(step, rope):
            q = torch.full((T, Hq, D), 7.0, device=cuda, dtype=torch.bfloat16)
            kc, vc = torch.full((n, Hkv, 16, D), 7.0, device=cuda).bfloat16(), torch.full((n, Hkv, D, 16), 7.0, device=cuda).bfloat16()
            for a in range(0, T, step):
                b = min(T, a + step)
                ops.rope_kv_write(qkv[a:b], pos[a:b].contiguous(), cs, slots[a:b].contiguous(), q[a:b], kc, vc, Hq, Hkv, D, rope)
            return q, kc, vc

        for rope in (True, False):
            assert all(torch.equal(x, y) for x, y in zip(run(T, rope), run(64, rope)))


@pytest.mark.parametrize("T,D,E,k", [(65, 32, 1, 1), (80, 96, 5, 5), (200, 4096, 8, 2), (1003, 1056, 16, 4), (97, 64, 3, 2), (66, 2080, 16, 16)])
def test_moe_router_rows(cuda, T, D, E, k):
    """Prompt-sized router against 64 bits: the same experts wherever two scores are further apart than the sums' error, softmax
    weights, equal logits in the order of their ids; W with padding rows, rows of a wider buffer, NaN rows stay NaN."""
    g = torch.Generator(device=cuda).manual_seed(T)
    W = torch.randn(E + 3, D, device=cuda, generator=g).bfloat16()
    x = (torch.randn(T, D + 8, device=cuda, generator=g) * D ** -0.5).bfloat16()[:, :D]
    x[3] = 0
    x[T - 1, D - 1] = float("nan")
    for W_ in (W, W[:E].contiguous()):
        ids, w = ops.moe_router(x, W_, E, k, 1e-9)
        z = x.double() @ W_[:E].double().t()
        err = D * 2.0 ** -24 * (x.double().abs() @ W_[:E].double().abs().t()).max(-1).values    # any order of the sum
        p = z.softmax(-1)
        want, order = torch.sort(p, dim=-1, descending=True, stable=True)
        got = torch.gather(p, 1, ids.long())
        ok = torch.arange(T, device=cuda) < T - 1
        tol = (4 * err + 1e-6)[:, None]     # exp: relative error of the logit's; division and the hardware exponential 1e-6
        assert ((got - want[:, :k]).abs() <= tol * want[:, :k] + 1e-9)[ok].all()
        assert ((w.double() - got / (got.sum(-1, keepdim=True) + 1e-9)).abs() <= 2 * tol + 1e-7)[ok].all()
        assert all(len(set(r)) == k for r in ids[:-1].tolist()) and ids[3].tolist() == list(range(k))
        assert w[T - 1].isnan().all()


@pytest.mark.parametrize("T,D,E,k", [(1, 4096, 8, 2), (64, 64, 16, 4), (5, 96, 5, 5), (7, 2048, 64, 8), (3, 40, 130, 16), (65, 64, 8, 2), (70, 64, 40, 3)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_moe_router_without_scores(cuda, T, D, E, k, bad):
    """A row whose scores are NaN gets expert 0 and NaN weights from every router, an id in range; the rows beside it what they get alone."""
    g = torch.Generator(device=cuda).manual_seed(E)
    W = torch.randn(E, D, device=cuda, generator=g).bfloat16()
    x = (torch.randn(T, D, device=cuda, generator=g) * D ** -0.5).bfloat16()
    want, wts = ops.moe_router(x, W, E, k)
    x[T // 2] = bad
    ids, w = ops.moe_router(x, W, E, k)
    rest = torch.arange(T, device=cuda) != T // 2
    assert (ids[T // 2] == 0).all() and w[T // 2].isnan().all()
    assert torch.equal(ids[rest], want[rest]) and torch.equal(w[rest], wts[rest])
    ids, w = ops.moe_route(x.float() @ W.float().t(), k)
    assert (ids[T // 2] == 0).all() and w[T // 2].isnan().all()


@pytest.mark.parametrize("T", [5, 64, 65, 200])
def test_moe_router_weight_layouts(cuda, T):
    """Router weights in fragment order, or (past 64 rows) rows of a wider buffer: the row-major ones' experts. (512 exact products of unit
    normals and weights of 512^-1/2, summed in fp32: scores to far less than 2^-10.)"""
    torch.manual_seed(T)
    W, x = (torch.randn(64, 512, device=cuda) * 512 ** -0.5).bfloat16(), torch.randn(T, 512, device=cuda).bfloat16()
    p = (x.double() @ W[:9].double().t()).softmax(-1)
    wide = torch.empty(9, 520, device=cuda, dtype=torch.bfloat16)[:, :512].copy_(W[:9])
    frag = W.clone()
    assert ops.to_fragment_layout_(frag)
    for w in (W, frag) + ((wide,) if T > 64 else ()):
        ids, wts = ops.moe_router(x, w, 9, 2)
        got = torch.gather(p, 1, ids.long())
        assert ((got - p.topk(2).values).abs() <= 2.0 ** -10).all()
        assert ((wts.double() - got / got.sum(-1, keepdim=True)).abs() <= 2.0 ** -10).all()


@pytest.mark.parametrize("T,D", [(1, 8), (5, 64), (33, 512), (3, 520), (300, 1024), (9, 1032), (7, 2048), (4, 2056), (0, 64)])
def test_embed_layer_norm(cuda, T, D):
    """The rows of separate gathers, additions and norm, bit for bit: ids outside the table (a row of zeros), the last position; past
    2048 columns those operations themselves run."""
    g = torch.Generator(device=cuda).manual_seed(T + D)
    word, ptab, typ, w, b = (torch.randn(*n, device=cuda, generator=g).bfloat16() for n in ((97, D), (31, D), (2, D), (D,), (D,)))
    ids = torch.randint(-1, 99, (T,), device=cuda, generator=g, dtype=torch.int32)
    pos = torch.randint(0, 31, (T,), device=cuda, generator=g, dtype=torch.int32)
    if T:
        pos[T - 1], ids[0] = 30, 96
    want = ops.layer_norm(ops.embedding(ids, word) + ptab[pos.long()] + typ[1], w, b, 1e-12)
    assert torch.equal(ops.embed_layer_norm(ids, pos, word, ptab, typ[1], w, b, 1e-12), want)


@pytest.mark.parametrize("mode", ["mean", "cls", "last"])
@pytest.mark.parametrize("L,lens,D", [(32, [23], 1024), (5, [5, 0, 1, 3], 64), (128, [128, 7, 0] * 30, 384), (9, [2, 9], 4096)])
def test_pool_padded(cuda, mode, L, lens, D):
    """The first lens[b] rows of each L: what the rows alone give, whatever stands in the padding (NaN here)."""
    torch.manual_seed(L)
    h = torch.randn(len(lens), L, D, device=cuda).bfloat16()
    for i, n in enumerate(lens):
        h[i, max(n, 1):] = float("nan")
        if n == 0 and mode == "mean":
            h[i] = float("nan")
    cu = torch.arange(len(lens) + 1, device=cuda, dtype=torch.int32) * L
    ln = torch.tensor(lens, device=cuda, dtype=torch.int32)
    for normalize in (False, True):
        got = ops.pool(h.view(-1, D), cu, mode, normalize, ln)
        want = ref.pool(h.view(-1, D).cpu(), cu.cpu(), mode, normalize, ln.cpu())
        _close(got, want, 1e-5, 1e-5, "padded pool")
        for other in (ln.long(), torch.stack([ln, ln], 1)[:, 0]):
            assert torch.equal(ops.pool(h.view(-1, D), cu, mode, normalize, other), got)


@pytest.mark.parametrize("D,lens", [(1024, [303, 1, 0, 65]), (384, [512, 7]), (64, [1000, 129, 128]), (8, [2000]), (8192, [3, 9]),
                                    (8208, [2, 20]), (1024, [31, 1, 0, 20, 9]), (2048, [33, 2]), (64, [5, 2, 16]), (8, [3, 30]),
                                    (4096, [1, 3, 17, 2] * 130)])  # the last five: 256 threads for means too
@pytest.mark.parametrize("mode", ["mean", "cls", "last"])
def test_pool_row_groups(cuda, D, lens, mode):
    """More and fewer rows than the groups and their loads hold, one group, widths beyond it; fp32 sums of up to 2000 rows in
    groups of at least two: error below 2000 * 2^-24 of the largest sum."""
    torch.manual_seed(D)
    h = torch.randn(sum(lens), D, device=cuda).to(torch.bfloat16)
    cu = torch.tensor([0] + lens).cumsum(0).to(cuda, torch.int32)
    got, at = ops.pool(h, cu, mode, False), 0
    for b, n in enumerate(lens):
        x = h[at:at + n].double()
        want = torch.zeros(D, device=cuda).double() if n == 0 else x.mean(0) if mode == "mean" else x[0 if mode == "cls" else -1]
        assert ((got[b].double() - want).abs() <= n * 2.0 ** -24 * (x.abs().sum(0) / max(n, 1) + 1e-30)).all()
        at += n


def test_embedding_pool_act(cuda):
    torch.manual_seed(10)
    table = torch.randn(1000, 256, device=cuda, dtype=torch.bfloat16)
    ids = torch.randint(0, 1500, (77,), device=cuda, dtype=torch.int32)
    e = ops.embedding(ids, table, 0, 1000)
    _close(e, ref.embedding(ids.cpu(), table.cpu(), 0, 1000), 0, 0, "embedding")
    e2 = ops.embedding(ids, table, 500, 1500)
    _close(e2, ref.embedding(ids.cpu(), table.cpu(), 500, 1500), 0, 0, "embedding vocab-parallel")
    h = torch.randn(60, 1024, device=cuda, dtype=torch.bfloat16)
    cu = torch.tensor([0, 10, 11, 60], dtype=torch.int32, device=cuda)
    for mode in ("mean", "cls", "last"):
        for norm in (True, False):
            _close(ops.pool(h, cu, mode, norm), ref.pool(h.cpu(), cu.cpu(), mode, norm), 2e-3, 2e-3, mode)
    x = torch.randn(13, 2 * 512, device=cuda, dtype=torch.bfloat16)
    _close(ops.silu_mul(x), ref.silu_mul(x.cpu()), 2e-2, 1e-2, "silu_mul")
    _close(ops.gelu(x), ref.gelu(x.cpu()), 2e-2, 1e-2, "gelu")


@pytest.mark.parametrize("M,N,K", [(2048, 2304, 1024), (1024, 4096, 4096), (3000, 1000, 512)])
def test_gemm_large_repeatable(cuda, M, N, K):
    """Race screen for the pipelined 256x256 kernel: repeated launches must be bit-identical and correct."""
    torch.manual_seed(11)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    y0 = ops.linear(x, w)
    for _ in range(20):
        assert torch.equal(ops.linear(x, w), y0)
    _close(y0, ref.linear(x.cpu(), w.cpu()), 3e-2, 2e-2, "gemm large")


def test_sample_split_path_matches_whole_row(cuda):
    """The split-row sampler (stats / candidate / resolve kernels, V >= 16K) must draw the whole-row
    kernel's token for the same (seed, step): greedy, pure temperature, top-k, top-p, top-k + top-p,
    masked rows, rows with more candidates than the LDS list holds and flat rows (-> whole-row fallback inside
    the resolve kernel)."""
    from generativeaiexamples_amd.ops import native

    torch.manual_seed(21)
    B, V = 64, 128256
    logits = torch.randn(B, V, device=cuda) * 1.28
    logits[5:8] *= 0.01           # flat rows: > 4096 candidates
    logits[9, 1000:] = float("-inf")  # heavily masked row
    logits[10, 5] = 40.0          # one dominant token
    logits[40:46] *= 3.0 / 1.28   # T = 1 on N(0, 3) rows: ~47K candidates, more than the LDS list holds
    temp = torch.full((B,), 0.2, device=cuda)
    temp[:4] = 0.0
    temp[20:28] = 0.9
    temp[40:46] = 1.0
    top_p = torch.full((B,), 0.7, device=cuda)
    top_p[20:24] = 1.0            # pure temperature rows
    top_p[40:46] = 0.9
    top_k = torch.zeros(B, dtype=torch.int32, device=cuda)
    top_k[24:28] = 50
    top_k[28:32] = 1
    top_k[44:46] = 20000          # top-k cut beyond the candidate list, then top-p
    seeds = torch.arange(B, dtype=torch.int64, device=cuda) * 7 + 3
    nat = native()
    assert nat.sample_ws_bytes(B, V) > 0
    agree, total = 0, 0
    for step in range(6):
        a = ops.sample(logits, temp, top_p, top_k, seeds, step)
        b = torch.empty_like(a)
        nat.sample(logits, temp, top_p, top_k, seeds, step, b)  # no workspace: whole-row kernel
        assert torch.equal(a[:4], logits[:4].argmax(-1).int())
        assert torch.equal(a[28:32], logits[28:32].argmax(-1).int())
        assert int(a[10]) == 5
        agree += int((a == b).sum())
        total += B
    assert agree >= 0.97 * total, (agree, total)


def test_sample_split_is_faster(cuda):
    from generativeaiexamples_amd.ops import native

    B, V = 64, 128256
    logits = torch.randn(B, V, device=cuda) * 1.28
    temp = torch.full((B,), 0.2, device=cuda)
    top_p = torch.full((B,), 0.7, device=cuda)
    top_k = torch.zeros(B, dtype=torch.int32, device=cuda)
    seeds = torch.arange(B, dtype=torch.int64, device=cuda)
    out = torch.empty(B, dtype=torch.int32, device=cuda)
    nat = native()
    ws = torch.empty(nat.sample_ws_bytes(B, V), dtype=torch.uint8, device=cuda)

    def timed(fn):
        for _ in range(3):
            fn()
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        for _ in range(20):
            fn()
        e.record()
        e.synchronize()
        return s.elapsed_time(e) / 20 * 1000

    t_split = timed(lambda: nat.sample(logits, temp, top_p, top_k, seeds, 1, out, ws))
    t_row = timed(lambda: nat.sample(logits, temp, top_p, top_k, seeds, 1, out))
    print(f"sampler B=64 V=128256: split {t_split:.1f} us, whole-row {t_row:.1f} us")
    assert t_split < t_row


@pytest.mark.parametrize("R", [2, 8])
def test_sample_tp_candidates_match_whole_row(cuda, R):
    """Vocab-parallel sampling (ops.sample_tp): R shard packets (stats + top-64 candidates) resolved by
    sample_tp_resolve must give the whole-row sampler's token for the same (seed, step): greedy, top-p,
    top-k, top-k + top-p and pure temperature rows. The shards are simulated on one GPU (the gather is a
    plain sum of zero-padded packets, what the TP all-reduce computes)."""
    from generativeaiexamples_amd.ops import native

    torch.manual_seed(31 + R)
    B, V = 64, 128256
    logits = torch.randn(B, V, device=cuda) * 1.28
    logits[3, 77] = 30.0
    temp = torch.full((B,), 0.2, device=cuda)
    temp[:4] = 0.0
    top_p = torch.full((B,), 0.7, device=cuda)
    top_p[40:48] = 1.0  # pure temperature (exact via the shard Gumbel maxima)
    temp[40:48] = 1.0
    top_k = torch.zeros(B, dtype=torch.int32, device=cuda)
    top_k[20:30] = 40
    seeds = torch.arange(B, dtype=torch.int64, device=cuda) + 5
    vl = -(-V // R)
    pad = torch.full((B, vl * R - V), float("-inf"), device=cuda)
    full = torch.cat([logits, pad], 1)
    C = 64
    W = (4 + 2 * C + 3) // 4 * 4
    nat = native()
    for step in range(4):
        buf = torch.zeros(R, B, W, device=cuda)
        for r in range(R):
            sh = full[:, r * vl:(r + 1) * vl].contiguous()
            n = min(vl, V - r * vl)
            nat.sample_tp_stats(sh, r * vl, V, temp, seeds, step, buf[r, :, :4])
            v, i = torch.topk(sh[:, :n], C, dim=-1)
            buf[r, :, 4:4 + C] = v
            buf[r, :, 4 + C:4 + 2 * C] = (i + r * vl).float()
        got = torch.empty(B, dtype=torch.int32, device=cuda)
        flags = torch.zeros(1, dtype=torch.int32, device=cuda)
        nat.sample_tp_resolve(buf, C, V, temp, top_p, top_k, seeds, step, got, flags)
        want = ops.sample(logits, temp, top_p, top_k, seeds, step)
        assert torch.equal(got[:4], logits[:4].argmax(-1).int())
        agree = int((got == want).sum())
        assert agree >= B - 2, (step, agree, (got != want).nonzero().flatten().tolist(), int(flags))


@pytest.mark.parametrize("W,Q,n,k", [(2, 64, 4, 4), (8, 5, 10, 10), (3, 33, 32, 17)])
def test_topk_merge_matches_torch(cuda, W, Q, n, k):
    """Cross-shard merge of W descending candidate lists per query (ops.topk_merge, the sharded index's merge) ==
    torch.topk over the concatenated lists."""
    torch.manual_seed(W * 100 + n)
    vals = torch.randn(W, Q, n, device=cuda).sort(dim=-1, descending=True).values
    vals[:, :, -1] = float("-inf")  # a shard short of n candidates pads with -inf
    top, pos = ops.topk_merge(vals, k)
    ref_v, ref_p = torch.topk(vals.permute(1, 0, 2).reshape(Q, W * n), k, dim=1)
    assert torch.equal(top, ref_v)
    flat = vals.permute(1, 0, 2).reshape(Q, W * n)
    assert torch.equal(torch.gather(flat, 1, pos), ref_v)
