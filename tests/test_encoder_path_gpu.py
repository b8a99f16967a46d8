"""Encoder self-attention path (BERT / E5 / CLIP / ViT): the page-packing kernel (ops.kv_pack) against the
per-(token, head) RoPE/KV writer with rotation off, the prefill attention reading q straight from the packed QKV rows
(strided q) against a contiguous q, and the fast branch-free GELU epilogue against PyTorch's exact erf GELU."""
import math

import pytest
import torch

from generativeaiexamples_amd import ops
from generativeaiexamples_amd.models.common import PackedAttention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,H", [(64, 16), (128, 8), (96, 4)])
def test_kv_pack_matches_rope_kv_writer(cuda, D, H):
    torch.manual_seed(D)
    lens = [1, 16, 17, 83, 130]
    T = sum(lens)
    qkv = torch.randn(T, 3 * H * D, device=cuda).to(torch.bfloat16)
    a = PackedAttention(lens, H, D, cuda)
    assert a.pack is not None
    ops.kv_pack(qkv, a.pack[0], a.pack[1], a.k_cache, a.v_cache, H, H, D)
    k2, v2 = torch.zeros_like(a.k_cache), torch.zeros_like(a.v_cache)
    q2 = torch.empty(T, H, D, device=cuda, dtype=torch.bfloat16)
    ops.rope_kv_write(qkv, a.positions, a.cs, a.slots, q2, k2, v2, H, H, D, rope=False)
    assert torch.equal(a.k_cache, k2) and torch.equal(a.v_cache, v2)
    # the CPU path of the op agrees too
    kc, vc = torch.zeros_like(a.k_cache).cpu(), torch.zeros_like(a.v_cache).cpu()
    ops.kv_pack(qkv.cpu(), a.pack[0].cpu(), a.pack[1].cpu(), kc, vc, H, H, D)
    assert torch.equal(kc, k2.cpu()) and torch.equal(vc, v2.cpu())


@pytest.mark.parametrize("D,H", [(64, 16), (128, 8)])
def test_packed_attention_strided_q_matches_fp32(cuda, D, H):
    torch.manual_seed(3)
    lens = [5, 64, 77, 512]
    T = sum(lens)
    qkv = torch.randn(T, 3 * H * D, device=cuda).to(torch.bfloat16)
    a = PackedAttention(lens, H, D, cuda)
    out = a(qkv, 1.0 / math.sqrt(D))
    kv = qkv.float().view(T, 3, H, D)
    ref, t0 = [], 0
    for n in lens:
        q, k, v = kv[t0:t0 + n, 0], kv[t0:t0 + n, 1], kv[t0:t0 + n, 2]
        s = torch.einsum("qhd,khd->hqk", q, k) / math.sqrt(D)
        ref.append(torch.einsum("hqk,khd->qhd", s.softmax(-1), v).reshape(n, H * D))
        t0 += n
    ref = torch.cat(ref)
    err = (out.float() - ref).abs().max().item()
    assert err < 2e-2, err


@pytest.mark.parametrize("M,N,K", [(8192, 4096, 1024), (300, 1024, 4096)])
def test_gelu_epilogue_matches_exact_erf(cuda, M, N, K):
    torch.manual_seed(M)
    x = torch.randn(M, K, device=cuda).to(torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    b = (torch.randn(N, device=cuda) * 0.5).to(torch.bfloat16)
    y = ops.linear(x, w, bias=b, act="gelu")
    ref = torch.nn.functional.gelu(x.float() @ w.float().t() + b.float())
    err = (y.float() - ref).abs().max().item()
    assert err <= 2e-2 * max(1.0, ref.abs().max().item()), err


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("lens,H,short", [([1], 1, 0), ([63, 64, 65, 1, 129], 2, 0), ([512, 7, 300, 128], 16, 0), ([96] * 5, 3, 41)])
def test_rows_attention_equals_paged(cuda, lens, H, short, causal):
    """Keys and values straight from the packed QKV rows: the bits of packing them into pages first; also where only the first
    keys of each sequence count (padded batches)."""
    torch.manual_seed(sum(lens))
    D, T = 64, sum(lens)
    qkv = torch.randn(T, 3 * H * D, device=cuda).to(torch.bfloat16)
    a = PackedAttention(lens, H, D, cuda, causal=causal)
    assert a.direct
    if short and not causal:
        a.ctx = (a.ctx - short).clamp_min(1)
    out = torch.full((T, H * D), float("nan"), device=cuda, dtype=torch.bfloat16)
    assert a(qkv, 0.2, out=out) is not None
    ops.kv_pack(qkv, a.pack[0], a.pack[1], a.k_cache, a.v_cache, H, H, D)
    want = torch.empty(T, H, D, device=cuda, dtype=torch.bfloat16)
    ops.attention_prefill(qkv.view(T, 3 * H, D)[:, :H], a.k_cache, a.v_cache, a.block_tables, a.cu_q, a.ctx, 0.2, causal=causal,
                          tiles=a.tiles, q_lens=lens, out=want)
    assert torch.equal(out, want.view(T, H * D))


@pytest.mark.parametrize("off", [2, 4])
def test_rows_off_16_bytes_take_the_pages(cuda, off):
    """QKV rows that begin off a 16-byte line: the bits of the same rows on one, and no call of the kernel that reads them by
    16-byte buffer loads, which refuses them."""
    torch.manual_seed(off)
    lens, H = [70, 1, 33], 2
    T = sum(lens)
    qkv = torch.randn(T * 3 * H * 64 + off, device=cuda).to(torch.bfloat16)[off:].view(T, 3 * H * 64)
    assert qkv.data_ptr() % 16
    a = PackedAttention(lens, H, 64, cuda)
    assert a.direct and torch.equal(a(qkv, 0.2), a(qkv.clone(), 0.2))
    with pytest.raises(RuntimeError, match="16 bytes"):
        ops.native().attn_rows(qkv, a.tiles, a.cu_q, a.ctx, torch.empty(T, H * 64, device=cuda, dtype=torch.bfloat16), H, 0.2, False)


@pytest.mark.parametrize("H,lens", [(16, [1]), (16, [31, 32, 1]), (16, [33, 17]), (16, [64]), (8, [32, 32]), (8, [5, 0, 40]), (16, [8] * 8)])
def test_attention_layer_norm_short(cuda, H, lens):
    """Attention, projection and norm of a few short sequences in two launches against the three: the attention has the same
    bits, the projection's fp32 sums another order, so a rounding of its bf16 result may fall the other way (2^-8 of it, a
    value of the norm then moves by as much of a standard deviation). Keys past ctx are masked, a sequence without any gives 0."""
    torch.manual_seed(29)
    D, T = H * 64, sum(lens)
    bf = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)  # noqa: E731
    W, b, g, lb, res, qkv = bf(D, D) * D ** -0.5, bf(D), bf(D), bf(D), bf(T, D), bf(T, 3 * D)
    row = W.clone()
    assert ops.to_fragment_layout_(W)
    a = PackedAttention(lens, H, 64, cuda)
    assert ops.attention_layer_norm_ok(qkv, H, a.q_lens, W, (res, b, g, lb))
    for short in (0, 3):
        a.ctx.copy_(torch.tensor([max(n - short, 0) for n in lens], dtype=torch.int32))
        want = ops.linear_layer_norm(a(qkv, 0.125), W, b, res, g, lb, 1e-5).float()
        got = ops.attention_linear_layer_norm(qkv, a.cu_q, a.ctx, a.q_lens, H, 0.125, W, b, res, g, lb, 1e-5).float()
        other = ops.attention_linear_layer_norm(qkv, a.cu_q, a.ctx, a.q_lens, H, 0.125, row, b, res, g, lb, 1e-5)
        assert torch.equal(other.float(), got)  # row-major: the same bits
        assert ((got - want).abs() <= 2 ** -6 * (1 + want.abs())).all() and (got != want).float().mean() < 0.01
    assert not ops.attention_layer_norm_ok(qkv, H, [1] * 9, W, ()) and not ops.attention_layer_norm_ok(bf(65, 3 * D), H, [65], W, ())
