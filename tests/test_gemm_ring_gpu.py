"""Persistent 256x256 prefill GEMMs (csrc/kernels/gemm.hip: w4p / w4d / w4r) against the fp32 reference.

Covers every epilogue, bf16 and fp32 output, partial M / N tiles, the ring tail (K / 32 close to the
ring depth) and launch-to-launch bit-repeatability (race screen for the counted-vmcnt pipeline)."""
import math

import pytest
import torch

from generativeaiexamples_amd import ops
from generativeaiexamples_amd.ops import reference as ref
from generativeaiexamples_amd.utils.graphs import hip_graph_capture

pytestmark = pytest.mark.gpu
# force codes in gai_gemm: persistent 4-wave ring (tile walk per CU), persistent full-line double-unit kernel, and
# its 5-part LDS ring variant (the default for M >= 1024), and that ring on the stream-K walk (K % 128 == 0; forced
# onto shapes with K % 128 != 0 it takes the tile walk)
KERNELS = {"w4p": 8, "w4d": 9, "w4r": 10, "w4s": 11, "w4x": 12,  # w4x: the split walk (k-parts per tile)
           "w4d192": 13}  # the double-slot walk on 192-row tiles (6 A fragments per wave)

SHAPES = [(1024, 256, 192), (1280, 1040, 256), (2048, 2304, 1024), (1100, 4096, 4096), (4096, 6144, 320),
          (1536, 512, 14336), (4608, 4096, 192), (8192, 8448, 256),  # last two: > 256 tiles, multi-tile walks
          (2406, 4096, 1024)]  # the 2406-token O / down row count: 192-row tiles by the auto policy


def _run(x, w, bias, res, act, out_dtype=torch.bfloat16, force=4):
    M, N = x.shape[0], w.shape[0]
    ncol = N // 2 if act == "swiglu" else N
    if act == "swiglu":
        epi = ops.EPI["swiglu"]
    elif act in ("gelu", "relu"):
        epi = ops.EPI[act]
    elif res is not None:
        epi = ops.EPI["bias_residual"] if bias is not None else ops.EPI["residual"]
    else:
        epi = ops.EPI["bias"] if bias is not None else 0
    out = torch.full((M, ncol), float("nan"), device=x.device, dtype=out_dtype)
    ops.native().gemm(x, w, out, bias, res, epi, force)
    return out


@pytest.mark.parametrize("kern", list(KERNELS))
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("act", [None, "bias", "gelu", "relu", "residual", "bias_residual", "swiglu"])
def test_ring_gemm(cuda, M, N, K, act, kern):
    if act == "swiglu" and N % 32:
        pytest.skip("SwiGLU weights interleave in 32-row groups")
    torch.manual_seed(M + 3 * N + K)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    bias = torch.randn(N, device=cuda, dtype=torch.bfloat16) if act in ("bias", "gelu", "relu", "bias_residual") else None
    res = torch.randn(M, N, device=cuda, dtype=torch.bfloat16) if act in ("residual", "bias_residual") else None
    a = act if act in ("gelu", "relu", "swiglu") else None
    y = _run(x, w, bias, res, a, force=KERNELS[kern])
    y_ref = ref.linear(x.cpu(), w.cpu(), None if bias is None else bias.cpu(), None if res is None else res.cpu(), a)
    err = (y.float().cpu() - y_ref.float()).abs()
    tol = 3e-2 + 2e-2 * y_ref.float().abs()
    assert not torch.isnan(y).any(), "unwritten output elements"
    assert (err <= tol).all(), f"ring {M}x{N}x{K} {act}: max err {err.max():.4g}, {(err > tol).sum()} bad"


@pytest.mark.parametrize("kern", list(KERNELS))
@pytest.mark.parametrize("M,N,K", [(1024, 1024, 512), (1300, 2000, 1024)])
def test_ring_gemm_fp32_out(cuda, M, N, K, kern):
    torch.manual_seed(5)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    y = _run(x, w, None, None, None, torch.float32, KERNELS[kern])
    y_ref = x.float().cpu() @ w.float().cpu().t()
    assert (y.cpu() - y_ref).abs().max() < 2e-3 + 2e-3 * y_ref.abs().max()


@pytest.mark.parametrize("kern", list(KERNELS))
@pytest.mark.parametrize("M,N,K", [(1024, 512, 256), (8192, 4352, 448)])
def test_ring_gemm_exact_layout(cuda, kern, M, N, K):
    """Small-integer operands make every product exact in fp32: any row/column mix-up in the swapped
    operand order or the permlane16 epilogue shows as a wrong integer (the second shape walks 2-3 tiles
    per CU in the persistent kernel, so a ring hand-over between tiles is checked exactly too)."""
    torch.manual_seed(9)
    x = torch.randint(-3, 4, (M, K), device=cuda).to(torch.bfloat16)
    w = torch.randint(-3, 4, (N, K), device=cuda).to(torch.bfloat16)
    y = _run(x, w, None, None, None, torch.float32, KERNELS[kern])
    assert torch.equal(y.cpu(), x.float().cpu() @ w.float().cpu().t())


@pytest.mark.parametrize("kern", list(KERNELS))
@pytest.mark.parametrize("M,N,K", [(4096, 4096, 4096), (2304, 6144, 1024)])
def test_ring_gemm_repeatable(cuda, M, N, K, kern):
    torch.manual_seed(11)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    f = KERNELS[kern]
    y0 = _run(x, w, None, None, None, force=f)
    for _ in range(20):
        assert torch.equal(_run(x, w, None, None, None, force=f), y0)
    y_ref = ref.linear(x.cpu(), w.cpu())
    assert ((y0.float().cpu() - y_ref.float()).abs() <= 3e-2 + 2e-2 * y_ref.float().abs()).all()


@pytest.mark.parametrize("walk", ["w4s", "w4x"])
@pytest.mark.parametrize("M,N,K", [(256, 256, 8192), (300, 512, 1024), (2406, 4096, 14336), (1111, 1040, 640)])
@pytest.mark.parametrize("act", [None, "residual", "swiglu"])
def test_stream_k_split_tiles(cuda, M, N, K, act, walk):
    """Stream-K walk with tiles split many ways (64 contributors on the single tile of the first shape, 8 per tile
    on the second, the 2406-token down projection, odd tile edges on the last): small-integer operands make the
    fp32 partial sums exact, so any lost, doubled or misplaced partial quadrant shows as a wrong integer; then
    launch-to-launch bit equality (the sum order does not depend on which contributor finishes last). The split walk
    (w4x) cuts each tile into up to 8 k-parts over the same hand-off."""
    if act == "swiglu" and N % 32:
        pytest.skip("SwiGLU weights interleave in 32-row groups")
    torch.manual_seed(M + N + K)
    x = torch.randint(-2, 3, (M, K), device=cuda).to(torch.bfloat16)
    w = torch.randint(-2, 3, (N, K), device=cuda).to(torch.bfloat16)
    res = torch.randint(-8, 9, (M, N), device=cuda).to(torch.bfloat16) if act == "residual" else None
    out_dtype = torch.bfloat16 if act == "swiglu" else torch.float32  # the SwiGLU epilogue writes bf16
    y = _run(x, w, None, res, act, out_dtype, force=KERNELS[walk])
    acc = x.float().cpu() @ w.float().cpu().t()
    if act == "swiglu":
        g = acc.view(M, N // 32, 2, 16)
        ref_y = (torch.nn.functional.silu(g[:, :, 0]) * g[:, :, 1]).reshape(M, N // 2)
        torch.testing.assert_close(y.float().cpu(), ref_y, rtol=1e-2, atol=1e-2)
    else:
        assert torch.equal(y.cpu(), acc + (0 if res is None else res.float().cpu()))
    for _ in range(5):
        assert torch.equal(_run(x, w, None, res, act, out_dtype, force=KERNELS[walk]), y)


# one tile per workgroup (8192 x 1024: 128 tiles; 1300 x 6144; 2406 x 6144 with bias) and a multi-tile walk
# (8192 x 6144: 768 tiles, 3 per workgroup - the epilogue reads the next tile's first fragments after its stores)
@pytest.mark.parametrize("M,K,Hq,Hkv,with_bias", [(8192, 512, 4, 2, False), (1300, 4096, 32, 8, False),
                                                  (2406, 1024, 32, 8, True), (8192, 256, 32, 8, False)])
def test_prefill_qkv_rope_kv_fused(cuda, M, K, Hq, Hkv, with_bias):
    """Prefill QKV GEMM with RoPE + paged K / V^T write in its epilogue == gemm + rope_kv_write (same
    accumulators, same bf16 roundings); skipped slots (-1) leave the caches untouched."""
    torch.manual_seed(M + K)
    D, nblk = 128, (M + 15) // 16 + 8
    N = (Hq + 2 * Hkv) * D
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    bias = torch.randn(N, device=cuda, dtype=torch.bfloat16) if with_bias else None
    pos = torch.randint(0, 4096, (M,), device=cuda, dtype=torch.int32)
    slots = torch.randperm(nblk * 16, device=cuda)[:M].to(torch.int32)
    slots[::7] = -1
    cs = ops.rope_cos_sin(4096, D, 500000.0, device=cuda)
    outs = []
    for fused in (True, False):
        q = torch.full((M, Hq, D), float("nan"), device=cuda, dtype=torch.bfloat16)
        kc = torch.zeros(nblk, Hkv, 16, D, device=cuda, dtype=torch.bfloat16)
        vc = torch.zeros(nblk, Hkv, D, 16, device=cuda, dtype=torch.bfloat16)
        if fused:
            assert ops.native().gemm_rope_kv(x, w, bias, pos, cs, slots, q, kc, vc, Hq, Hkv, D, 1.0, 1.0,
                                             torch.empty(0, device=cuda), False, None)
        else:
            qkv = torch.empty(M, N, device=cuda, dtype=torch.bfloat16)
            # the fused kernel's tile walk (w4d): same accumulation order (the auto policy may pick the stream-K
            # walk, whose partial sums round differently)
            ops.native().gemm(x, w, qkv, bias, None, ops.EPI["bias"] if with_bias else 0, KERNELS["w4d"])
            ops.rope_kv_write(qkv, pos, cs, slots, q, kc, vc, Hq, Hkv, D, True)
        outs.append((q, kc, vc))
    # same accumulators and roundings; hipcc may contract the rotation's mul-sub into an FMA differently at
    # the two call sites, so a value that cancels to ~0 can differ in its last bit (as the decode test)
    for a, b in zip(*outs):
        torch.testing.assert_close(a.float(), b.float(), rtol=1e-2, atol=1e-5)
        assert (a != b).sum().item() <= max(2, a.numel() // 10000)
    assert not torch.isnan(outs[0][0]).any()
    assert outs[0][1].float().abs().sum() > 0 and outs[0][2].float().abs().sum() > 0  # caches written


def test_prefill_qkv_rope_kv_narrow_declines(cuda):
    """A QKV projection whose 256x256 tiles fill less than half the CUs (1024 x 1024: 16 tiles) is not fused: the
    call returns False and ops.linear_rope_kv takes the plain GEMM + rope_kv path, with the same results."""
    torch.manual_seed(2)
    M, K, Hq, Hkv, D = 1024, 512, 4, 2, 128
    N, nblk = (Hq + 2 * Hkv) * D, 1024 // 16 + 4
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    pos = torch.arange(M, device=cuda, dtype=torch.int32)
    slots = torch.arange(M, device=cuda, dtype=torch.int32)
    cs = ops.rope_cos_sin(4096, D, 500000.0, device=cuda)
    q = torch.empty(M, Hq, D, device=cuda, dtype=torch.bfloat16)
    kc = torch.zeros(nblk, Hkv, 16, D, device=cuda, dtype=torch.bfloat16)
    vc = torch.zeros(nblk, Hkv, D, 16, device=cuda, dtype=torch.bfloat16)
    assert not ops.native().gemm_rope_kv(x, w, None, pos, cs, slots, q, kc, vc, Hq, Hkv, D, 1.0, 1.0,
                                         torch.empty(0, device=cuda), False, None)
    ops.linear_rope_kv(x, w, None, pos, cs, slots, q, kc, vc, Hq, Hkv, D)
    qkv = ref.linear(x.cpu(), w.cpu())
    q2, k2, v2 = torch.empty(M, Hq, D), kc.cpu().float().zero_(), vc.cpu().float().zero_()
    ref.rope_kv_write(qkv, pos.cpu(), cs.cpu(), slots.cpu(), q2, k2, v2, Hq, Hkv, D)
    assert (q.float().cpu() - q2).abs().max().item() < 5e-2
    assert (kc.float().cpu() - k2).abs().max().item() < 5e-2
    assert (vc.float().cpu() - v2).abs().max().item() < 5e-2


@pytest.mark.parametrize("plan", [8101, 8103, 8202, 8204, 12201, 12203])  # 1000 * rows / 16 + 100 * columns / 64 + parts of K
@pytest.mark.parametrize("M,N,K", [(1, 64, 128), (65, 272, 256), (128, 1040, 640), (193, 320, 1152), (700, 2304, 512), (192, 512, 4224)])
@pytest.mark.parametrize("act", [None, "bias", "gelu", "relu", "residual", "bias_residual", "swiglu", "f32"])
def test_mid_gemm(cuda, M, N, K, act, plan):
    """The kernel for a few hundred rows: partial row / column tiles, one to 33 K steps of uneven parts, row-major and
    fragment-ordered weights (same sums), launch after launch the same bits."""
    if act == "swiglu" and N % 32:
        pytest.skip("SwiGLU weights interleave in 32-row groups")
    torch.manual_seed(M + 3 * N + K)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    bias = torch.randn(N, device=cuda, dtype=torch.bfloat16) if act in ("bias", "gelu", "relu", "bias_residual") else None
    res = torch.randn(M, N, device=cuda, dtype=torch.bfloat16) if act in ("residual", "bias_residual") else None
    a = act if act in ("gelu", "relu", "swiglu") else None
    dt = torch.float32 if act == "f32" else torch.bfloat16
    y = _run(x, w, bias, res, a, dt, force=plan)
    y_ref = ref.linear(x.cpu(), w.cpu(), None if bias is None else bias.cpu(), None if res is None else res.cpu(), a, dt)
    err = (y.float().cpu() - y_ref.float()).abs()
    assert not torch.isnan(y).any(), "unwritten output elements"
    tol = 1e-4 if act == "f32" else 3e-2 + 2e-2 * y_ref.float().abs()   # f32: sums of up to 4224 products of unit size / sqrt(K)
    assert (err <= tol).all(), f"{M}x{N}x{K} {act}: max err {err.max():.4g}"
    f = ops.shuffle_fragments(w)
    out = torch.full_like(y, float("nan"))
    for _ in range(3):
        ops.native().gemm(x, f, out, bias, res, {"f32": 0, None: 0}.get(act, ops.EPI.get(act, 0)), plan, True)
        assert torch.equal(out, y)


@pytest.mark.parametrize("M,N,K,act,frag,mid", [
    # the kernels it would replace are the faster ones: short K, sums of the parts past the caches, K deep and tiles even
    (1535, 2176, 384, None, False, False), (2048, 4096, 512, None, True, False), (252, 13936, 128, None, False, False),
    (1536, 11264, 2048, "swiglu", False, False),
    (2048, 4096, 14336, "residual", True, False), (1024, 4096, 14336, "residual", True, False), (128, 1024, 1024, "bias", False, False),
    # and here they are not
    (187, 4096, 14336, "residual", True, True), (65, 1024, 4096, "bias", False, True), (1024, 1024, 1024, "bias_residual", False, True), (768, 6144, 4096, None, True, True),
    (2048, 2048, 2048, "residual", False, True)])
def test_mid_gemm_choice(cuda, M, N, K, act, frag, mid):
    """Where products of 65 - 2048 rows go, at shapes measured with both kernels (the model's comment has the sweep)."""
    x, w = (torch.empty(n, K, device=cuda, dtype=torch.bfloat16) for n in (M, N))
    b = torch.empty(N, device=cuda, dtype=torch.bfloat16) if act in ("bias", "bias_residual") else None
    out = torch.empty(M, N // 2 if act == "swiglu" else N, device=cuda, dtype=torch.bfloat16)
    res = out if act in ("residual", "bias_residual") else None
    assert ops.native().gemm_mid_rows(x, w, out, b, res, ops.EPI[act], frag) == (M if mid else 0)


@pytest.mark.parametrize("M,N,K,act,mid", [
    (1536, 2048, 2048, None, True), (2048, 2048, 2048, None, True), (100, 5632, 2048, "swiglu", True), (128, 5632, 2048, "swiglu", True),
    (400, 8192, 8192, "residual", True), (448, 4096, 14336, "residual", True), (768, 4096, 14336, "residual", True),
    (1536, 4096, 14336, "residual", True), (150, 28672, 4096, "swiglu", True), (512, 6144, 4096, None, True),
    (1024, 4096, 11008, "residual", False), (2048, 2048, 16384, None, False), (512, 14336, 4096, None, False)])
@pytest.mark.parametrize("frag", [False, True])
def test_mid_gemm_choice_near_the_line(cuda, M, N, K, act, mid, frag):
    """Products that a margin or the row-major steps' share decide, timed on both kernels in both layouts: one choice for both,
    and not the slower one in either."""
    x, w = (torch.empty(n, K, device=cuda, dtype=torch.bfloat16) for n in (M, N))
    out = torch.empty(M, N // 2 if act == "swiglu" else N, device=cuda, dtype=torch.bfloat16)
    res = out if act == "residual" else None
    assert ops.native().gemm_mid_rows(x, w, out, None, res, ops.EPI[act], frag) == (M if mid else 0)


@pytest.mark.parametrize("plan", [8105, 8116, 8206, 12208, 0])  # 0: as chosen
@pytest.mark.parametrize("M,N,K,act", [(65, 320, 4224, "bias_residual"), (193, 272, 2048, None), (187, 1024, 14336, "residual"),
                                       (413, 1056, 2176, "swiglu"), (1000, 1024, 1024, "gelu"), (2047, 272, 3072, "relu")])
def test_mid_gemm_many_parts(cuda, M, N, K, act, plan):
    """More parts than one round of the sum takes (four): whole and partial later rounds, uneven parts, both layouts; and the
    plan that is chosen. Repeated launches, also beside each other on two streams, give the same bits."""
    if act == "swiglu" and plan // 100 % 10 == 1:
        pytest.skip("a gated pair needs 128 columns")
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    b = torch.randn(N, device=cuda, dtype=torch.bfloat16) if act in ("gelu", "relu", "bias_residual") else None
    res = torch.randn(M, N, device=cuda, dtype=torch.bfloat16) if act in ("residual", "bias_residual") else None
    y = torch.full((M, N // 2 if act == "swiglu" else N), float("nan"), device=cuda, dtype=torch.bfloat16)
    f, epi = ops.shuffle_fragments(w), ops.EPI[act]
    ops.native().gemm(x, f, y, b, res, epi, plan, True)
    y_ref = ref.linear(x.cpu(), w.cpu(), None if b is None else b.cpu(), None if res is None else res.cpu(),
                       act if act in ("gelu", "relu", "swiglu") else None).float()
    assert ((y.float().cpu() - y_ref).abs() <= 3e-2 + 2e-2 * y_ref.abs()).all()   # the bound of test_mid_gemm: roundings to bf16
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [[torch.full_like(y, float("nan")) for _ in range(4)] for _ in streams]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    for i in range(4):
        for s, o in zip(streams, outs):
            with torch.cuda.stream(s):
                ops.native().gemm(x, f, o[i], b, res, epi, plan, True)
    torch.cuda.synchronize()
    assert all(torch.equal(t, y) for o in outs for t in o)
    ops.native().gemm(x, w, outs[0][0], b, res, epi, plan, False)
    assert torch.equal(outs[0][0], y)


@pytest.mark.parametrize("M,N,K,act", [(187, 4096, 14336, "residual"), (300, 6144, 4096, None), (513, 4096, 4096, "residual"),
                                       (1100, 2048, 4096, "swiglu"), (1536, 11264, 2048, "swiglu"), (128, 1024, 1024, "bias"),
                                       (1400, 3072, 1024, "bias"), (513, 4096, 14336, "residual")])
def test_mid_gemm_choice_is_one_for_both_layouts(cuda, M, N, K, act):
    """Products where the best number of parts, or the best kernel, differs between the weight layouts: equal bits."""
    torch.manual_seed(M)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    b = torch.randn(N, device=cuda, dtype=torch.bfloat16) if act == "bias" else None
    res = torch.randn(M, N, device=cuda, dtype=torch.bfloat16) if act == "residual" else None
    f, epi = ops.shuffle_fragments(w), ops.EPI[act]
    y, yf = (torch.empty(M, N // 2 if act == "swiglu" else N, device=cuda, dtype=torch.bfloat16) for _ in range(2))
    assert ops.native().gemm_mid_rows(x, w, y, b, res, epi, False) == ops.native().gemm_mid_rows(x, f, y, b, res, epi, True)
    ops.native().gemm(x, w, y, b, res, epi, 0, False)
    ops.native().gemm(x, f, yf, b, res, epi, 0, True)
    assert torch.equal(y, yf)


@pytest.mark.parametrize("M,N,K", [(65, 1024, 4096), (192, 1024, 4096), (1536, 1024, 4096), (300, 2048, 5632)])
def test_mid_gemm_captured_equals_eager(cuda, M, N, K):
    """A captured product with parts of K takes the eager one's plan, sums and bits, whatever runs between the replays or
    beside them on the capture stream and on another one."""
    torch.manual_seed(M + K)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w1, w2 = (torch.randn(n, k, device=cuda).div_(math.sqrt(k)).to(torch.bfloat16) for n, k in ((N, K), (K, N)))
    gemm = ops.native().gemm

    def chain(out, mid):
        gemm(x, w1, mid, None, None, 0, 0)
        gemm(mid, w2, out, None, x, ops.EPI["residual"], 0)
        gemm(out, w1, mid, None, None, 0, 0)

    want, mid = torch.empty_like(x), torch.empty(M, N, device=cuda, dtype=torch.bfloat16)
    assert ops.native().gemm_mid_rows(x, w1, mid, None, None, 0, False) == M
    chain(want, mid)
    want_mid = mid.clone()
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    out, gmid = torch.empty_like(x), torch.empty_like(mid)
    s.wait_stream(torch.cuda.current_stream())
    with hip_graph_capture(g, s):
        chain(out, gmid)
    for _ in range(4):
        for t in (out, gmid):
            t.fill_(float("nan"))
        e, emid = torch.empty_like(x), torch.empty_like(mid)
        s.wait_stream(torch.cuda.current_stream())
        g.replay()
        with torch.cuda.stream(s):
            chain(e, emid)
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(gmid, want_mid)
        assert torch.equal(e, want) and torch.equal(emid, want_mid)


def test_mid_gemm_without_memory_for_its_parts(cuda):
    """A full card: the product takes one part of K, which needs no workspace, and nothing is left to fail later."""
    M, N, K = 512, 2048, 4096
    x, w = torch.randn(M, K, device=cuda).bfloat16(), torch.randn(N, K, device=cuda).div_(64).bfloat16()
    one, out = (torch.empty(M, N, device=cuda, dtype=torch.bfloat16) for _ in range(2))
    ops.native().gemm(x, w, one, None, None, 0, 8101)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total, held = torch.cuda.get_device_properties(0).total_memory, []
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            while True:
                held.append(torch.empty(32 << 20, device=cuda, dtype=torch.uint8))
        ops.native().gemm(x, w, out, None, None, 0, 8116)   # 64 MB of partial sums
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        held.clear()
    assert torch.equal(out, one)   # (the comparison takes memory too)
    out.fill_(float("nan"))
    ops.native().gemm(x, w, out, None, None, 0, 8116)
    assert (out.float() - one.float()).abs().max() <= 2.0 ** -6 * one.float().abs().max()


def test_gelu_whole_range(cuda):
    """Every bf16 value through the erf GELU: the 1.5e-7 of the erfc formula (7.1.26) times |x| / 2 and one bf16 rounding;
    the limits at the infinities, NaN kept. The formula is a1 t exp(-z^2) far out, 0.778 / z against erfc's 0.564 / z, so a
    negative x also stays within 0.38 of the (vanishing) value itself."""
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    y = ops.gelu(x.view(64, 1024).to(cuda)).cpu().flatten().double()
    xd = x.double()
    fin = torch.isfinite(xd)
    r = xd[fin] * 0.5 * torch.erfc(-xd[fin] / math.sqrt(2))
    # denormals may be flushed: 1e-37
    tail = torch.where(xd[fin] < 0, torch.minimum(0.75e-7 * xd[fin].abs(), 0.39 * r.abs()), 0.75e-7 * xd[fin])
    assert ((y[fin] - r).abs() <= 2.0 ** -8 * r.abs() + tail + 1e-37).all()
    assert (y[xd == math.inf] == math.inf).all() and (y[xd == -math.inf] == 0).all()
    assert y[torch.isnan(xd)].isnan().all()


@pytest.mark.parametrize("kern", ["w4d", "w4r", "w4d192", "w4x"])
@pytest.mark.parametrize("M,N,K,bias", [(1100, 272, 256, True), (8192, 8448, 256, False), (700, 4096, 1024, True)])
def test_ring_residual_in_place(cuda, M, N, K, bias, kern):
    """The residual may be the output: it is read ahead of the stores, each lane only what it stores itself."""
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    b = torch.randn(N, device=cuda, dtype=torch.bfloat16) if bias else None
    res = torch.randn(M, N, device=cuda, dtype=torch.bfloat16)
    y = _run(x, w, b, res, None, force=KERNELS[kern])
    ops.native().gemm(x, w, res, b, res, ops.EPI["bias_residual" if bias else "residual"], KERNELS[kern])
    assert torch.equal(res, y)


@pytest.mark.parametrize("M,N,K,act,tail", [
    (18337, 1024, 1024, "bias_residual", 1953), (16385, 1024, 4096, "bias_residual", 1), (18484, 1024, 4096, "residual", 2100),
    (13100, 1040, 2048, "gelu", 44), (22000, 720, 1152, "bias", 240), (14500, 1200, 2048, "relu", 1444), (9000, 2048, 4096, "f32", 808),
    (65600, 256, 512, None, 64), (9300, 1792, 1536, "quick_gelu", 84)])
@pytest.mark.parametrize("frag", [False, True])
def test_tail_rows_of_a_large_gemm(cuda, M, N, K, act, tail, frag):
    """Rows past the last whole round of 256x256 tiles go to the mid-size kernel (64- and 128-row tiles), which takes the
    same sums in the same order: the bits of the 256x256 kernel alone, and of equal rows further up."""
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=cuda, dtype=torch.bfloat16)
    x[-5:] = x[:5] if tail >= 5 else x[-5:]
    w = (torch.randn(N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    b = torch.randn(N, device=cuda, dtype=torch.bfloat16) if act in ("gelu", "bias", "relu", "quick_gelu", "bias_residual") else None
    res = torch.randn(M, N, device=cuda, dtype=torch.bfloat16) if act in ("residual", "bias_residual") else None
    if res is not None:
        res[-5:] = res[:5]
    dt = torch.float32 if act == "f32" else torch.bfloat16
    epi = 0 if act == "f32" else ops.EPI[act]
    one, out = (torch.full((M, N), float("nan"), device=cuda, dtype=dt) for _ in range(2))
    ops.native().gemm(x, w, one, b, res, epi, KERNELS["w4r"])
    wf = ops.shuffle_fragments(w) if frag else w
    assert ops.native().gemm_mid_rows(x, wf, out, b, res, epi, frag) == tail
    ops.native().gemm(x, wf, out, b, res, epi, 0, frag)
    assert torch.equal(out, one)
    assert tail < 5 or torch.equal(out[-5:], out[:5])


@pytest.mark.parametrize("sizes", [[300, 0, 1, 700, 256, 0, 257, 40], [0, 0, 5], [1025], [0, 513, 255, 0]])
@pytest.mark.parametrize("N,K", [(64, 128), (1056, 320), (4128, 192)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_grouped_experts(cuda, sizes, N, K, swiglu):
    """Rows sorted by expert in one launch: empty experts, one row, partial row and column tiles, the shortest K, more and
    fewer tiles than CUs. The same bits as each expert by itself on the same kernel: a tile's sums do not depend on its
    neighbours."""
    torch.manual_seed(sum(sizes) + N + K)
    E, rows = len(sizes), sum(sizes)
    x = torch.randn(rows, K, device=cuda, dtype=torch.bfloat16)
    w = (torch.randn(E, N, K, device=cuda) / math.sqrt(K)).to(torch.bfloat16)
    offs = torch.tensor([0] + sizes, dtype=torch.int32).cumsum(0).to(torch.int32).to(cuda)
    y = torch.full((rows, N // 2 if swiglu else N), float("nan"), device=cuda, dtype=torch.bfloat16)
    for _ in range(2):
        assert ops.native().moe_gemm_large(x, w, y, offs, swiglu)
    lo = 0
    for e, n in enumerate(sizes):
        if n:
            part = x[lo:lo + n].contiguous()
            r = ref.linear(part.cpu(), w[e].cpu(), act="swiglu" if swiglu else None).float()
            d = (y[lo:lo + n].float().cpu() - r).abs()
            assert (d <= 3e-2 + 2e-2 * r.abs()).all(), (e, d.max())  # the bound of the walks above: bf16 rounding of both
            if K >= 192:
                assert torch.equal(y[lo:lo + n], _run(part, w[e].contiguous(), None, None, "swiglu" if swiglu else None,
                                                      force=10)), e
        lo += n


def test_grouped_experts_declines(cuda):
    x = torch.zeros(64, 96, device=cuda, dtype=torch.bfloat16)
    w = torch.zeros(2, 64, 96, device=cuda, dtype=torch.bfloat16)
    offs = torch.tensor([0, 30, 64], dtype=torch.int32, device=cuda)
    assert ops.moe_gemm_large(x, w, offs) is None  # K % 64
