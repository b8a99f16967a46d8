"""Qwen3-Next on gfx950: the gated-DeltaNet decode kernel (in-place slot-pool state update) vs the
fp32 recurrence, and the tiny hybrid model served by the engine (bf16, HIP kernels) vs its CPU fp32
copy, eager vs HIP-graph decode."""
import pytest
import torch

from generativeaiexamples_amd import ops
from generativeaiexamples_amd.engine import EngineConfig, LLMEngine, SamplingParams
from generativeaiexamples_amd.engine.tokenizer import small_byte_tokenizer
from generativeaiexamples_amd.models.qwen3_next import Qwen3NextConfig, Qwen3NextModel, gdn_recurrent_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dk,dv", [(128, 128), (64, 256)])
def test_gdn_decode_kernel(cuda, dk, dv):
    torch.manual_seed(0)
    B, H, NS = 5, 4, 9
    q = torch.nn.functional.normalize(torch.randn(B, H, dk, device=cuda), dim=-1) * dk ** -0.5
    k = torch.nn.functional.normalize(torch.randn(B, H, dk, device=cuda), dim=-1)
    v = torch.randn(B, H, dv, device=cuda)
    g = -torch.rand(B, H, device=cuda)
    beta = torch.rand(B, H, device=cuda)
    state = torch.randn(NS, H, dk, dv, device=cuda) * 0.1
    slots = torch.tensor([7, 0, 3, 8, 5], dtype=torch.int32, device=cuda)
    want_o, want_S = gdn_recurrent_step(q, k, v, g, beta, state[slots.long()])
    before = state.clone()
    out = torch.empty(B, H, dv, device=cuda)
    ops.native().gdn_decode(q, k, v, g, beta, state, slots, out)
    assert torch.allclose(out, want_o, atol=1e-4, rtol=1e-4)
    assert torch.allclose(state[slots.long()], want_S, atol=1e-4, rtol=1e-4)
    untouched = [s for s in range(NS) if s not in slots.tolist()]
    assert torch.equal(state[untouched], before[untouched])


@pytest.mark.parametrize("lens,Hk,Hv,dk,dv", [([1], 1, 1, 64, 16), ([63, 1, 65], 2, 4, 128, 128), ([200, 64], 2, 2, 64, 48),
                                              ([3, 129], 1, 3, 256, 32), ([1000], 2, 4, 128, 128)])
def test_gdn_chunks_against_float64(cuda, lens, Hk, Hv, dk, dv):
    """Chunked rule on the matrix cores, resumed from a non-zero state, against the token-by-token recurrence in float64.
    Bound: the running sum of the log decay reaches -40 in a chunk of these inputs, so a factor e^(G_t - G_s) carries a
    relative error of up to 2 x 40 x 2^-24 = 4.8e-6 however it is computed from fp32 sums; the products' own rounding is
    below it."""
    g_ = torch.Generator().manual_seed(sum(lens))
    T, S = sum(lens), len(lens)
    rn = lambda *s: torch.randn(*s, generator=g_, dtype=torch.float64)  # noqa: E731
    q, k = (torch.nn.functional.normalize(rn(T, Hk, dk), dim=-1) for _ in range(2))
    q, v = q * dk ** -0.5, rn(T, Hv, dv)
    g, beta = -torch.rand(T, Hv, generator=g_, dtype=torch.float64) ** 4 * 3, torch.sigmoid(rn(T, Hv))
    state, slots = rn(S + 2, Hv, dk, dv) * 0.1, list(range(S + 1, 1, -1))
    ins = [t.float() for t in (q, k, v, g, beta)]
    q, k, v, g, beta = (t.double() for t in ins)
    s32 = state.float().to(cuda)
    want, Sw, at = torch.empty(T, Hv, dv, dtype=torch.float64), state.float().double(), 0
    r = Hv // Hk
    for n, slot in zip(lens, slots):
        St = Sw[slot][None].clone()
        for t in range(at, at + n):
            o, St = gdn_recurrent_step(q[t:t + 1].repeat_interleave(r, 1), k[t:t + 1].repeat_interleave(r, 1), v[t:t + 1],
                                       g[t:t + 1], beta[t:t + 1], St)
            want[t] = o[0]
        Sw[slot] = St[0]
        at += n
    out = torch.full((T, Hv, dv), float("nan"), device=cuda)
    chunks, chunk0 = ops.gdn_chunk_plan(lens, cuda)
    ops.gdn_chunks(*(t.to(cuda) for t in ins), chunks, chunk0, torch.tensor(slots, dtype=torch.int32, device=cuda), s32, out)
    for a, b in ((out, want), (s32, Sw)):
        assert (a.cpu().double() - b).norm() <= 4.8e-6 * b.norm()


@pytest.mark.parametrize("lens,Hv,dv", [([1, 64, 0, 65, 130, 7] * 5, 8, 64), ([3, 200] * 32, 8, 64)])
def test_gdn_chunks_many_portions(cuda, lens, Hv, dv):
    """Many short portions of narrow heads, whose kernel differs from that of a few: the bits of every portion by itself."""
    torch.manual_seed(len(lens))
    T, S, Hk, dk = sum(lens), len(lens), 4, 64
    q, k = (torch.nn.functional.normalize(torch.randn(T, Hk, dk, device=cuda), dim=-1) for _ in range(2))
    v, g, beta = torch.randn(T, Hv, dv, device=cuda), -torch.rand(T, Hv, device=cuda), torch.rand(T, Hv, device=cuda)
    state = torch.randn(S, Hv, dk, dv, device=cuda) * 0.1

    def run(at, n, slots):
        st, out = state.clone(), torch.full((sum(n), Hv, dv), float("nan"), device=cuda)
        part = [t[at:at + sum(n)].contiguous() for t in (q, k, v, g, beta)]
        chunks, chunk0 = ops.gdn_chunk_plan(n, cuda)
        ops.gdn_chunks(*part, chunks, chunk0, torch.tensor(slots, dtype=torch.int32, device=cuda), st, out)
        return out, st

    out, st = run(0, lens, list(range(S)))
    at = 0
    for s, n in enumerate(lens):
        if n:
            o1, s1 = run(at, [n], [s])
            assert torch.equal(out[at:at + n], o1) and torch.equal(st[s], s1[s])
        else:
            assert torch.equal(st[s], state[s])
        at += n


@pytest.mark.parametrize("lens,Hk,Hv,dk,dv,dt", [([1, 2, 5], 2, 4, 64, 64, torch.bfloat16), ([700, 1, 3, 0, 9], 1, 3, 128, 48, torch.bfloat16),
                                                 ([1] * 5, 2, 2, 256, 16, torch.float32)])
def test_gdn_prep_matches_torch(cuda, lens, Hk, Hv, dk, dv, dt):
    """Convolution over sequence starts (history from the slot), unit q / k, gates; then the history that is kept."""
    torch.manual_seed(1)
    T, S, kd, vd = sum(lens), len(lens), Hk * dk, Hv * dv
    cd = 2 * kd + vd
    proj = torch.randn(T, cd + vd + 2 * Hv, device=cuda).to(dt)
    cw, cs = torch.randn(cd, 4, device=cuda), torch.randn(S + 3, 3, cd, device=cuda)
    A_log, dt_bias = torch.randn(Hv, device=cuda), torch.randn(Hv, device=cuda)
    slots = torch.randperm(S + 3)[:S].to(cuda, torch.int32)
    cu = torch.tensor([0] + lens).cumsum(0).to(cuda, torch.int32)
    q, k, v, g, beta = ops.gdn_prep(proj, cw, cs, cu, slots, A_log, dt_bias, Hk, dk, Hv, dv)
    x, at, conv, kept = proj[:, :cd].double(), 0, [], cs.double()
    for s, n in enumerate(lens):
        xs = torch.cat([kept[slots[s]], x[at:at + n]])
        if n:
            conv.append((xs.unfold(0, 4, 1) * cw.double()).sum(-1))
            kept[slots[s]] = xs[-3:]
        at += n
    conv = torch.nn.functional.silu(torch.cat(conv))
    unit = lambda t: t * torch.rsqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    b, a = proj[:, cd + vd:cd + vd + Hv].double(), proj[:, cd + vd + Hv:].double()
    want = (unit(conv[:, :kd].view(T, Hk, dk)) * dk ** -0.5, unit(conv[:, kd:2 * kd].view(T, Hk, dk)), conv[:, 2 * kd:].view(T, Hv, dv),
            -torch.exp(A_log.double()) * torch.nn.functional.softplus(a + dt_bias.double()), torch.sigmoid(b))
    for got, w in zip((q, k, v, g, beta), want):
        assert torch.allclose(got.double(), w, rtol=2e-6, atol=2e-6)
    ops.state_tail_write(proj[:, :cd], cs, cu, slots)
    assert torch.allclose(cs.double(), kept, rtol=1e-6, atol=0)


@pytest.mark.parametrize("Hv,dv,dt", [(4, 128, torch.bfloat16), (3, 48, torch.float32), (1, 16, torch.bfloat16)])
def test_gdn_rows_wider_than_their_tensors(cuda, Hv, dv, dt):
    """Projected rows and gates as columns of a wider buffer: the bits of contiguous ones; the gated norm against torch with
    the same roundings (fp32 sums of up to 128 squares: one rounding of the type may fall the other way)."""
    torch.manual_seed(Hv)
    T, Hk, dk, eps = 70, 1, 64, 1e-6
    cd, vd = 2 * Hk * dk + Hv * dv, Hv * dv
    wide = torch.randn(T, 5 + cd + vd + 2 * Hv + 3, device=cuda).to(dt)
    proj = wide[:, 5:5 + cd + vd + 2 * Hv]
    cw, cs = torch.randn(cd, 4, device=cuda), torch.randn(2, 3, cd, device=cuda)
    cu, slots = (torch.tensor(x, dtype=torch.int32, device=cuda) for x in ([0, 30, T], [1, 0]))
    A_log, dt_bias = torch.randn(Hv, device=cuda), torch.randn(Hv, device=cuda)
    for a, b in zip(*(ops.gdn_prep(p, cw, cs, cu, slots, A_log, dt_bias, Hk, dk, Hv, dv) for p in (proj, proj.contiguous()))):
        assert torch.equal(a, b)
    z, o, w = proj[:, cd:cd + vd], torch.randn(T, Hv, dv, device=cuda), torch.randn(dv, device=cuda).to(dt)
    y = ops.gdn_out(o, z, w, eps)
    assert torch.equal(y, ops.gdn_out(o, z.contiguous(), w, eps))
    n = (o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + eps)).to(dt)
    want = (w * n).float() * torch.nn.functional.silu(z.float().view(T, Hv, dv))
    tol = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -20
    assert ((y.view(T, Hv, dv).float() - want).abs() <= tol * want.abs() + 1e-30).all()


@pytest.mark.parametrize("T,Hv,dv,dt", [(4097, 2, 128, torch.bfloat16), (2731, 3, 40, torch.float32), (3, 5, 129, torch.bfloat16),
                                        (9, 1, 256, torch.float32), (2, 3, 300, torch.bfloat16)])
def test_gdn_out_widths(cuda, T, Hv, dv, dt):
    """One head a wave, with a remainder, heads wider than the registers hold: against torch with the
    same roundings (the order of up to 300 squares: one rounding of the type may fall the other way)."""
    torch.manual_seed(dv)
    o, w, z = torch.randn(T, Hv, dv, device=cuda), torch.randn(dv, device=cuda).to(dt), torch.randn(T, Hv * dv, device=cuda).to(dt)
    y = ops.gdn_out(o, z, w, 1e-6)
    n = (o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + 1e-6)).to(dt)
    want = (w * n).float() * torch.nn.functional.silu(z.float().view(T, Hv, dv))
    tol = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -20
    assert ((y.view(T, Hv, dv).float() - want).abs() <= tol * want.abs() + 1e-30).all()


@pytest.mark.parametrize("T,Hv,dv,dt", [(8193, 2, 128, torch.bfloat16), (5463, 3, 40, torch.float32), (16385, 1, 65, torch.bfloat16)])
def test_gdn_out_many_heads_equal_few(cuda, T, Hv, dv, dt):
    """More than 16384 heads run four a wave, with a remainder here: the bits of two calls of one head a wave, which
    test_gdn_out_widths holds against torch."""
    torch.manual_seed(T)
    o, w, z = torch.randn(T, Hv, dv, device=cuda), torch.randn(dv, device=cuda).to(dt), torch.randn(T, Hv * dv, device=cuda).to(dt)
    h = T // 2
    assert h * Hv <= 16384 < T * Hv and (T - h) * Hv <= 16384 and T * Hv % 4
    y = ops.gdn_out(o, z, w, 1e-6)
    assert torch.equal(y, torch.cat([ops.gdn_out(o[:h], z[:h], w, 1e-6), ops.gdn_out(o[h:], z[h:], w, 1e-6)]))


def test_gdn_prep_rows_do_not_depend_on_their_run(cuda):
    """Rows that start, end or lie inside a run of tokens get the bits that they have one token a wave (short calls)."""
    torch.manual_seed(2)
    Hk, Hv, dk, dv, lens = 2, 3, 128, 40, [5, 0, 500, 11, 3, 24, 130]
    T, cd = sum(lens), 2 * Hk * dk + Hv * dv
    proj = torch.randn(T, cd + Hv * dv + 2 * Hv, device=cuda).to(torch.bfloat16)
    cw, cs = torch.randn(cd, 4, device=cuda), torch.randn(len(lens), 3, cd, device=cuda)
    A_log, dt_bias = torch.randn(Hv, device=cuda), torch.randn(Hv, device=cuda)
    cu = torch.tensor([0] + lens).cumsum(0).to(cuda, torch.int32)
    slots = torch.arange(len(lens), dtype=torch.int32, device=cuda)
    many = ops.gdn_prep(proj, cw, cs, cu, slots, A_log, dt_bias, Hk, dk, Hv, dv)
    at = 0
    for s, n in enumerate(lens):
        if n:
            one = ops.gdn_prep(proj[at:at + n], cw, cs, torch.tensor([0, n], dtype=torch.int32, device=cuda), slots[s:s + 1],
                               A_log, dt_bias, Hk, dk, Hv, dv)
            for a, b in zip(many, one):
                assert torch.equal(a[at:at + n], b)
        at += n


def _pair(cuda):
    cfg = Qwen3NextConfig.tiny()
    g = Qwen3NextModel(cfg, device=cuda).random_init(3)
    c = Qwen3NextModel(cfg, device="cpu", dtype=torch.float32)
    for k in c.w:
        c.w[k].copy_(ops.natural_weight(g.w[k]).float().cpu())
    return g, c


def test_qwen3_next_gpu_matches_cpu(cuda):
    g, c = _pair(cuda)
    tok = small_byte_tokenizer(512)
    prompts = [list(range(3, 3 + n)) for n in (9, 40, 100)]
    outs = []
    for m in (g, c):
        eng = LLMEngine(m, tok, EngineConfig(num_blocks=64, max_model_len=512, use_graphs=False))
        for p in prompts:
            eng.add_request(p, SamplingParams(temperature=0.0, max_tokens=1))
        fb, _ = eng._make_batch(eng.sched.schedule())
        outs.append(m.forward(fb, eng.kv, eng.decode_ws).float().cpu())
    err = (outs[0] - outs[1]).abs().max().item()
    assert err < 0.05 * outs[1].abs().max().item() + 0.05, err


def test_qwen3_next_graph_decode_equals_eager(cuda):
    g, _ = _pair(cuda)
    tok = small_byte_tokenizer(512)
    sp = SamplingParams(temperature=0.0, max_tokens=10, ignore_eos=True)
    prompts = [list(range(5, 5 + n)) for n in (7, 30, 64)]
    res = []
    for graphs in (False, True):
        eng = LLMEngine(g, tok, EngineConfig(num_blocks=128, max_model_len=512, use_graphs=graphs,
                                             graph_batch_sizes=(1, 2, 4)))
        res.append([r.output_ids for r in eng.generate(prompts, sp)])
        if graphs:
            assert eng.stats["graph_steps"] > 0
    assert res[0] == res[1]
    assert not g.slot_of


def test_qwen3_next_fragment_weights(cuda):
    """Weights loaded into fragment order: once, again and drawn anew they are the row-major ones reordered, and prompts from a
    token to many rows get the row-major model's bits."""
    pytest.importorskip("transformers")
    from transformers.models.qwen3_next import Qwen3NextConfig as HFConfig, Qwen3NextForCausalLM

    cfg = Qwen3NextConfig.tiny(hidden_size=512, num_heads=8, intermediate_size=512, num_experts=0, linear_num_value_heads=8)
    hc = HFConfig(vocab_size=512, hidden_size=512, intermediate_size=512, num_hidden_layers=4, num_attention_heads=8, num_key_value_heads=2,
                  head_dim=64, linear_num_key_heads=2, linear_num_value_heads=8, linear_key_head_dim=64, linear_value_head_dim=64,
                  num_experts=0, max_position_embeddings=2048, tie_word_embeddings=False, bos_token_id=1, eos_token_id=2)
    g, row = Qwen3NextModel(cfg, device=cuda), Qwen3NextModel(cfg, device="cpu")

    def rows():
        m = Qwen3NextModel(cfg, device=cuda)
        for k in m.w:
            m.w[k].copy_(ops.natural_weight(g.w[k]))
        return m

    for seed in (1, 2):
        torch.manual_seed(seed)
        sd = Qwen3NextForCausalLM(hc).state_dict()
        g.load_hf_state(sd), row.load_hf_state(sd)
        assert ops.is_frag(g.w["l0.out"]) and ops.is_frag(g.w["l3.o"]) and ops.is_frag(g.w["lm_head"]) and not ops.is_frag(g.w["embed"])
        for k in row.w:
            assert torch.equal(ops.natural_weight(g.w[k]).cpu(), row.w[k]), k
    a = rows()
    g.random_init(5), a.random_init(5)
    assert all(torch.equal(ops.natural_weight(g.w[k]), ops.natural_weight(a.w[k])) for k in a.w)
    a = rows()
    assert not any(ops.is_frag(t) for t in a.w.values())
    for n in (1, 9, 90, 700):
        got = []
        for m in (g, a):
            eng = LLMEngine(m, small_byte_tokenizer(512), EngineConfig(num_blocks=64, max_model_len=1024, use_graphs=False))
            eng.add_request([3 + i % 400 for i in range(n)], SamplingParams(temperature=0.0, max_tokens=1))
            fb, _ = eng._make_batch(eng.sched.schedule())
            got.append(m.forward(fb, eng.kv, eng.decode_ws))
        assert torch.equal(*got), n
