"""Model-level numerics on MI355X: the HIP-kernel forward vs the CPU fp32-reference forward of the same
weights, HIP-graph decode vs eager decode, and the embedder / index / engine end to end."""
import pytest
import torch

from generativeaiexamples_amd import ops
from generativeaiexamples_amd.engine import EngineConfig, LLMEngine, SamplingParams
from generativeaiexamples_amd.engine.embedder import Embedder
from generativeaiexamples_amd.engine.tokenizer import bert_byte_tokenizer, small_byte_tokenizer
from generativeaiexamples_amd.models import LlamaConfig, LlamaModel
from generativeaiexamples_amd.models.bert import BertConfig, BertModel

pytestmark = pytest.mark.gpu


def _pair_llama(cuda, **kw):
    cfg = LlamaConfig.tiny(**kw)
    g = LlamaModel(cfg, device=cuda).random_init(3)
    c = LlamaModel(cfg, device="cpu")
    for k in c.w:
        c.w[k].copy_(ops.natural_weight(g.w[k]).cpu())
    return g, c


@pytest.mark.parametrize("kw", [{}, dict(num_heads=8, num_kv_heads=2, head_dim=128, hidden_size=512)])
def test_llama_logits_match_cpu_reference(cuda, kw):
    g, c = _pair_llama(cuda, **kw)
    tok = small_byte_tokenizer(512)
    prompts = [list(range(3, 3 + n)) for n in (9, 40, 100)]
    outs = []
    for m in (g, c):
        eng = LLMEngine(m, tok, EngineConfig(num_blocks=64, max_model_len=512, use_graphs=False))
        for p in prompts:
            eng.add_request(p, SamplingParams(temperature=0.0, max_tokens=1))
        b = eng.sched.schedule()
        fb, _ = eng._make_batch(b)
        outs.append(m.forward(fb, eng.kv, eng.decode_ws).float().cpu())
    err = (outs[0] - outs[1]).abs().max().item()
    assert err < 0.05 * outs[1].abs().max().item() + 0.05, err


def test_llama_graph_decode_equals_eager(cuda):
    g, _ = _pair_llama(cuda)
    tok = small_byte_tokenizer(512)
    sp = SamplingParams(temperature=0.0, max_tokens=12, ignore_eos=True)
    prompts = [list(range(5, 5 + n)) for n in (7, 30, 64, 3)]
    res = []
    for graphs in (False, True):
        eng = LLMEngine(g, tok, EngineConfig(num_blocks=128, max_model_len=512, use_graphs=graphs,
                                             graph_batch_sizes=(1, 2, 4, 8)))
        reqs = eng.generate(prompts, sp)
        res.append([r.output_ids for r in reqs])
        if graphs:
            assert eng.stats["graph_steps"] > 0
    assert res[0] == res[1]


def test_bert_embed_matches_cpu(cuda):
    cfg = BertConfig.tiny()
    g = BertModel(cfg, device=cuda).random_init(1)
    c = BertModel(cfg, device="cpu")
    for k in c.w:
        c.w[k].copy_(ops.natural_weight(g.w[k]).cpu())
    tok = bert_byte_tokenizer(cfg.vocab_size)
    texts = ["hello world", "a much longer passage about accelerators " * 5, "x"]
    eg = Embedder(g, tok).embed(texts).cpu()
    ec = Embedder(c, tok).embed(texts).cpu()
    assert (eg - ec).abs().max().item() < 3e-2
    assert torch.allclose(eg.norm(dim=-1), torch.ones(3), atol=1e-3)


def test_cross_encoder_scores(cuda):
    from generativeaiexamples_amd.engine.embedder import Reranker

    cfg = BertConfig.tiny(num_labels=1, pooling="cls", normalize=False)
    g = BertModel(cfg, device=cuda).random_init(2)
    c = BertModel(cfg, device="cpu")
    for k in c.w:
        c.w[k].copy_(ops.natural_weight(g.w[k]).cpu())
    tok = bert_byte_tokenizer(cfg.vocab_size)
    ps = ["first passage", "second, longer passage " * 4, "third"]
    sg = Reranker(g, tok).score("query text", ps)
    sc = Reranker(c, tok).score("query text", ps)
    assert max(abs(a - b) for a, b in zip(sg, sc)) < 5e-2


def test_hbm_index_roundtrip(cuda, tmp_path):
    from generativeaiexamples_amd.index.hbm_index import Document, HBMIndex

    idx = HBMIndex(64, "cosine", device=cuda, capacity=16)
    v = torch.randn(100, 64, device=cuda)
    idx.add(v, [Document(f"t{i}", {"filename": f"f{i % 5}.txt"}) for i in range(100)])
    hits = idx.search(v[:3], k=1)
    assert [h[0].row for h in hits] == [0, 1, 2]
    assert idx.delete_filename("f0.txt") == 20
    hits = idx.search(v[:1], k=3)[0]
    assert all(h.row % 5 != 0 for h in hits)
    idx.save(str(tmp_path))
    idx2 = HBMIndex.load(str(tmp_path), device=cuda)
    h2 = idx2.search(v[1:2], k=1)[0][0]
    assert h2.row == 1 and h2.document.page_content == "t1"
    l2 = HBMIndex(64, "l2", device=cuda)
    l2.add(v)
    assert l2.search(v[7:8], k=1)[0][0].row == 7


def test_multi_step_graph_decode_equals_single_step(cuda):
    """K=8 decode steps in one captured graph (sampler + decode_advance feedback on device, padded bucket)
    must reproduce one-token-per-step eager decoding (greedy)."""
    g, _ = _pair_llama(cuda)
    tok = small_byte_tokenizer(512)
    prompts = [list(range(9, 9 + n)) for n in (5, 17, 31)]
    sps = [SamplingParams(temperature=0.0, max_tokens=n, ignore_eos=True) for n in (26, 19, 40)]
    res = []
    for steps, graphs in ((1, False), (8, True)):
        eng = LLMEngine(g, tok, EngineConfig(num_blocks=128, max_model_len=512, use_graphs=graphs,
                                             graph_batch_sizes=(1, 2, 4, 8), decode_steps=steps))
        reqs = eng.generate(prompts, sps)
        res.append([r.output_ids for r in reqs])
        if steps > 1:
            assert eng.stats["multi_step_runs"] > 0 and eng.stats["graph_steps"] > 0
            assert eng.sched.num_free_blocks() == eng.sched.num_blocks()
    assert res[0] == res[1]
    # sampled (temperature) multi-step runs stay in range and honour max_tokens
    eng = LLMEngine(g, tok, EngineConfig(num_blocks=128, max_model_len=512, graph_batch_sizes=(1, 2, 4, 8)))
    reqs = eng.generate(prompts, SamplingParams(temperature=0.8, top_p=0.9, max_tokens=24, ignore_eos=True))
    for r in reqs:
        assert len(r.output_ids) == 24 and all(0 <= t < g.cfg.vocab_size for t in r.output_ids)



FUSABLE = dict(hidden_size=1024, intermediate_size=2048, num_heads=8, num_kv_heads=2, head_dim=128)


def test_fused_add_rmsnorm_decode_matches(cuda, monkeypatch):
    """TP=1 decode folds split-K reduce + residual add + RMSNorm into one kernel: the logits of a small
    prefill step (T <= 64, sampled rows) match the unfused path and the CPU fp32 reference, and those of
    a pure decode step (every row sampled: the final norm is fused too) match the unfused path."""
    g, c = _pair_llama(cuda, **FUSABLE)
    assert g.preshuffle_decode_weights() > 0  # fused path on fragment-shuffled weights too
    tok = small_byte_tokenizer(512)
    prompts = [list(range(3, 3 + n)) for n in (9, 20, 30)]
    eng = LLMEngine(g, tok, EngineConfig(num_blocks=64, max_model_len=512, use_graphs=False))
    ceng = LLMEngine(c, tok, EngineConfig(num_blocks=64, max_model_len=512, use_graphs=False))
    for e in (eng, ceng):
        for p in prompts:
            e.add_request(p, SamplingParams(temperature=0.0, max_tokens=4, ignore_eos=True))

    def both(fb):
        outs = {}
        for flag in ("1", "0"):
            monkeypatch.setenv("GAI_FUSE_NORM", flag)
            outs[flag] = g.forward(fb, eng.kv, eng.decode_ws).float().cpu()
        return outs

    fb, _ = eng._make_batch(eng.sched.schedule())
    outs = both(fb)
    cfb, _ = ceng._make_batch(ceng.sched.schedule())
    ref_logits = c.forward(cfb, ceng.kv, ceng.decode_ws).float()
    scale = ref_logits.abs().max().item()
    assert (outs["1"] - outs["0"]).abs().max().item() < 0.02 * scale + 0.02
    assert (outs["1"] - ref_logits).abs().max().item() < 0.05 * scale + 0.05
    # fresh engine state: one full step (prefill + sample), then a pure decode batch
    eng2 = LLMEngine(g, tok, EngineConfig(num_blocks=64, max_model_len=512, use_graphs=False))
    for p in prompts:
        eng2.add_request(p, SamplingParams(temperature=0.0, max_tokens=4, ignore_eos=True))
    eng2.step()
    while eng2._pending is not None:  # the prefill step's tokens are read by the next step() (async launch)
        eng2.step()
    b = eng2.sched.schedule()
    assert b.num_prefill_tokens == 0 if hasattr(b, "num_prefill_tokens") else True
    fb, _ = eng2._make_batch(b)
    outs = {}
    for flag in ("1", "0"):
        monkeypatch.setenv("GAI_FUSE_NORM", flag)
        outs[flag] = g.forward(fb, eng2.kv, eng2.decode_ws).float().cpu()
    assert outs["1"].shape[0] == len(prompts)
    assert (outs["1"] - outs["0"]).abs().max().item() < 0.02 * outs["0"].abs().max().item() + 0.02


def test_metrics_expose_per_gpu_hbm(cuda):
    from generativeaiexamples_amd.utils.metrics import METRICS

    txt = METRICS.render().decode()
    line = next(ln for ln in txt.splitlines() if ln.startswith('gai_gpu_hbm_total_bytes{gpu="0"}'))
    assert float(line.split()[-1]) > 1e11  # 288 GB HBM3E
    assert 'gai_gpu_hbm_used_bytes{gpu="0"}' in txt and 'gai_gpu_hbm_allocated_bytes{gpu="0"}' in txt


def test_query_embed_graph_matches_packed(cuda):
    """Query-sized batches replay a captured fixed-shape (B, L) encoder graph (padded rows, keys masked by the
    real length): embeddings must equal the packed varlen path."""
    cfg = BertConfig.tiny()
    m = BertModel(cfg, device=cuda).random_init(4)
    emb = Embedder(m, bert_byte_tokenizer(cfg.vocab_size))
    qs = [f"what is question {i} about" + " x" * (3 * i) for i in range(5)]
    assert emb.use_graphs
    a = emb.embed(qs, "query")
    assert emb._graphs, "graph path not taken"
    emb.use_graphs = False
    b = emb.embed(qs, "query")
    assert torch.allclose(a, b, atol=2e-2), (a - b).abs().max()
    cos = torch.nn.functional.cosine_similarity(a, b, dim=-1)
    assert bool((cos > 0.999).all()), cos


@pytest.mark.parametrize("hidden,heads,ff", [(1024, 16, 4096), (512, 8, 1024), (512, 16, 2048), (384, 12, 1536)])
def test_encoder_fragment_weights(cuda, hidden, heads, ff):
    """A service's weights in fragment order give the row-major model's bits, from one token to large products (heads padded, and
    projections off the layout's grid, among them); checkpoints come out and go in row-major."""
    cfg = BertConfig(vocab_size=2048, hidden_size=hidden, intermediate_size=ff, num_layers=2, num_heads=heads)
    m = BertModel(cfg, device=cuda).random_init(7)
    state = m.export_hf_state()
    row = BertModel(cfg, device=cuda).load_hf_state(state)
    emb = Embedder(m, bert_byte_tokenizer(cfg.vocab_size))
    assert ops.is_frag(m.w["l1.down"]) and ops.is_frag(m.w["l0.qkv"]) == (hidden % 512 == 0) and not ops.is_frag(row.w["l1.down"])
    after = m.export_hf_state()
    assert all(torch.equal(after[k], state[k]) for k in state)

    def same():
        for lens in ([1], [23], [64, 1], [60, 5], [300, 17], [512] * 9, [33] * 70):
            ids = torch.randint(3, 2048, (sum(lens),), device=cuda, dtype=torch.int32)
            cu = torch.tensor([0] + lens, device=cuda).cumsum(0).int()
            assert torch.equal(m.embed(ids, cu, lens), row.embed(ids, cu, lens))

    same()
    state = BertModel(cfg, device=cuda).random_init(8).export_hf_state()
    m.load_hf_state(state), row.load_hf_state(state)
    same()
    m.random_init(9), row.random_init(9)
    same()
    Embedder(m, emb.tok)    # a second service on the same model
    same()


@pytest.mark.parametrize("L", [40, 100])
def test_query_embed_graph_e5_large_batch64(cuda, L):
    """The headline's query encoder (e5-large-v2 shape) through the graph path at batch 64."""
    cfg = BertConfig.e5_large_v2()
    m = BertModel(cfg, device=cuda).random_init(4)
    emb = Embedder(m, bert_byte_tokenizer(cfg.vocab_size))
    qs = [("q%d " % i) + "y" * (L - 12 - (i % 7)) for i in range(64)]
    a = emb.embed(qs, "query")
    torch.cuda.synchronize()
    assert emb._graphs
    emb.use_graphs = False
    b = emb.embed(qs, "query")
    cos = torch.nn.functional.cosine_similarity(a, b, dim=-1)
    assert bool((cos > 0.999).all()), cos.min()
