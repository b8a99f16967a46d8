"""What a user of this framework has it do, as cases that can be measured: one retrieval-augmented query from its
embedding to its last token, and the decoders served besides the Llama family.

  embed     Embedder.embed_ids              questions (a captured graph) and passages (a packed ragged batch)
  search    HBMIndex.search_raw             exact top-k over the resident index
  prefill   LlamaModel.forward              prompts of one serving step, packed, written to scattered KV pages
  decode    LlamaModel.forward              one token per sequence, replayed from a captured graph as the engine does
  moe       MixtralModel.forward            prompts through routed experts
  delta     Qwen3NextModel.forward          prompts through the gated delta rule and gated attention
  hybrid    BamanexModel.forward            one token per sequence of a windowed-attention hybrid, from a captured graph

Sizes are those of the end-to-end benchmark (Llama-3-8B + e5-large-v2, 506-token chunks, 1M-vector index, ~2400-token
prompts, up to 64 sequences), of the Mixtral 8x7B layers and of the hybrid benchmark's "2k" stacks. Weights are random
tensors under the checkpoints' names, made from the seed, so that `exact` can make the same ones.
"""
from __future__ import annotations

import math
import random
import zlib

import torch
import torch.nn.functional as F

F64 = torch.float64
BF16 = torch.bfloat16
DEV = "cuda"
PAGE = 16                 # tokens of a KV page
MAX_LEN = 8192            # the serving engine's default context limit

LLAMA = dict(D=4096, ff=14336, layers=32, H=32, G=8, hd=128, vocab=128256, theta=500000.0, eps=1e-5)
MIXTRAL = dict(D=4096, ff=14336, layers=4, H=32, G=8, hd=128, vocab=32000, theta=1e6, eps=1e-5, experts=8, top=2)
BERT = dict(D=1024, ff=4096, layers=24, H=16, hd=64, vocab=30522, positions=512, eps=1e-12)
DELTA = dict(D=2048, ff=5632, layers=6, H=16, G=4, hd=128, rot=32, vocab=32768, theta=1e7, eps=1e-6, Hk=8, Hv=16, d=128,
             conv=4, every=3)
HYBRID = dict(D=2048, ff=5632, layers=6, H=16, G=4, hd=128, window=1024, vocab=32768, eps=1e-6)


# ---------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # one question on its way to the index: nothing but latency
        dict(name="embed_question", kind="embed", batch=1, low=23, high=23, questions=True),
        # a document being ingested: chunks of up to 510 tokens, the last of each section shorter
        dict(name="embed_passages", kind="embed", batch=61, low=90, high=510, questions=False),
        # retrieval for one question, the chain server's default of four chunks
        dict(name="search_question", kind="search", queries=1, rows=1_000_000, dim=1024, k=4, metric="cosine"),
        # retrieval for a batch of evaluation questions, forty candidates each for the reranker, euclidean metric
        dict(name="search_batch", kind="search", queries=300, rows=250_007, dim=1024, k=40, metric="l2"),
        # a chat turn without context: a short prompt on the whole model
        dict(name="prefill_short", kind="prefill", batch=1, low=187, high=187),
        # a full step of retrieval-augmented prompts
        dict(name="prefill_rag", kind="prefill", batch=6, low=2203, high=2611),
        # a lone stream's next token
        dict(name="decode_one", kind="decode", batch=1, low=2531, high=2531, cache="bf16"),
        # the benchmark's burst: 64 streams at different points of their answers
        dict(name="decode_batch", kind="decode", batch=64, low=640, high=2663, cache="bf16"),
        # long conversations on the 8-bit cache, an odd number of them
        dict(name="decode_long_fp8", kind="decode", batch=23, low=1900, high=7900, cache="fp8"),
        # prompts of the agentic benchmark's model (layers of the real width)
        dict(name="moe_prefill", kind="moe", batch=2, low=1100, high=1893),
        # a long and a middling prompt through the linear-attention decoder
        dict(name="delta_prefill", kind="delta", batch=2, low=2191, high=6000),
        # many small kernels a token: a hybrid decoder's step at a moderate batch
        dict(name="hybrid_decode", kind="hybrid", batch=24, low=400, high=1700),
    ]


def draw(rng):
    def log(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    def split(total, most):
        """A step of up to `total` tokens as (batch, low, high)."""
        n = rng.randint(1, max(1, min(most, total // 16)))
        mid = max(1, total // n)
        return n, max(1, int(mid * rng.uniform(0.5, 1.0))), mid

    kind = rng.choice(("embed", "embed", "search", "search", "prefill", "prefill", "decode", "decode", "moe", "delta", "hybrid"))
    if kind == "embed":
        if rng.random() < 0.5:
            high = rng.randint(12, 120)
            return dict(kind=kind, batch=log(1, 64), low=rng.randint(8, high), high=high, questions=True)
        high = rng.randint(140, 510)
        return dict(kind=kind, batch=log(2, 61), low=rng.randint(40, high), high=high, questions=False)
    if kind == "search":
        k = rng.choice((1, 3, 4, 4, 8, 10, 20, 40, 50))     # long candidate lists belong to the wide embedder's index
        return dict(kind=kind, queries=log(1, 300), rows=log(5_000, 250_007), dim=1024 if k > 16 else rng.choice((384, 768, 1024)),
                    k=k, metric=rng.choice(("cosine", "cosine", "ip", "l2")))
    if kind == "prefill":
        n, low, high = split(log(17, 14000), 6)
        return dict(kind=kind, batch=n, low=low, high=min(high, 8000))
    if kind == "decode":
        if rng.random() < 0.3:
            return dict(kind=kind, batch=log(1, 23), low=rng.randint(40, 1900), high=rng.randint(1900, 7900), cache="fp8")
        return dict(kind=kind, batch=log(1, 64), low=rng.randint(40, 640), high=rng.randint(700, 2663), cache="bf16")
    if kind == "moe":
        n, low, high = split(log(16, 3000), 4)
        return dict(kind=kind, batch=n, low=low, high=high)
    if kind == "delta":
        n, low, high = split(log(65, 8191), 8)
        return dict(kind=kind, batch=n, low=low, high=high)
    return dict(kind=kind, batch=log(1, 64), low=rng.randint(30, 400), high=rng.randint(401, 3000))


def lengths(case):
    """The case's ragged lengths: evenly spread from low to high, in a fixed mixed-up order."""
    n, lo, hi = case["batch"], case["low"], max(case["low"], case["high"])
    out = [lo + (hi - lo) * (i + 1) // n for i in range(n)] if n > 1 else [hi]
    random.Random(n).shuffle(out)
    return out


# ---------------------------------------------------------------------------------------------------- made-up data
def gen(seed, name):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 2654435761 + zlib.crc32(name.encode())) % (1 << 62))
    return g


def normal(seed, name, *shape, std=1.0, dtype=BF16):
    return torch.randn(*shape, device=DEV, generator=gen(seed, name), dtype=dtype).mul_(std)


def tokens(seed, name, n, vocab):
    return torch.randint(3, vocab, (n,), device=DEV, generator=gen(seed, name))


class Checkpoint:
    """Tensors by checkpoint name, made when they are asked for: {name: (shape, mean, std)}."""

    def __init__(self, seed, shapes):
        self.seed, self.shapes = seed, shapes

    def __iter__(self):
        return iter(self.shapes)

    def __contains__(self, name):
        return name in self.shapes

    def __getitem__(self, name):
        shape, mean, std = self.shapes[name]
        t = normal(self.seed, name, *shape, std=std)
        return t.add_(mean) if mean else t

    def f64(self, name):
        return self[name].to(F64)


class RoutedCheckpoint(Checkpoint):
    """A decoder with experts whose routers have clear preferences, as trained ones do (a router of pure noise has its second
    and third expert within bf16 rounding for every hundredth token, and such a token's result says nothing): a token's
    embedding leans towards a first and, half as much, a second expert's direction, which every layer's router reads."""

    def __getitem__(self, name):
        t = super().__getitem__(name)
        if name == "model.embed_tokens.weight" or name.endswith("block_sparse_moe.gate.weight"):
            D, E = t.shape[1], MIXTRAL["experts"]
            u = normal(self.seed, "experts", E, D, std=D ** -0.5, dtype=torch.float32)
            if t.shape[0] == E:
                return t.mul_(0.5).add_(0.25 * u)
            ids = torch.arange(t.shape[0], device=DEV)
            first = ids % E
            t.add_(32 * u[first] + 16 * u[(first + 1 + ids // E % (E - 1)) % E])
        return t


def lin(out, inn):
    return (out, inn), 0.0, inn ** -0.5


def decoder_shapes(m):
    D, hd = m["D"], m["hd"]
    s = {"model.embed_tokens.weight": ((m["vocab"], D), 0.0, 1.0 if m.get("experts") else 0.02),
         "lm_head.weight": lin(m["vocab"], D), "model.norm.weight": ((D,), 1.0, 0.05)}
    for i in range(m["layers"]):
        p = f"model.layers.{i}."
        s[p + "input_layernorm.weight"] = s[p + "post_attention_layernorm.weight"] = ((D,), 1.0, 0.05)
        s[p + "self_attn.q_proj.weight"] = lin(m["H"] * hd, D)
        s[p + "self_attn.k_proj.weight"] = s[p + "self_attn.v_proj.weight"] = lin(m["G"] * hd, D)
        s[p + "self_attn.o_proj.weight"] = lin(D, m["H"] * hd)
        if m.get("experts"):
            s[p + "block_sparse_moe.gate.weight"] = lin(m["experts"], D)
            for e in range(m["experts"]):
                q = p + f"block_sparse_moe.experts.{e}."
                s[q + "w1.weight"] = s[q + "w3.weight"] = lin(m["ff"], D)
                s[q + "w2.weight"] = lin(D, m["ff"])
        else:
            s[p + "mlp.gate_proj.weight"] = s[p + "mlp.up_proj.weight"] = lin(m["ff"], D)
            s[p + "mlp.down_proj.weight"] = lin(D, m["ff"])
    return s


def decoder_checkpoint(m, seed):
    return (RoutedCheckpoint if m.get("experts") else Checkpoint)(seed, decoder_shapes(m))


def bert_shapes(m):
    D, s = m["D"], {}
    norm, bias = ((D,), 1.0, 0.05), ((D,), 0.0, 0.02)
    e = "embeddings."
    s[e + "word_embeddings.weight"] = ((m["vocab"], D), 0.0, 0.02)
    s[e + "position_embeddings.weight"] = ((m["positions"], D), 0.0, 0.02)
    s[e + "token_type_embeddings.weight"] = ((2, D), 0.0, 0.02)
    s[e + "LayerNorm.weight"], s[e + "LayerNorm.bias"] = norm, bias
    for i in range(m["layers"]):
        p = f"encoder.layer.{i}."
        for n in ("attention.self.query", "attention.self.key", "attention.self.value", "attention.output.dense"):
            s[p + n + ".weight"], s[p + n + ".bias"] = lin(D, D), bias
        s[p + "intermediate.dense.weight"], s[p + "intermediate.dense.bias"] = lin(m["ff"], D), ((m["ff"],), 0.0, 0.02)
        s[p + "output.dense.weight"], s[p + "output.dense.bias"] = lin(D, m["ff"]), bias
        for n in ("attention.output.LayerNorm", "output.LayerNorm"):
            s[p + n + ".weight"], s[p + n + ".bias"] = norm, bias
    return s


def delta_full(m, i):
    return (i + 1) % m["every"] == 0


def delta_shapes(m):
    D, hd, d = m["D"], m["hd"], m["d"]
    s = {"model.embed_tokens.weight": ((m["vocab"], D), 0.0, 0.02), "lm_head.weight": lin(m["vocab"], D),
         "model.norm.weight": ((D,), 0.0, 0.05)}
    for i in range(m["layers"]):
        p = f"model.layers.{i}."
        s[p + "input_layernorm.weight"] = s[p + "post_attention_layernorm.weight"] = ((D,), 0.0, 0.05)
        if delta_full(m, i):
            a = p + "self_attn."
            s[a + "q_proj.weight"] = lin(2 * m["H"] * hd, D)
            s[a + "k_proj.weight"] = s[a + "v_proj.weight"] = lin(m["G"] * hd, D)
            s[a + "q_norm.weight"] = s[a + "k_norm.weight"] = ((hd,), 0.0, 0.05)
            s[a + "o_proj.weight"] = lin(D, m["H"] * hd)
        else:
            a, kd, vd = p + "linear_attn.", m["Hk"] * d, m["Hv"] * d
            s[a + "in_proj_qkvz.weight"] = lin(2 * kd + 2 * vd, D)
            s[a + "in_proj_ba.weight"] = lin(2 * m["Hv"], D)
            s[a + "conv1d.weight"] = ((2 * kd + vd, 1, m["conv"]), 0.0, m["conv"] ** -0.5)
            s[a + "A_log"] = ((m["Hv"],), 1.5, 0.7)      # decay rates of about 1 to 16
            s[a + "dt_bias"] = ((m["Hv"],), -4.0, 1.0)   # time steps of about 0.01 to 0.1, as trained models start
            s[a + "norm.weight"] = ((d,), 1.0, 0.05)
            s[a + "out_proj.weight"] = lin(D, vd)
        s[p + "mlp.gate_proj.weight"] = s[p + "mlp.up_proj.weight"] = lin(m["ff"], D)
        s[p + "mlp.down_proj.weight"] = lin(D, m["ff"])
    return s


def hybrid_shapes(m):
    D, hd, H, G = m["D"], m["hd"], m["H"], m["G"]
    s = {"embed": ((m["vocab"], D), 0.0, 1.0), "head": ((m["vocab"], D), 0.0, 2 * D ** -0.5), "final.norm": ((D,), 0.0, 0.1)}
    for i in range(m["layers"]):
        p, x = f"l{i}.", f"l{i}.mix."
        s[p + "norm1"] = s[p + "norm2"] = ((D,), 0.0, 0.1)
        s[p + "ls1"] = s[p + "ls2"] = ((D,), 0.5, 0.1)
        for n, rows in (("q", H * hd), ("k", G * hd), ("v", G * hd)):
            s[x + n], s[x + n + ".b"] = lin(rows, D), ((rows,), 0.0, 0.1)
        s[x + "sink"], s[x + "g"] = ((H,), 0.0, 1.0), lin(H, D)
        s[x + "o"], s[x + "o.b"] = lin(D, H * hd), ((D,), 0.0, 0.1)
        for n in ("gate", "up"):
            s[p + "mlp." + n] = ((m["ff"], D), 0.0, 1.5 * D ** -0.5)
        s[p + "mlp.down"] = lin(D, m["ff"])
    return s


def page_tables(seed, lens):
    """One page table per sequence over the pages of a server that has run for a while (shuffled)."""
    need = [-(-n // PAGE) for n in lens]
    order = torch.randperm(sum(need), device=DEV, generator=gen(seed, "pages")).to(torch.int32)
    return list(torch.split(order, need))


def cached(seed, layer, blocks, G, hd, dtype):
    """A layer's cached keys [pages, G, 16, hd] and values [pages, G, hd, 16]: unit variance, as random projections of
    normed rows give."""
    k = normal(seed, f"k{layer}", blocks, G, PAGE, hd)
    v = normal(seed, f"v{layer}", blocks, G, hd, PAGE)
    return (k, v) if dtype == BF16 else (k.to(dtype), v.to(dtype))


# ---------------------------------------------------------------------------------------------------- prepare
def prepare(case, seed):
    return {"embed": prepare_embed, "search": prepare_search, "prefill": prepare_prefill, "moe": prepare_prefill,
            "delta": prepare_prefill, "decode": prepare_decode, "hybrid": prepare_decode}[case["kind"]](case, seed)


def bert_batch(case, seed):
    lens = lengths(case)
    flat = tokens(seed, "ids", sum(lens), BERT["vocab"]).tolist()
    out, at = [], 0
    for n in lens:
        out.append(flat[at:at + n])
        at += n
    return out


def prepare_embed(case, seed):
    from generativeaiexamples_amd.engine.embedder import Embedder
    from generativeaiexamples_amd.engine.tokenizer import bert_byte_tokenizer
    from generativeaiexamples_amd.models.bert import BertConfig, BertModel

    model = BertModel(BertConfig.e5_large_v2(), device=DEV).load_hf_state(Checkpoint(seed, bert_shapes(BERT)))
    embedder = Embedder(model, bert_byte_tokenizer(BERT["vocab"]))
    batch = bert_batch(case, seed)
    if case["questions"]:       # a service captures its question buckets when it starts
        embedder.embed_ids(batch)
    return dict(kind="embed", embedder=embedder, batch=batch)


def search_data(case, seed):
    """Index vectors, and questions near some of them."""
    X = normal(seed, "rows", case["rows"], case["dim"], dtype=torch.float32)
    near = torch.randint(0, case["rows"], (case["queries"],), device=DEV, generator=gen(seed, "near"))
    q = X[near] + normal(seed, "questions", case["queries"], case["dim"], std=2.0, dtype=torch.float32)
    return X, q


def prepare_search(case, seed):
    from generativeaiexamples_amd.index.hbm_index import HBMIndex

    X, q = search_data(case, seed)
    index = HBMIndex(case["dim"], case["metric"], device=DEV, capacity=case["rows"])
    index.add(X)
    return dict(kind="search", index=index, q=q, k=case["k"])


def llama(case, seed):
    from generativeaiexamples_amd.models import LlamaConfig, LlamaModel

    model = LlamaModel(LlamaConfig.llama3_8b(), device=DEV).load_hf_state(decoder_checkpoint(LLAMA, seed))
    model.preshuffle_decode_weights(in_place=True)     # the engine's weight layout
    return model


def mixtral(case, seed):
    from generativeaiexamples_amd.models.mixtral import MixtralConfig, MixtralModel

    cfg = MixtralConfig.mixtral_8x7b(num_layers=MIXTRAL["layers"])
    model = MixtralModel(cfg, device=DEV).load_hf_state(decoder_checkpoint(MIXTRAL, seed))
    model.preshuffle_decode_weights(in_place=True)
    return model


def delta(case, seed):
    from generativeaiexamples_amd.models.qwen3_next import Qwen3NextConfig, Qwen3NextModel

    m = DELTA
    cfg = Qwen3NextConfig(name="qwen3-next-2k", vocab_size=m["vocab"], hidden_size=m["D"], intermediate_size=m["ff"],
                          num_layers=m["layers"], num_heads=m["H"], num_kv_heads=m["G"], head_dim=m["hd"],
                          linear_num_key_heads=m["Hk"], linear_num_value_heads=m["Hv"], linear_key_head_dim=m["d"],
                          linear_value_head_dim=m["d"], num_experts=0, mlp_only_layers=tuple(range(m["layers"])),
                          full_attention_interval=m["every"], max_position=32768, bos_token_id=1, eos_token_ids=(2,))
    return Qwen3NextModel(cfg, device=DEV).load_hf_state(Checkpoint(seed, delta_shapes(m)))


def hybrid(case, seed):
    from generativeaiexamples_amd.models.bamanex import BamanexConfig, BamanexModel

    m = HYBRID
    cfg = BamanexConfig.sized(m["D"], m["layers"], m["ff"], m["H"], m["hd"], window=m["window"], vocab=m["vocab"], moe_every=0)
    ck = Checkpoint(seed, hybrid_shapes(m))
    return BamanexModel(cfg, device=DEV).load_state({n: ck[n].cpu() for n in ck})


MODELS = dict(prefill=(llama, LLAMA), moe=(mixtral, MIXTRAL), delta=(delta, DELTA), decode=(llama, LLAMA), hybrid=(hybrid, HYBRID))


def prepare_prefill(case, seed):
    from generativeaiexamples_amd import ops
    from generativeaiexamples_amd.engine.kv_cache import KVCache
    from generativeaiexamples_amd.models.common import ForwardBatch

    make, m = MODELS[case["kind"]]
    model = make(case, seed)
    lens = lengths(case)
    T = sum(lens)
    pages = page_tables(seed, lens)
    blocks = sum(len(p) for p in pages)
    kv = KVCache(getattr(model, "num_kv_layers", m["layers"]), blocks + 1, m["G"], m["hd"], DEV, BF16)
    i32 = dict(dtype=torch.int32, device=DEV)
    pos = torch.cat([torch.arange(n, **i32) for n in lens])
    slots = torch.cat([p.repeat_interleave(PAGE)[:n] * PAGE for p, n in zip(pages, lens)]) + pos % PAGE
    table = torch.zeros(len(lens), max(len(p) for p in pages), **i32)
    for b, p in enumerate(pages):
        table[b, : len(p)] = p
    cu = torch.tensor([0] + lens, **i32).cumsum(0).to(torch.int32)
    fb = ForwardBatch(
        token_ids=tokens(seed, "ids", T, m["vocab"]).to(torch.int32), positions=pos, slots=slots, num_prefill_tokens=T,
        cu_q=cu, prefill_ctx=torch.tensor(lens, **i32), prefill_block_tables=table,
        prefill_tiles=ops.build_prefill_tiles(lens, m["H"], m["G"], DEV, head_dim=m["hd"]), prefill_qlen=lens,
        prefill_ctx_host=list(lens), seq_ids=list(range(1, len(lens) + 1)),
        # a served step wants each prompt's last row; the routed model scores every row, as an evaluation does
        sample_rows=None if case["kind"] == "moe" else cu[1:].long() - 1)
    return dict(kind=case["kind"], model=model, kv=kv, fb=fb)


def prepare_decode(case, seed):
    from generativeaiexamples_amd import ops
    from generativeaiexamples_amd.engine.kv_cache import KVCache
    from generativeaiexamples_amd.models.common import ForwardBatch
    from generativeaiexamples_amd.utils.graphs import hip_graph_capture

    make, m = MODELS[case["kind"]]
    model = make(case, seed)
    lens = lengths(case)
    B = len(lens)
    pages = page_tables(seed, lens)
    blocks = sum(len(p) for p in pages)
    dtype = torch.float8_e4m3fn if case.get("cache") == "fp8" else BF16
    layout = model.kv_layout() if hasattr(model, "kv_layout") else None
    kv = KVCache(m["layers"], blocks + 1, m["G"], m["hd"], DEV, dtype, layout=layout)
    for i in range(m["layers"]):
        k, v = cached(seed, i, blocks, m["G"], m["hd"], dtype)
        kv.layer(i)[0][:blocks] = k
        kv.layer(i)[1][:blocks] = v
    i32 = dict(dtype=torch.int32, device=DEV)
    ctx = torch.tensor(lens, **i32)
    table = torch.full((B, MAX_LEN // PAGE), blocks, **i32)     # unused entries: the scratch page
    for b, p in enumerate(pages):
        table[b, : len(p)] = p
    slots = torch.stack([p[-1] for p in pages]) * PAGE + (ctx - 1) % PAGE
    fb = ForwardBatch(token_ids=tokens(seed, "ids", B, m["vocab"]).to(torch.int32), positions=ctx - 1, slots=slots.to(torch.int32),
                      num_prefill_tokens=0, decode_ctx=ctx, decode_block_tables=table, max_decode_ctx=MAX_LEN)
    ws = None
    if layout is None:
        ws = ops.DecodeWorkspace(B, m["H"], m["hd"], MAX_LEN, torch.device(DEV))
    else:
        fb.extra = model.graph_static_inputs(B)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.inference_mode():
        with torch.cuda.stream(stream):
            model.forward(fb, kv, ws)
        torch.cuda.current_stream().wait_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with hip_graph_capture(graph, stream):
            logits = model.forward(fb, kv, ws)
    return dict(kind=case["kind"], model=model, kv=kv, fb=fb, ws=ws, graph=graph, logits=logits)


# ---------------------------------------------------------------------------------------------------- run
def run(state):
    kind = state["kind"]
    if kind == "embed":
        return state["embedder"].embed_ids(state["batch"])
    if kind == "search":
        return state["index"].search_raw(state["q"], state["k"])
    if kind in ("decode", "hybrid"):
        state["graph"].replay()
        kv = state["kv"]
        return [state["logits"]] + ([kv.storage] if kv.storage is not None else list(kv.k) + list(kv.v))
    model = state["model"]
    with torch.inference_mode():
        if kind == "delta":
            model.prepare_batch(state["fb"])
            out = [model.forward(state["fb"], state["kv"]), state["kv"].storage, model.ssm_state, model.conv_state]
        else:
            out = [model.forward(state["fb"], state["kv"]), state["kv"].storage]
    return out


# ---------------------------------------------------------------------------------------------------- work
def attended(lens, window=0):
    """(query, key) pairs of causal prompts."""
    return sum(n * (n + 1) // 2 if not window or n <= window else window * (window + 1) // 2 + (n - window) * window for n in lens)


def work(case):
    kind = case["kind"]
    if kind == "embed":
        m, lens = BERT, lengths(case)
        layer, T = 4 * m["D"] ** 2 + 2 * m["D"] * m["ff"], sum(lens)
        return dict(bytes=2 * (m["layers"] * layer + T * m["D"]) + 4 * len(lens) * m["D"],
                    flops=2 * m["layers"] * (layer * T + 2 * m["D"] * sum(n * n for n in lens)))
    if kind == "search":
        n = case["rows"] * case["dim"]
        return dict(bytes=2 * n + 4 * case["rows"] + 4 * case["queries"] * case["dim"] + 12 * case["queries"] * case["k"],
                    flops=2 * case["queries"] * n)
    m, lens = MODELS[kind][1], lengths(case)
    D, hd, H, G, L = m["D"], m["hd"], m["H"], m["G"], m["layers"]
    step = kind in ("decode", "hybrid")
    T = len(lens) if step else sum(lens)
    rows = T if kind == "moe" else len(lens)
    attn = (2 * H + 2 * G) * hd * D
    full, ff = L, 3 * D * m["ff"]
    used = read = attn + ff
    linear = 0
    if kind == "moe":
        used, read = attn + m["top"] * ff, attn + m["experts"] * ff
    if kind == "delta":
        full = sum(delta_full(m, i) for i in range(L))
        attn += H * hd * D
        vd, kd = m["Hv"] * m["d"], m["Hk"] * m["d"]
        lin_attn = (2 * kd + 3 * vd + 2 * m["Hv"]) * D
        used = read = ff + (full * attn + (L - full) * lin_attn) / L
        linear = (L - full) * T * m["Hv"] * m["d"] * m["d"] * 3       # decay, read and write of the state
    window = m.get("window", 0)
    pairs = sum(min(n, window or n) for n in lens) if step else attended(lens)
    size = 1 if case.get("cache") == "fp8" else 2
    moved = pairs if step else 2 * T                # cached rows read (decode), rows written and read once (prefill)
    return dict(bytes=2 * (L * read + m["vocab"] * D + T * D) + 2 * size * full * moved * G * hd + 4 * rows * m["vocab"],
                flops=2 * (L * used * T + rows * m["vocab"] * D + 2 * full * pairs * H * hd + linear))


# ---------------------------------------------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times what the path differs from `exact`."""
    if case["kind"] == "search":
        return dict(rel=1e-5, differ=0.02)      # fp32 sums of bf16 products; near-ties may swap places
    return dict(rel=dict(embed=0.04, prefill=0.07, decode=0.16, moe=0.06, delta=0.1, hybrid=0.025)[case["kind"]])


# ---------------------------------------------------------------------------------------------------- exact
def exact(case, seed):
    with torch.no_grad():
        return {"embed": exact_embed, "search": exact_search, "prefill": exact_prefill, "moe": exact_prefill,
                "delta": exact_delta, "decode": exact_decode, "hybrid": exact_hybrid}[case["kind"]](case, seed)


def rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def rope(x, pos, theta, rot=None):
    """x [T, heads, d]: channels i and i + rot / 2 turned together."""
    rot = rot or x.shape[-1]
    h = rot // 2
    ang = pos.to(F64)[:, None] * theta ** (-torch.arange(0, rot, 2, device=x.device, dtype=F64) / rot)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., :h], x[..., h:rot]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., rot:]], -1)


def attend(q, k, v, scale, causal):
    """q [T, H, d], k / v [S, G, d] of one sequence -> [T, H * d]."""
    rep = q.shape[1] // k.shape[1]
    out = torch.empty_like(q)
    for g in range(k.shape[1]):
        s = torch.matmul(q[:, g * rep:(g + 1) * rep].transpose(0, 1), k[:, g].t()) * scale
        if causal:
            s.masked_fill_(torch.ones(q.shape[0], k.shape[0], dtype=torch.bool, device=q.device).triu(1), -math.inf)
        out[:, g * rep:(g + 1) * rep] = torch.matmul(s.softmax(-1), v[:, g]).transpose(0, 1)
    return out.reshape(q.shape[0], -1)


def swiglu(x, gate, up, down):
    return (F.silu(x @ gate.t()) * (x @ up.t())) @ down.t()


def pieces(lens):
    at = 0
    for n in lens:
        yield at, at + n
        at += n


def write_pages(K, V, k, v, pages, lens):
    """Rows of packed prompts into their pages of K [pages, G, 16, d] and V [pages, G, d, 16]."""
    for (a, b), p in zip(pieces(lens), pages):
        pad = len(p) * PAGE - (b - a)
        for X, x, swap in ((K, k, False), (V, v, True)):
            t = F.pad(x[a:b], (0, 0, 0, 0, 0, pad)).view(len(p), PAGE, *x.shape[1:]).transpose(1, 2)
            X[p.long()] = t.transpose(2, 3) if swap else t


def exact_embed(case, seed):
    m, ck, lens = BERT, Checkpoint(seed, bert_shapes(BERT)), lengths(case)
    D, H, hd = m["D"], m["H"], m["hd"]
    ids = torch.tensor([t for s in bert_batch(case, seed) for t in s], device=DEV)
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens])

    def norm(x, p):
        return F.layer_norm(x, (D,), ck.f64(p + ".weight"), ck.f64(p + ".bias"), m["eps"])

    def lin64(x, p):
        return x @ ck.f64(p + ".weight").t() + ck.f64(p + ".bias")

    e = "embeddings."
    h = ck.f64(e + "word_embeddings.weight")[ids] + ck.f64(e + "position_embeddings.weight")[pos]
    h = norm(h + ck.f64(e + "token_type_embeddings.weight")[0], e + "LayerNorm")
    for i in range(m["layers"]):
        p = f"encoder.layer.{i}."
        q, k, v = (lin64(h, p + f"attention.self.{n}").view(-1, H, hd) for n in ("query", "key", "value"))
        a = torch.cat([attend(q[s:t], k[s:t], v[s:t], hd ** -0.5, False) for s, t in pieces(lens)])
        h = norm(lin64(a, p + "attention.output.dense") + h, p + "attention.output.LayerNorm")
        f = F.gelu(lin64(h, p + "intermediate.dense"))
        h = norm(lin64(f, p + "output.dense") + h, p + "output.LayerNorm")
    return F.normalize(torch.stack([h[s:t].mean(0) for s, t in pieces(lens)]), dim=-1)


def exact_search(case, seed):
    """The index stores and compares bf16 vectors: what is rounded is its input, the sums are exact here."""
    X, q = search_data(case, seed)
    if case["metric"] == "cosine":
        X, q = F.normalize(X, dim=-1), F.normalize(q, dim=-1)
    X, qb = X.to(BF16).to(F64), q.to(BF16).to(F64)
    s = qb @ X.t()
    if case["metric"] == "l2":
        s -= 0.5 * X.square().sum(-1)
    s, rows = s.topk(min(case["k"], case["rows"]), -1)
    if case["metric"] == "l2":
        s = 1 - (q.to(F64).square().sum(-1, keepdim=True) - 2 * s).clamp_min(0).sqrt() / math.sqrt(2)
    return s, rows


def exact_prefill(case, seed):
    m, lens = MODELS[case["kind"]][1], lengths(case)
    ck, T, D, H, G, hd = decoder_checkpoint(m, seed), sum(lens), m["D"], m["H"], m["G"], m["hd"]
    pages = page_tables(seed, lens)
    blocks = sum(len(p) for p in pages) + 1
    kv = torch.zeros(m["layers"], 2, blocks * G * PAGE * hd, device=DEV, dtype=F64)
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens])
    h = ck.f64("model.embed_tokens.weight")[tokens(seed, "ids", T, m["vocab"])]
    for i in range(m["layers"]):
        p = f"model.layers.{i}."
        x = rms(h, ck.f64(p + "input_layernorm.weight"), m["eps"])
        q, k, v = ((x @ ck.f64(p + f"self_attn.{n}_proj.weight").t()).view(T, -1, hd) for n in "qkv")
        q, k = rope(q, pos, m["theta"]), rope(k, pos, m["theta"])
        write_pages(kv[i, 0].view(blocks, G, PAGE, hd), kv[i, 1].view(blocks, G, hd, PAGE), k, v, pages, lens)
        a = torch.cat([attend(q[s:t], k[s:t], v[s:t], hd ** -0.5, True) for s, t in pieces(lens)])
        h = h + a @ ck.f64(p + "self_attn.o_proj.weight").t()
        del q, k, v, a
        x = rms(h, ck.f64(p + "post_attention_layernorm.weight"), m["eps"])
        if not m.get("experts"):
            h = h + swiglu(x, *(ck.f64(p + f"mlp.{n}_proj.weight") for n in ("gate", "up", "down")))
            continue
        q = p + "block_sparse_moe."
        w, ids = (x @ ck.f64(q + "gate.weight").t()).softmax(-1).topk(m["top"], -1)
        w = w / w.sum(-1, keepdim=True)
        out = torch.zeros_like(h)
        for e in range(m["experts"]):
            t, j = (ids == e).nonzero(as_tuple=True)
            y = swiglu(x[t], *(ck.f64(q + f"experts.{e}.{n}.weight") for n in ("w1", "w3", "w2")))
            out.index_add_(0, t, w[t, j][:, None] * y)
        h = h + out
    if case["kind"] != "moe":
        h = h[torch.tensor(lens, device=DEV).cumsum(0) - 1]
    return [rms(h, ck.f64("model.norm.weight"), m["eps"]) @ ck.f64("lm_head.weight").t(), kv]


def exact_decode(case, seed):
    """The logits; the cache that the step adds one row a sequence to is not rebuilt."""
    m, lens = LLAMA, lengths(case)
    ck, B, G, hd = decoder_checkpoint(m, seed), len(lens), m["G"], m["hd"]
    pages = page_tables(seed, lens)
    blocks = sum(len(p) for p in pages)
    dtype = torch.float8_e4m3fn if case["cache"] == "fp8" else BF16
    pos = torch.tensor(lens, device=DEV) - 1
    h = ck.f64("model.embed_tokens.weight")[tokens(seed, "ids", B, m["vocab"])]
    for i in range(m["layers"]):
        p = f"model.layers.{i}."
        x = rms(h, ck.f64(p + "input_layernorm.weight"), m["eps"])
        q, k, v = ((x @ ck.f64(p + f"self_attn.{n}_proj.weight").t()).view(B, -1, hd) for n in "qkv")
        q, k = rope(q, pos, m["theta"]), rope(k, pos, m["theta"])
        K, V = cached(seed, i, blocks, G, hd, dtype)
        a = torch.cat([attend(q[b:b + 1], *context(K, V, pages[b], lens[b], k[b], v[b]), hd ** -0.5, False) for b in range(B)])
        h = h + a @ ck.f64(p + "self_attn.o_proj.weight").t()
        x = rms(h, ck.f64(p + "post_attention_layernorm.weight"), m["eps"])
        h = h + swiglu(x, *(ck.f64(p + f"mlp.{n}_proj.weight") for n in ("gate", "up", "down")))
    return [rms(h, ck.f64("model.norm.weight"), m["eps"]) @ ck.f64("lm_head.weight").t(), None]


def context(K, V, pages, n, k_new, v_new, first=0):
    """One sequence's keys and values [n - first, G, d], its newest row in place of what its page holds."""
    at = first // PAGE
    p = pages[at:].long()
    k = K[p].to(F64).transpose(1, 2).reshape(-1, K.shape[1], K.shape[3])[first - at * PAGE:n - at * PAGE]
    v = V[p].to(F64).permute(0, 3, 1, 2).reshape(-1, V.shape[1], V.shape[2])[first - at * PAGE:n - at * PAGE]
    k[-1], v[-1] = k_new, v_new
    return k, v


def exact_hybrid(case, seed):
    m, lens = HYBRID, lengths(case)
    ck, B, H, G, hd, eps = Checkpoint(seed, hybrid_shapes(m)), len(lens), m["H"], m["G"], m["hd"], m["eps"]
    pages = page_tables(seed, lens)
    blocks = sum(len(p) for p in pages)
    pos = torch.tensor(lens, device=DEV) - 1
    # half of each head is rotated; waves longer than the original context are slowed down by 8
    f = 500000.0 ** (-torch.arange(0, hd // 2, 2, device=DEV, dtype=F64) / (hd // 2))
    turns = 8192 * f / (2 * math.pi)
    mix = ((turns - 1.0) / (4.0 - 1.0)).clamp(0, 1)
    f = torch.where(turns < 1.0, f / 8, torch.where(turns > 4.0, f, (1 - mix) * f / 8 + mix * f))
    ang = pos.to(F64)[:, None] * f
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    n = hd // 4

    def turn(x):
        a, b = x[..., :n], x[..., n:2 * n]
        return rms(torch.cat([a * c - b * s, b * c + a * s, x[..., 2 * n:]], -1), 1.0, eps)

    x = ck.f64("embed")[tokens(seed, "ids", B, m["vocab"])]
    for i in range(m["layers"]):
        p, w = f"l{i}.", f"l{i}.mix."
        h = rms(x, 1 + ck.f64(p + "norm1"), eps)
        q, k, v = ((h @ ck.f64(w + t).t() + ck.f64(w + t + ".b")).view(B, -1, hd) for t in "qkv")
        q, k = turn(q), turn(k)
        K, V = cached(seed, i, blocks, G, hd, BF16)
        sink, rows = ck.f64(w + "sink"), []
        for b in range(B):
            kb, vb = context(K, V, pages[b], lens[b], k[b], v[b], max(0, lens[b] - m["window"]))
            sc = torch.einsum("grd,sgd->grs", q[b].view(G, H // G, hd), kb).reshape(H, -1) * hd ** -0.5
            pr = torch.cat([sc, sink[:, None]], -1).softmax(-1)[:, :-1]
            rows.append(torch.einsum("grs,sgd->grd", pr.view(G, H // G, -1), vb).reshape(H, hd))
        a = torch.stack(rows) * torch.sigmoid(h @ ck.f64(w + "g").t())[..., None]
        y = (a.reshape(B, -1) @ ck.f64(w + "o").t() + ck.f64(w + "o.b")) * ck.f64(p + "ls1")
        h = rms(x, 1 + ck.f64(p + "norm2"), eps)
        g, u, d = (ck.f64(p + "mlp." + t) for t in ("gate", "up", "down"))
        x = x + y + ((F.gelu(h @ g.t(), approximate="tanh") * (h @ u.t())) @ d.t()) * ck.f64(p + "ls2")
    return [rms(x, 1 + ck.f64("final.norm"), eps) @ ck.f64("head").t()] + [None] * (2 * m["layers"])


def exact_delta(case, seed):
    """The logits, token by token through the recurrence; the pages and states are not rebuilt."""
    m, lens = DELTA, lengths(case)
    ck, T, D, H, G, hd = Checkpoint(seed, delta_shapes(m)), sum(lens), m["D"], m["H"], m["G"], m["hd"]
    Hk, Hv, d, eps = m["Hk"], m["Hv"], m["d"], m["eps"]
    r = Hv // Hk
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens])
    h = ck.f64("model.embed_tokens.weight")[tokens(seed, "ids", T, m["vocab"])]
    for i in range(m["layers"]):
        p = f"model.layers.{i}."
        x = rms(h, 1 + ck.f64(p + "input_layernorm.weight"), eps)
        if delta_full(m, i):
            a = p + "self_attn."
            qg = (x @ ck.f64(a + "q_proj.weight").t()).view(T, H, 2, hd)
            k, v = ((x @ ck.f64(a + f"{n}_proj.weight").t()).view(T, G, hd) for n in "kv")
            q = rope(rms(qg[:, :, 0], 1 + ck.f64(a + "q_norm.weight"), eps), pos, m["theta"], m["rot"])
            k = rope(rms(k, 1 + ck.f64(a + "k_norm.weight"), eps), pos, m["theta"], m["rot"])
            o = torch.cat([attend(q[s:t], k[s:t], v[s:t], hd ** -0.5, True) for s, t in pieces(lens)])
            h = h + (o * torch.sigmoid(qg[:, :, 1]).reshape(T, -1)) @ ck.f64(a + "o_proj.weight").t()
        else:
            h = h + delta_mixer(x, ck, p + "linear_attn.", m, lens, T, Hk, Hv, d, r, eps)
        x = rms(h, 1 + ck.f64(p + "post_attention_layernorm.weight"), eps)
        h = h + swiglu(x, *(ck.f64(p + f"mlp.{n}_proj.weight") for n in ("gate", "up", "down")))
    h = h[torch.tensor(lens, device=DEV).cumsum(0) - 1]
    return [rms(h, 1 + ck.f64("model.norm.weight"), eps) @ ck.f64("lm_head.weight").t(), None, None, None]


def delta_mixer(x, ck, a, m, lens, T, Hk, Hv, d, r, eps):
    y = (x @ ck.f64(a + "in_proj_qkvz.weight").t()).view(T, Hk, 2 * d + 2 * r * d)
    q, k, v, z = y.split([d, d, r * d, r * d], -1)
    b, al = (x @ ck.f64(a + "in_proj_ba.weight").t()).view(T, Hk, 2 * r).split([r, r], -1)
    mixed = torch.cat([t.reshape(T, -1) for t in (q, k, v)], -1)
    cw = ck.f64(a + "conv1d.weight")
    conv = F.silu(torch.cat([F.conv1d(F.pad(mixed[s:t].t(), (m["conv"] - 1, 0))[None], cw, groups=cw.shape[0])[0].t()
                             for s, t in pieces(lens)]))
    q, k, v = conv.split([Hk * d, Hk * d, Hv * d], -1)
    q, k = (t.reshape(T, Hk, d) * torch.rsqrt(t.reshape(T, Hk, d).square().sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    q, k, v = (q * d ** -0.5).repeat_interleave(r, 1), k.repeat_interleave(r, 1), v.reshape(T, Hv, d)
    beta = torch.sigmoid(b.reshape(T, Hv))
    decay = torch.exp(-torch.exp(ck.f64(a + "A_log")) * F.softplus(al.reshape(T, Hv) + ck.f64(a + "dt_bias")))
    o = torch.empty(T, Hv, d, device=DEV, dtype=F64)
    # all sequences side by side, one token each a step
    starts = [s for s, _ in pieces(lens)]
    order = sorted(range(len(lens)), key=lambda j: -lens[j])
    at = torch.tensor([starts[j] for j in order], device=DEV)
    S = torch.zeros(len(lens), Hv, d, d, device=DEV, dtype=F64)
    for t in range(max(lens)):
        n = sum(lens[j] > t for j in order)
        rows, St = at[:n] + t, S[:n]
        kt = k[rows]
        St.mul_(decay[rows][..., None, None])
        u = (v[rows] - torch.matmul(kt[:, :, None], St)[:, :, 0]) * beta[rows][..., None]
        St.add_(kt[..., None] * u[:, :, None])
        o[rows] = torch.matmul(q[rows][:, :, None], St)[:, :, 0]
    o = rms(o, ck.f64(a + "norm.weight"), eps) * F.silu(z.reshape(T, Hv, d))
    return o.reshape(T, -1) @ ck.f64(a + "out_proj.weight").t()
