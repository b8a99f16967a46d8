"""The last layer's projections run over the sampled rows only: their logits are those of a step that scores every row, the caches
are the same to the bit, and a step that samples no row returns none."""
import pytest
import torch

from generativeaiexamples_amd import ops
from generativeaiexamples_amd.engine.kv_cache import KVCache
from generativeaiexamples_amd.models import LlamaConfig, LlamaModel
from generativeaiexamples_amd.models.common import ForwardBatch
from generativeaiexamples_amd.models.mixtral import MixtralConfig, MixtralModel
from generativeaiexamples_amd.models.qwen3_next import Qwen3NextConfig, Qwen3NextModel

FAMILIES = [(LlamaConfig.tiny, LlamaModel), (MixtralConfig.tiny_moe, MixtralModel), (Qwen3NextConfig.tiny, Qwen3NextModel)]


def batch(m, lens, dev):
    T, hq, hkv = sum(lens), m.cfg.num_heads, m.cfg.num_kv_heads
    pages = [-(-n // ops.BLOCK) for n in lens]
    table = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = torch.arange(at, at + n)
        at += n
    pos = torch.cat([torch.arange(n) for n in lens])
    slots = torch.cat([table[b, torch.arange(n) // ops.BLOCK] * ops.BLOCK + torch.arange(n) % ops.BLOCK for b, n in enumerate(lens)])
    i32 = dict(dtype=torch.int32, device=dev)
    return ForwardBatch(token_ids=torch.randint(3, 200, (T,), generator=torch.Generator().manual_seed(T)).to(**i32), positions=pos.to(**i32),
                        slots=slots.to(**i32), num_prefill_tokens=T, cu_q=torch.tensor([0] + lens).cumsum(0).to(**i32),
                        prefill_ctx=torch.tensor(lens, **i32), prefill_block_tables=table.to(dev),
                        prefill_tiles=ops.build_prefill_tiles(lens, hq, hkv, dev, head_dim=m.cfg.head_dim) if dev != "cpu" else None,
                        prefill_qlen=lens, prefill_ctx_host=list(lens), seq_ids=list(range(1, len(lens) + 1)), sample_rows=None), at


def check(config, Model, lens, dev, tol):
    m = Model(config(), device=dev).random_init(3)
    fb, pages = batch(m, lens, dev)
    outs = []
    rows = torch.tensor([sum(lens) - 1, 2], device=dev)
    for r in (None, rows, rows[:0]):
        kv = KVCache(getattr(m, "num_kv_layers", m.cfg.num_layers), pages + 1, m.cfg.num_kv_heads, m.cfg.head_dim, m.device, m.dtype)
        fb.sample_rows = r
        with torch.inference_mode():
            if hasattr(m, "prepare_batch"):
                m.prepare_batch(fb)
            outs.append((m.forward(fb, kv).float().cpu(), kv.storage.float().cpu()))
    (full, kv), (few, kv1), (none, kv2) = outs
    assert few.shape[0] == 2 and none.shape[0] == 0 and torch.equal(kv, kv1) and torch.equal(kv, kv2)
    want = full[rows.cpu()]
    assert (few - want).norm() <= tol * want.norm()


@pytest.mark.parametrize("config,Model", FAMILIES)
def test_sampled_rows_cpu(config, Model):
    # the same bf16 operations over fewer rows: sums of products may be split otherwise (2^-8 a rounding, a handful of them in a row)
    check(config, Model, [19, 7], "cpu", 2.0 ** -6)


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[19, 7], [70, 41], [300, 211]])
@pytest.mark.parametrize("config,Model", FAMILIES)
def test_sampled_rows_gpu(cuda, config, Model, lens):
    check(config, Model, lens, "cuda", 2.0 ** -6)
