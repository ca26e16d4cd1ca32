"""k_attn_step at the edges of its blocks of 16 positions, of its rounds of four waves (64) and of its splits; more than 64 blocks of a
wave, so that a wave's page numbers come in two parts; scores that rise again and again.  The reference is each
sequence served alone, or its prompt with the token behind it."""
import numpy as np
import pytest
import torch

from tests._util import assert_vec_close
from tests.test_gpu_batch_attention import _model

pytestmark = pytest.mark.gpu


def both(model, lens, max_blocks, graph=False):
    rng = np.random.default_rng(len(lens))
    prompts = [rng.integers(0, 512, n).astype(np.int32) for n in lens]
    model.enable_paged_kv(num_pages=sum(n // 64 + 1 for n in lens) + 1, max_blocks=max_blocks)
    feed, out = torch.arange(3, 3 + len(lens), dtype=torch.int32, device="cuda"), []
    for batch in (False, True):
        caches = [model.make_cache() for _ in lens]
        for p, c in zip(prompts, caches):
            model.step(torch.from_numpy(p).cuda(), c)
        out.append(model.step_batch(feed, caches, graph=graph)[2].float().cpu().numpy() if batch
                   else np.stack([model.step(feed[i:i + 1], c)[2].float().cpu().numpy().reshape(-1) for i, c in enumerate(caches)]))
        for c in caches:
            c[0].page_manager.release()
    return out


@pytest.mark.parametrize("Hq,Hkv,rows", [(1, 1, 12), (2, 1, 40), (6, 2, 9), (16, 4, 72), (16, 4, 20)])
def test_blocks_rounds_and_pieces(Hq, Hkv, rows):
    """Rows in one piece and in up to four (of 64 positions and more); lengths (the new position included) one off 16, 32, 64, 128 and beside them."""
    lens = [(14, 15, 16, 30, 31, 32, 47, 62, 63, 64, 79, 126, 127, 128, 129, 200, 255, 256, 300)[i % 19] for i in range(rows)]
    model = _model(128 * Hq, Hq, Hkv, 128, False, True, False)
    for max_blocks in (5, 12):
        alone, batched = both(model, lens, max_blocks)
        for i, n in enumerate(lens):
            assert_vec_close(batched[i], alone[i], "bfloat16", what=f"row {i}, {n} positions cached, tables of {max_blocks}")


@pytest.mark.parametrize("long,rows,kv_heads", [(4300, 43, 4), (17000, 32, 4), (1500, 6, 1)])
def test_a_long_sequence_among_short_ones(long, rows, kv_heads):
    """In four pieces (of 17000 positions: 67 blocks of a wave) and in seventeen, beside rows in one."""
    lens = [20 + i for i in range(rows - 1)]
    lens.insert(3, long)
    alone, batched = both(_model(512, 4, kv_heads, 128, False, True, False), lens, long // 64 + 1)
    for i, n in enumerate(lens):
        assert_vec_close(batched[i], alone[i], "bfloat16", what=f"row {i}, {n} positions cached")


def test_replays_of_a_captured_step_merge_anew():
    """The counters are zero again behind every launch: the captured step, replayed while rows cross from one piece to two, against the launches."""
    model = _model(512, 4, 4, 128, False, True, False)
    lens = [60, 61, 62, 63, 250, 251, 500]
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, 512, n).astype(np.int32) for n in lens]
    model.enable_paged_kv(num_pages=2 * sum(n // 64 + 2 for n in lens), max_blocks=10)
    feed, runs = torch.arange(3, 3 + len(lens), dtype=torch.int32, device="cuda"), []
    for graph in (True, False):
        caches = [model.make_cache() for _ in lens]
        model.prefill_batch(prompts, caches)
        runs.append([model.step_batch(feed, caches, graph=graph)[2].clone() for _ in range(8)])
        for c in caches:
            c[0].page_manager.release()
    for a, b in zip(*runs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("rep", [1, 2, 3, 4, 5, 6, 7, 8])
def test_a_step_is_the_prompt_with_its_token(rep, D, dtype):
    """One sequence in its own buffers and on pages (bit for bit the same), and a batch, against prompts that end with the token: prompt attention has its own kernel.  Both sides round: each within
    four ulps of the largest logit of what unrounded layers give (assert_vec_close's bound), the two within eight."""
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    Hkv = 2
    cfg = {"model_type": "llama", "hidden_size": 256, "num_hidden_layers": 2, "intermediate_size": 256, "num_attention_heads": rep * Hkv, "num_key_value_heads": Hkv, "head_dim": D, "vocab_size": 512,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "max_position_embeddings": 2048}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=rep, dtype=getattr(torch, dtype)))
    rng = np.random.default_rng(rep)
    lens = [6, 15, 16, 33, 64, 65, 129, 500]
    prompts = [torch.from_numpy(rng.integers(0, 512, n + 1).astype(np.int32)).cuda() for n in lens]
    want, alone = [], []
    for p in prompts:
        cache = m.make_cache()
        want.append(m.step(p, cache)[2].float().cpu().numpy().reshape(-1))
        cache = m.make_cache()
        m.step(p[:-1], cache)
        alone.append(m.step(p[-1:], cache)[2].clone().reshape(-1))
    m.enable_paged_kv(num_pages=sum(n // 64 + 1 for n in lens), max_blocks=8)
    caches = [m.make_cache() for _ in lens]
    for p, c, a in zip(prompts, caches, alone):
        m.step(p[:-1], c)
        assert torch.equal(m.step(p[-1:], c)[2].reshape(-1), a)
        for layer in c:
            layer.trim(1)
    batch = m.step_batch(torch.stack([p[-1] for p in prompts]), caches, graph=False)[2]
    for i, n in enumerate(lens):
        assert_vec_close(alone[i].float().cpu().numpy(), want[i], dtype, c_max=8.0, c_rms=8.0, what=f"alone, {n} positions")
        assert_vec_close(batch[i].float().cpu().numpy(), want[i], dtype, c_max=8.0, c_rms=8.0, what=f"batch, {n} positions")


def bits_over_pools(model, lens, max_blocks, run):
    """What `run(caches, feed)` gives behind prompts of these lengths, with a pool full of zeros, of NaN and of infinities."""
    prompts = [torch.from_numpy(np.random.default_rng(i).integers(0, 512, n).astype(np.int32)).cuda() for i, n in enumerate(lens)]
    pool = model.enable_paged_kv(num_pages=sum(n // 64 + 1 for n in lens) + 1, max_blocks=max_blocks)
    feed, got = torch.arange(3, 3 + len(lens), dtype=torch.int32, device="cuda"), []
    for fill in (0.0, float("nan"), float("inf")):
        for slab in pool.slab:
            slab.view(torch.bfloat16).fill_(fill)
        caches = [model.make_cache() for _ in lens]
        for p, c in zip(prompts, caches):
            model.step(p, c)
        got.append(run(caches, feed))
        for c in caches:
            c[0].page_manager.release()
    return got


@pytest.mark.parametrize("Hq,Hkv,D", [(24, 8, 128), (4, 4, 128), (8, 1, 128), (32, 4, 64), (8, 2, 64), (5, 5, 64)])
def test_a_paged_sequence_reads_no_row_that_nobody_wrote(Hq, Hkv, D):
    """Splits of a multiple of 16 positions that end on another page than some wave's last block: what lies behind the sequence in the pool counts nothing, not even with weight 0.  The new
    position included, 129 .. 145 and some up to the 1024 where the consumer merges the splits."""
    model = _model(512, Hq, Hkv, D, False, False, False)
    lens = [*range(128, 145), 149, 159, 192, 199, 256, 299, 399, 449, 640, 830, 1000]
    got = bits_over_pools(model, lens, 16, lambda caches, feed: torch.stack([model.step(feed[i:i + 1], c)[2].clone().reshape(-1) for i, c in enumerate(caches)]))
    assert torch.isfinite(got[0]).all()
    for g in got[1:]:
        assert [lens[i] for i in range(len(lens)) if not torch.equal(g[i], got[0][i])] == []


@pytest.mark.parametrize("Hq,Hkv,D", [(8, 8, 128), (24, 8, 128), (16, 8, 64)])
@pytest.mark.parametrize("short", [4, 7])
def test_a_batch_reads_no_row_that_nobody_wrote(short, Hq, Hkv, D):
    """One row in pieces beside rows in one: pieces that end on another page than some wave's last block, in front of a last piece that is short."""
    model = _model(512, Hq, Hkv, D, False, False, False)
    for n in (*range(400, 417, 3), 415, *range(672, 689, 4)):
        lens = [40] * short
        lens.insert(2, n)
        got = bits_over_pools(model, lens, 12, lambda caches, feed: model.step_batch(feed, caches, graph=False)[2].clone())
        assert torch.isfinite(got[0]).all()
        assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2]), n
