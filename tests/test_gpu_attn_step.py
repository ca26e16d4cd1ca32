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


def attention_shown(Hq, Hkv, D, dtype, gain=1.0):
    """A layer that shows its attention: embeddings, MLP and the projections' weights are 0, q, k and v their biases -- q and k in dims that position does not turn (theta 1e30: from a quarter of the
    pairs on no angle reaches 1e-3 of a step, and the bias is 0 in the others) --, o_proj and lm_head identities (o_proj times gain, a
    power of two, by which v's bias is divided): logits = T(norm(T(attention)))."""
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    H = Hq * D
    cfg = {"model_type": "llama", "hidden_size": H, "num_hidden_layers": 1, "intermediate_size": 64, "num_attention_heads": Hq, "num_key_value_heads": Hkv, "head_dim": D, "rms_norm_eps": 1e-5,
           "vocab_size": H, "rope_theta": 1e30, "max_position_embeddings": 2048, "tie_word_embeddings": False, "attention_bias": True}
    w = {n: torch.zeros_like(t) for n, t in synthetic_checkpoint(cfg, seed=1, dtype=dtype).items()}
    g = torch.Generator().manual_seed(Hq * D)
    still = (torch.arange(D) % (D // 2)) >= D // 4
    for n, heads in (("q", Hq), ("k", Hkv), ("v", Hkv)):
        b = torch.randn(heads, D, generator=g) / (gain if n == "v" else 1.0)
        w[f"model.layers.0.self_attn.{n}_proj.bias"] = (b if n == "v" else b * still).reshape(-1).to(dtype).cuda()
    w["model.layers.0.self_attn.o_proj.weight"] = (torch.eye(H) * gain).to(dtype).cuda()
    w["lm_head.weight"] = torch.eye(H, dtype=dtype, device="cuda")
    for n in w:
        if "norm" in n:
            w[n] = torch.ones_like(w[n])
    return Model(ModelArgs(**cfg), w), [w[f"model.layers.0.self_attn.{n}_proj.bias"].double().cpu().view(-1, D) for n in "qkv"]


def check_shown(Hq, Hkv, D, dtype, lens, keys, values, gain=1.0, batch=True, paged=True):
    """The step against float64, from the rows that lie in the cache: attention good to the sums' fp32 (K 2^-24 of the weighted magnitudes, weights to 2^-20 of themselves: their scores are sums of
    D products of up to 8 log2 units and more), and three roundings of eps each: of attention, in the norm and behind it."""
    model, (q, k_new, v_new) = attention_shown(Hq, Hkv, D, dtype, gain)
    pool = model.enable_paged_kv(num_pages=sum(n // 64 + 1 for n in lens) + 1, max_blocks=16) if paged else None
    if paged:
        for slab in pool.slab:
            slab.view(dtype).fill_(torch.nan)
    caches, rows = [model.make_cache() for _ in lens], []
    for i, (n, c) in enumerate(zip(lens, caches)):
        model.step(torch.zeros(n, dtype=torch.int32, device="cuda"), c)
        K, V = keys(i, n, q).to(dtype), values(i, n).to(dtype)   # [Hkv, n, D]
        if paged:
            for p in range(0, n, 64):
                page = pool.slab[0].view(dtype).view(-1, 2, Hkv, 64, D)[c[0].page_manager.pages[p // 64]]
                page[0, :, :min(64, n - p)], page[1, :, :min(64, n - p)] = K[:, p:p + 64].cuda(), V[:, p:p + 64].cuda()
        else:
            c[0].keys[0, :, :n], c[0].values[0, :, :n] = K.cuda(), V.cuda()
        rows.append((torch.cat([K.double(), k_new[:, None]], 1), torch.cat([V.double(), v_new[:, None]], 1)))
    feed = torch.zeros(len(lens), dtype=torch.int32, device="cuda")
    if batch:
        got = model.step_batch(feed, caches, graph=False)[2].double().cpu()
    else:
        got = torch.stack([model.step(feed[i:i + 1], c)[2].double().cpu().reshape(-1) for i, c in enumerate(caches)])
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for i, (K, V) in enumerate(rows):
        K, V = K.repeat_interleave(Hq // Hkv, 0), V.repeat_interleave(Hq // Hkv, 0)
        p = torch.softmax((K @ q[:, :, None]).squeeze(-1) * D ** -0.5, -1)
        x = (p[:, None] @ V).reshape(-1) * gain
        noise = ((p[:, None] @ V.abs()).reshape(-1) * abs(gain)) * (2.0 ** -20 + V.shape[1] * 2.0 ** -24)
        norm = (x.square().mean() + 1e-5).rsqrt()
        bound = (x.abs() * 3.1 * eps + noise + noise.square().mean().sqrt() * x.abs() * norm) * norm
        assert torch.isfinite(got[i]).all(), lens[i]
        assert ((got[i] - x * norm).abs() <= bound).all(), (lens[i], float(((got[i] - x * norm).abs() / bound).max()))


SHOWN = [1, 15, 31, 47, 63, 64, 100, 129, 191, 300, 415, 513]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("Hq,Hkv,D", [(8, 8, 64), (6, 2, 64), (8, 1, 64), (4, 4, 128), (4, 2, 128), (6, 2, 128), (5, 1, 128), (8, 1, 128), (8, 2, 128)])
@pytest.mark.parametrize("how", ["batch", "paged", "alone"])
def test_the_attention_of_a_step_against_float64(how, Hq, Hkv, D, dtype):
    """Random keys (scores of a few units, maxima that rise again and again) and values: batches with one long row, one sequence on pages and in its own buffers."""
    g = torch.Generator().manual_seed(D)
    draw = lambda i, n, *_: torch.randn(Hkv, n, D, generator=g) * 2
    lens = SHOWN + [900] if how != "batch" else SHOWN + [1000]
    check_shown(Hq, Hkv, D, dtype, lens, draw, draw, batch=how == "batch", paged=how != "alone")


@pytest.mark.parametrize("power", [118, -124])
@pytest.mark.parametrize("Hq,Hkv,D", [(6, 2, 64), (4, 4, 128), (8, 2, 128)])
@pytest.mark.parametrize("how", ["batch", "paged", "alone"])
def test_values_near_the_limits_of_bf16(how, Hq, Hkv, D, power):
    """Weights that rise by seven powers of two over the row and values of 2^118 or 2^-124: a value times the row's length at most is what the sums have to hold, and nothing more."""
    def keys(i, n, q):   # (the scores of a group's first query; the others lean on its direction more or less)
        u = q.view(Hkv, Hq // Hkv, D)[:, 0]
        return (u / u.square().sum(-1, keepdim=True))[:, None] * (torch.arange(n)[None, :, None] / n * 5) * D ** 0.5

    g = torch.Generator().manual_seed(D)
    values = lambda i, n: (1 + torch.rand(Hkv, n, D, generator=g)) * 2.0 ** power
    check_shown(Hq, Hkv, D, torch.bfloat16, SHOWN[5:], keys, values, gain=2.0 ** -power, batch=how == "batch", paged=how != "alone")


def test_a_batch_of_many_rows_against_float64():
    """More rows than one workgroup's threads sum at a time, idle of pieces beside one row that is in several."""
    g = torch.Generator().manual_seed(7)
    draw = lambda i, n, *_: torch.randn(1, n, 64, generator=g)
    check_shown(2, 1, 64, torch.bfloat16, [5 + i % 40 for i in range(700)] + [1000], draw, draw)
