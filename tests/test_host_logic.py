"""CPU: host-side mirrors of the reference's cache / prompt-cache / sampler logic behave like the oracle's
restatement (and therefore like cache/kv_cache/reusable.py, cache/prompt_cache.py, samplers/__init__.py)."""
import numpy as np
import pytest
import torch

from oracle import pie_oracle as po
from proxy_inference_engine_amd.cache import PromptCache, ReusableKVCache
from proxy_inference_engine_amd.logits_processors import make_repetition_penalty
from proxy_inference_engine_amd.models.base import create_attention_mask, create_causal_mask
from proxy_inference_engine_amd.models.llama import ModelArgs
from proxy_inference_engine_amd.samplers import make_sampler


def test_reusable_cache_capacity_sequence_matches_oracle():
    ref, mine = po.OracleKVCache(), ReusableKVCache()
    k = np.ones((1, 2, 128, 8), np.float32)
    ref.update_and_fetch(k, k)
    mine.update_and_fetch(torch.ones(1, 2, 128, 8), torch.ones(1, 2, 128, 8))
    one = torch.full((1, 2, 1, 8), 2.0)
    for _ in range(1100):
        ref.update_and_fetch(one.numpy(), one.numpy())
        kk, vv = mine.update_and_fetch(one, one)
        assert (mine.offset, mine.capacity) == (ref.offset, ref.keys.shape[2])
    assert kk.shape[2] == mine.offset and np.array_equal(mine.keys.numpy(), ref.keys)
    assert mine.trim(28) == 28 and mine.offset == 1200 and mine.is_trimmable() and mine.to_quantized() is mine
    # reserve()/advance() = the two halves of update_and_fetch used by the fused decoder
    c = ReusableKVCache()
    c.reserve(300, 2, 8, torch.float32, "cpu")
    assert c.capacity == 512 and c.offset == 0
    c.advance(300)
    c.reserve(300, 2, 8, torch.float32, "cpu")
    assert c.capacity == 768
    capped = ReusableKVCache(max_capacity=256)
    capped.reserve(200, 1, 8, torch.float32, "cpu")
    capped.advance(200)
    with pytest.raises(RuntimeError):
        capped.reserve(100, 1, 8, torch.float32, "cpu")


@pytest.mark.parametrize("chunks", [(520, 300), (700, 400), (255, 2, 300), (256, 300), (100, 1, 1, 700, 5, 900)])
def test_reusable_cache_growth_at_unaligned_offsets_matches_oracle(chunks):
    """reusable.py:125-129: growing at an offset that is not a multiple of `step` first slices the buffers to the offset, so the
    new capacity is computed from the offset (520 then 300 tokens -> 1024, not 1280).  Both halves of the product's API."""
    ref, mine, split = po.OracleKVCache(), ReusableKVCache(), ReusableKVCache()
    for n in chunks:
        ref.update_and_fetch(np.ones((1, 2, n, 8), np.float32), np.ones((1, 2, n, 8), np.float32))
        mine.update_and_fetch(torch.ones(1, 2, n, 8), torch.ones(1, 2, n, 8))
        split.reserve(n, 2, 8, torch.float32, "cpu")
        split.advance(n)
        assert (mine.offset, mine.capacity) == (ref.offset, ref.keys.shape[2])
        assert (split.offset, split.capacity) == (ref.offset, ref.keys.shape[2])
    if chunks == (520, 300):
        assert mine.capacity == 1024


def test_prompt_cache_history_is_cut_on_reuse():
    """A -> B -> A: after B diverged at k the caches hold B beyond k; the history must say so (deviation from
    prompt_cache.py:52-76, which keeps A + B[k:] and would let the third request reuse B's rows as A's)."""
    pc = PromptCache()
    pc.cache = [ReusableKVCache()]
    A, B = list(range(100, 140)), list(range(100, 120)) + list(range(500, 530))
    one = lambda n: torch.ones(1, 1, n, 8)

    def request(ids):
        todo = pc(torch.tensor(ids))
        pc.cache[0].update_and_fetch(one(len(todo)), one(len(todo)))
        pc.update(todo)
        return len(todo)

    assert request(A) == 40 and pc.computed_ids == A
    assert request(B) == 30 and pc.computed_ids == B and pc.cache[0].offset == 50
    assert request(A) == 20 and pc.computed_ids == A and pc.cache[0].offset == 40      # the reference would process 1 token here


def test_prompt_cache_lcp_matches_oracle():
    ref, mine = po.OraclePromptCache(), PromptCache()
    ref.cache, mine.cache = [po.OracleKVCache()], [ReusableKVCache()]
    k = np.ones((1, 2, 128, 8), np.float32)
    ref.cache[0].update_and_fetch(k, k)
    mine.cache[0].update_and_fetch(torch.ones(1, 2, 128, 8), torch.ones(1, 2, 128, 8))
    ref.update(np.arange(128)); mine.update(torch.arange(128))
    for prompt in (np.arange(128), np.concatenate([np.arange(50), np.arange(900, 1200)]), np.array([999, 1, 2]), np.arange(3)):
        a, b = ref(prompt), mine(torch.from_numpy(prompt))
        assert list(a) == list(b.tolist())
        assert (mine.cache[0].offset, mine.cache[0].capacity) == (ref.cache[0].offset, ref.cache[0].keys.shape[2])
    assert PromptCache()(torch.arange(5)).tolist() == [0, 1, 2, 3, 4]     # nothing cached yet


def test_sampler_and_processor_conventions():
    assert not getattr(make_sampler(temp=0.7, top_p=0.9), "is_greedy", False)
    assert getattr(make_sampler(temp=0), "is_greedy", False)
    with pytest.raises(ValueError):
        make_repetition_penalty(-1.0)
    proc = make_repetition_penalty(2.0, context_size=3)
    logits = torch.tensor([[1.0, -1.0, 4.0, -4.0, 8.0]])
    out = proc([4, 0, 1, 2, 3], logits.clone())                         # only the last 3 tokens count
    assert out.tolist() == [[1.0, -2.0, 2.0, -8.0, 8.0]]


def test_masks_and_model_args():
    m = create_causal_mask(3, offset=2)
    assert m.shape == (3, 5) and m[0].tolist() == [0, 0, 0, -1e9, -1e9] and m[2].tolist() == [0, 0, 0, 0, 0]
    assert np.array_equal(m.numpy().astype(np.float32), po.causal_mask(3, 2, "float32"))
    assert create_attention_mask(torch.zeros(1, 1, 8)) is None          # L == 1: no mask (models/base.py:39-53)
    a = ModelArgs(model_type="llama", hidden_size=64, num_hidden_layers=1, intermediate_size=128, num_attention_heads=2,
                  rms_norm_eps=1e-5, vocab_size=10, some_unknown_key=1)
    assert a.tie_word_embeddings is True and a.rope_theta == 10000 and not hasattr(a, "some_unknown_key")


def _ref_sets(logprobs, temp, top_p=0.0, min_p=0.0, keep=1, top_k=-1):
    """Numpy restatement of which vocabulary ids the reference's filters leave drawable (samplers/{top_p,min_p,top_k}.py)."""
    x = logprobs.astype(np.float64) / temp
    if 0 < top_p < 1.0:
        p = np.exp(x - x.max()); p /= p.sum()
        order = np.argsort(p, kind="stable")
        cum = np.cumsum(p[order].astype(np.float32))
        return set(order[cum > np.float32(1 - top_p)].tolist())
    if min_p != 0.0:
        order = np.argsort(-x, kind="stable")
        kept = x[order] >= x[order][0] + np.log(min_p)
        kept[:keep] = True
        return set(order[kept].tolist())
    if top_k > 0:
        return set(np.argsort(-x, kind="stable")[:top_k].tolist())
    return set(range(len(x)))


@pytest.mark.parametrize("kw", [dict(top_p=0.6), dict(top_p=0.95), dict(min_p=0.1), dict(min_p=0.3, min_tokens_to_keep=4),
                                dict(top_k=5), dict()])
def test_sampler_reference_keep_sets_and_distribution(kw):
    """tests/sampler_reference.py (the reference's samplers/*.py restated with torch ops, the comparator of the HIP kernels): every draw lies
    in the set the reference's filter keeps (numpy restatement above), every kept token with non-negligible mass is drawn, and the empirical
    frequencies follow the renormalised probabilities (total variation < 0.05 over 4000 draws)."""
    from tests import sampler_reference as sr
    rng = np.random.default_rng(11)
    V, temp = 64, 0.8
    logits = rng.standard_normal(V).astype(np.float32) * 2.0
    logprobs = logits - np.log(np.exp(logits.astype(np.float64)).sum()).astype(np.float32)
    sampler = sr.make_sampler(temp=temp, **kw)
    sr.seed(1234)
    x = torch.from_numpy(logprobs)[None].repeat(4000, 1)                # 4000 independent rows, one call
    draws = sampler(x).numpy()
    assert draws.shape == (4000,) and draws.dtype == np.int32
    allowed = _ref_sets(logprobs, temp, kw.get("top_p", 0.0), kw.get("min_p", 0.0), kw.get("min_tokens_to_keep", 1), kw.get("top_k", -1))
    assert set(draws.tolist()) <= allowed
    p = np.exp(logprobs.astype(np.float64) / temp)
    mask = np.zeros(V, bool); mask[list(allowed)] = True
    p = np.where(mask, p, 0.0); p /= p.sum()
    freq = np.bincount(draws, minlength=V) / 4000.0
    assert 0.5 * np.abs(freq - p).sum() < 0.05
    assert all(freq[i] > 0 for i in allowed if p[i] > 0.01)
    sr.seed(1234)
    assert np.array_equal(sampler(x).numpy(), draws)                   # seed() restarts the stream


def test_stochastic_sampler_argument_errors_and_no_host_path():
    x = torch.zeros((1, 16))
    with pytest.raises(ValueError):
        make_sampler(temp=1.0, top_k=16)(x)                             # top_k must be < vocab (top_k.py:20-24)
    with pytest.raises(ValueError):
        make_sampler(temp=1.0, min_p=1.5)(x)                            # min_p.py:33-36
    with pytest.raises(ValueError):
        make_sampler(temp=1.0, min_p=0.1, min_tokens_to_keep=0)(x)      # min_p.py:37-40
    # the product has no CPU path: a host tensor is refused by every stochastic branch, not sampled by torch
    for kw in (dict(top_p=0.6), dict(min_p=0.1), dict(top_k=5), dict()):
        with pytest.raises(ValueError, match="device tensors"):
            make_sampler(temp=1.0, **kw)(x)


def test_prompt_cache_persistence_round_trip(tmp_path):
    """cache_prompt / load_cached_prompt (prompt_cache.py:78-125) through BaseCache.save_cache / load_cache
    (kv_cache/__init__.py:163-210): file named by sha256 of the id list, arrays "<layer>.<0|1>", metadata
    "0.<i>" / "1.computed_ids" / "2.<i>"; a request with the same ids then re-processes exactly one token."""
    from safetensors import safe_open
    pc = PromptCache(directory=tmp_path, cache=[ReusableKVCache() for _ in range(3)])
    ids = list(range(40, 50))
    for i, c in enumerate(pc.cache):
        c.update_and_fetch(torch.full((1, 2, 10, 8), float(i + 1)), torch.full((1, 2, 10, 8), -float(i + 1)))
    pc.update(ids)
    pc.cache_prompt()
    files = list(tmp_path.glob("*.safetensors"))
    assert len(files) == 1 and files[0].stem == PromptCache._compute_prompt_hash(ids)
    with safe_open(str(files[0]), framework="pt") as f:
        assert sorted(f.keys()) == ["0.0", "0.1", "1.0", "1.1", "2.0", "2.1"]
        assert f.metadata()["1.computed_ids"] == str(ids).replace("'", "") and f.metadata()["2.1"] == "ReusableKVCache"
    fresh = PromptCache(directory=tmp_path)
    fresh.load_cached_prompt(list(range(7)))                            # no such file: nothing happens
    assert fresh.cache == [] and fresh.computed_ids == []
    fresh.load_cached_prompt(ids)
    assert fresh.computed_ids == ids and len(fresh.cache) == 3
    assert fresh.cache[2].offset == 256                                 # the reference quirk: offset = saved capacity ...
    assert torch.equal(fresh.cache[1].keys.cpu(), pc.cache[1].keys.cpu()) and float(fresh.cache[2].values[0, 0, 9, 0]) == -3.0
    todo = fresh(ids)                                                   # ... until the prefix match trims it
    assert list(todo) == ids[-1:] and fresh.cache[0].offset == 9


def test_reference_import_paths_resolve_to_the_same_modules():
    """Code written against the reference imports `proxy_inference_engine.<module>` (src/proxy_inference_engine/...): every
    such path must give the very module object of the implementation (shared sampler RNG state, one loaded library)."""
    import importlib
    for m in ("engine.inference_engine", "samplers", "samplers.top_p", "samplers.min_p", "samplers.top_k", "samplers.categorical",
              "cache", "cache.prompt_cache", "cache.kv_cache", "cache.kv_cache.reusable", "logits_processors",
              "logits_processors.repetition", "models", "models.base", "models.utils", "models.llama", "models.llama.language",
              "models.llama.utils", "pie_core"):
        assert importlib.import_module(f"proxy_inference_engine.{m}") is importlib.import_module(f"proxy_inference_engine_amd.{m}"), m
    from proxy_inference_engine import InferenceEngine, pie_core
    from proxy_inference_engine.engine.inference_engine import InferenceEngine as IE2
    assert InferenceEngine is IE2 and pie_core.hello() == "pie_core \u2713"
    with pytest.raises(ImportError):
        importlib.import_module("proxy_inference_engine.server")       # the HTTP server is out of scope: absent, not stubbed


def test_oracle_forward_from_input_embeddings_equals_forward_from_ids():
    """`h = inputs_embeds` (models/intern/language.py:155-158): feeding the oracle the embedding rows of the ids must give
    exactly the logits of feeding the ids."""
    cfg = {"model_type": "llama", "hidden_size": 128, "num_hidden_layers": 2, "intermediate_size": 256, "num_attention_heads": 4,
           "num_key_value_heads": 2, "rms_norm_eps": 1e-5, "vocab_size": 320, "rope_theta": 10000.0, "tie_word_embeddings": True,
           "quantization": {"group_size": 64, "bits": 4}}
    w = po.synth_checkpoint(cfg, seed=2, dtype="bfloat16")
    orc = po.OracleLlama(cfg, w, "bfloat16")
    ids = np.random.default_rng(0).integers(0, 320, 9)
    a = orc.forward(ids, [po.OracleKVCache() for _ in orc.layers])
    rows = po.dequantize(w["model.embed_tokens.weight"], w["model.embed_tokens.scales"], w["model.embed_tokens.biases"], dtype="bfloat16")[ids]
    b = orc.forward(None, [po.OracleKVCache() for _ in orc.layers], inputs_embeds=rows)
    assert np.array_equal(a, b)


def test_generate_step_mask_arrays_that_the_reference_loop_can_carry():
    """generate_step forwards ONE mask array to the prompt pass and to every single-token step (inference_engine.py:246-249): only arrays that are
    constant per head broadcast against every [1, H, L, S]; those cannot hide a key, so they are accepted (and change nothing); the rest is
    refused with the reason."""
    from proxy_inference_engine_amd.engine.inference_engine import check_generate_mask
    for ok in (torch.zeros(()), torch.zeros(1, 1), torch.full((1, 1, 1, 1), -3.5), torch.ones(1, 4, 1, 1, dtype=torch.bool), torch.zeros(4, 1, 1), np.zeros((1, 1), np.float32)):
        check_generate_mask(ok, 4)
    for bad, why in ((torch.zeros(12, 12), "broadcast"), (torch.zeros(1, 1, 1, 9), "broadcast"), (torch.zeros(2, 1, 1, 1), "broadcast"),
                     (torch.zeros(1, 3, 1, 1), "broadcast"), (torch.zeros(1, 1, dtype=torch.bool), "hides every key"),
                     (torch.full((1, 1), float("-inf")), "hides every key")):
        with pytest.raises(ValueError, match=why):
            check_generate_mask(bad, 4)


@pytest.mark.parametrize("tokens", [1, 256, 257])
def test_first_buffers_of_all_layers_are_slices_of_one(tokens):
    """reserve_layers gives every layer what reserve gives it: zeros of the same capacity, each its own rows; layers that already hold something, and growth, go one by one."""
    from proxy_inference_engine_amd.cache.kv_cache import reserve_layers
    caches, want = [ReusableKVCache() for _ in range(3)], ReusableKVCache()
    reserve_layers(caches, tokens, 2, 8, torch.float32, "cpu")
    want.reserve(tokens, 2, 8, torch.float32, "cpu")
    for i, c in enumerate(caches):
        assert c.keys.shape == c.values.shape == want.keys.shape and c.offset == 0 and c.keys.is_contiguous() and c.values.is_contiguous() and not c.keys.any() and not c.values.any()
        c.update_and_fetch(torch.full((1, 2, tokens, 8), 2.0 * i + 1), torch.full((1, 2, tokens, 8), 2.0 * i + 2))
    for i, c in enumerate(caches):
        assert (c.keys[:, :, :tokens] == 2 * i + 1).all() and (c.values[:, :, :tokens] == 2 * i + 2).all() and not c.keys[:, :, tokens:].any()
    held = caches[0].keys
    mixed = [caches[0], ReusableKVCache(max_capacity=300)]
    reserve_layers(mixed, 1, 2, 8, torch.float32, "cpu")
    assert mixed[0].keys.shape[2] >= tokens + 1 and (mixed[0].keys is held) == (tokens % 256 != 0) and mixed[1].keys.shape[2] == 256
    with pytest.raises(RuntimeError):
        reserve_layers([ReusableKVCache(max_capacity=300) for _ in range(2)], 301, 2, 8, torch.float32, "cpu")


@pytest.mark.parametrize("dim,storages", [(8, 1), (256, 2), (512, 3), (1024, 10)])
def test_shared_buffers_of_layers_are_small(dim, storages):
    """What outlives a layer that has grown, until its neighbours have: at most 64 MiB, whatever the model's cache takes (layers of 16 MiB by
    four, of 32 MiB by two, of 64 MiB and more by themselves, keys and values apart)."""
    from proxy_inference_engine_amd.cache.kv_cache import reserve_layers
    caches = [ReusableKVCache() for _ in range(5)]
    reserve_layers(caches, 4000, 2, dim, torch.float32, "cpu")   # 4096 positions
    held = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() for c in caches for t in (c.keys, c.values)}
    own = caches[0].keys.nbytes
    assert len(held) == storages and all(n <= max(64 << 20, own) for n in held.values())
    assert sum(held.values()) == 10 * own and all(c.keys.shape == c.values.shape == (1, 2, 4096, dim) for c in caches)
