"""Int8 models' steps of several sequences on the codes themselves (k_w4a_gemm, W8M tiles): fewer groups of K than waves, groups that are no multiple of eight, splits of K, every count of half strips per
workgroup, a last workgroup that is not full, eight, sixteen and 32 rows and the 33 that go another way, biases."""
import numpy as np
import pytest
import torch

from _util import assert_vec_close

pytestmark = pytest.mark.gpu


# [N, K] in half strips of 16 and groups of 64: hidden 192: 3 groups; 1088: 17, q|k|v in one, vocab in two; 2048: gate|up in three, vocab in five, o_proj and down split; 512: gate|up in seven, vocab
# in eight, in 268 workgroups; 3136: q|k|v, o_proj and gate|up in one, seven steps a wave, down two
@pytest.mark.parametrize("hidden,inter,vocab,heads,kv,dim,bias", [(192, 448, 96, 4, 2, 64, True), (1088, 1472, 5216, 17, 17, 64, False), (2048, 5632, 16896, 16, 4, 128, True), (512, 14336, 34240, 8, 2, 64, False),
                                                                  (3136, 1024, 96, 49, 7, 64, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_rows_against_single_sequences(hidden, inter, vocab, heads, kv, dim, bias, dtype):
    """One layer, every sequence's step alone (the GEMV: fp32 sums of unrounded weights, one rounding) as the reference: four ulps of the largest logit, rms four ulps, as everywhere; 33 rows multiply
    weights that are rounded first, one more ulp in each of the layer's four products and the head."""
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": hidden, "num_hidden_layers": 1, "intermediate_size": inter, "num_attention_heads": heads, "num_key_value_heads": kv, "head_dim": dim,
           "vocab_size": vocab, "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "attention_bias": bias, "mlp_bias": bias, "quantization": {"group_size": 64, "bits": 8}}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=2, dtype=dtype))
    m.enable_paged_kv(num_pages=40, max_blocks=1)
    name = "bfloat16" if dtype == torch.bfloat16 else "float16"
    ids = np.random.default_rng(3).integers(0, vocab, 33).astype(np.int32)
    feed, want = torch.from_numpy(ids).cuda(), []
    for i in range(33):
        c = m.make_cache()
        want.append(m.step(feed[i:i + 1], c)[2].float().cpu().numpy().reshape(-1))
        c[0].page_manager.release()
    for B in (2, 3, 8, 9, 16, 17, 32, 33):
        caches = [m.make_cache() for _ in range(B)]
        got = m.step_batch(feed[:B], caches, graph=False)[2].float().cpu().numpy()
        for i in range(B):
            assert_vec_close(got[i], want[i], name, what=f"B {B} row {i}", **({"c_max": 9.0, "c_rms": 9.0} if B == 33 else {}))
        for c in caches:
            c[0].page_manager.release()
    # a prompt: rotated and appended by the product where q|k|v is not split
    c, p = m.make_cache(), m.make_cache()
    for i in range(12):
        last = m.step(feed[i:i + 1], c)[2].float().cpu().numpy().reshape(-1)
    assert_vec_close(m.step(feed[:12], p)[2].float().cpu().numpy().reshape(-1), last, name, what="prompt")
    for cache in (c, p):
        cache[0].page_manager.release()


@pytest.mark.parametrize("bits,rows", [(8, 2), (4, 3), (4, 8)])
def test_a_step_over_pages_rotates_in_its_attention(bits, rows):
    """Up to 1024 columns (q|k|v in one pass over K): the product could rotate, but the attention's launch does it for less.  The kernels of one step, by name."""
    from torch.profiler import ProfilerActivity, profile
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": 1024, "num_hidden_layers": 2, "intermediate_size": 512, "num_attention_heads": 8, "num_key_value_heads": 4, "head_dim": 128, "vocab_size": 320,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "quantization": {"group_size": 64, "bits": bits}}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=2))
    m.enable_paged_kv(num_pages=16, max_blocks=1)
    caches, feed = [m.make_cache() for _ in range(rows)], torch.arange(rows, dtype=torch.int32, device="cuda")
    m.step_batch(feed, caches, graph=False)
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        m.step_batch(feed, caches, graph=False)
        torch.cuda.synchronize()
    names = [(e.key, e.count) for e in p.key_averages()]
    assert sum(n for k, n in names if "k_w4a_gemm" in k) == 9 and sum(n for k, n in names if "k_attn_step" in k) == 2, names


@pytest.mark.parametrize("budget,copies", [(1, True), (2, False)], ids=["tight", "ample"])
def test_prompts_copies_come_before_steps_tiles(budget, copies, knobs):
    """Steps of two sequences before the first long prompt, 0.9 GiB of 16-bit copies, half of that of the codes' tiles: in a budget of 1 GiB the steps multiply the copies that the prompt finds there, in one
    of 2 GiB they take tiles, and the prompt's copies have room beside them."""
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": 2048, "num_hidden_layers": 7, "intermediate_size": 8192, "num_attention_heads": 16, "num_key_value_heads": 4, "head_dim": 128, "vocab_size": 16384,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "quantization": {"group_size": 64, "bits": 8}}
    layers = 7 * 2048 * (3072 + 2048 + 3 * 8192)   # weights
    head = 16384 * 2048
    knobs("prefill_resident", budget)
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=2))
    m.enable_paged_kv(num_pages=40, max_blocks=2)
    caches = [m.make_cache() for _ in range(2)]
    feed = torch.arange(2, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    free = [torch.cuda.mem_get_info()[0]]
    m.step_batch(feed, caches, graph=False)
    torch.cuda.synchronize()
    free.append(torch.cuda.mem_get_info()[0])
    m.step(torch.arange(100, dtype=torch.int32, device="cuda"), m.make_cache())
    torch.cuda.synchronize()
    free.append(torch.cuda.mem_get_info()[0])
    steps, prompt = free[0] - free[1], free[1] - free[2]
    if copies:   # (tiles and scratch would be 0.6 GiB; what the prompt takes beside is its own scratch)
        assert steps >= 2 * (layers + head)
    else:   # (the last layer's o_proj, gate|up and down have one row left and take tiles, which are there)
        assert 1.0625 * (layers + head) <= steps < 1.6 * (layers + head) and prompt >= 2 * layers * 6 // 7
