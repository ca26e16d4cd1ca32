"""k_w4a_gemm through steps of several sequences and short prompts: fewer groups of K than waves, groups that are no multiple of eight, splits of K, every count of strips per workgroup,
a last workgroup that is not full, eight rows and sixteen, biases."""
import numpy as np
import pytest
import torch

from _util import assert_vec_close

pytestmark = pytest.mark.gpu


# [N, K] in strips of 32 and groups of 64: hidden 192: 3 groups; 1088: 17, every matrix strip by strip; 2048: gate|up in twos, vocab in threes, o_proj and down split; 512: gate|up in fours, vocab too, in
# 268 workgroups; 4096: q|k|v, o_proj and down in twos, split; 3136: q|k|v, o_proj and gate|up strip by strip, seven steps a wave, down two
@pytest.mark.parametrize("hidden,inter,vocab,heads,kv,dim,bias", [(192, 448, 96, 4, 2, 64, True), (1088, 1472, 5216, 17, 17, 64, False), (2048, 5632, 16896, 16, 4, 128, True),
                                                                  (512, 14336, 34240, 8, 2, 64, False), (4096, 4096, 12320, 32, 8, 128, False), (3136, 1024, 96, 49, 7, 64, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_rows_against_single_sequences(hidden, inter, vocab, heads, kv, dim, bias, dtype):
    """One layer, every sequence's step alone (the GEMV, the same arithmetic: fp32 sums of unrounded weights, one rounding) as the reference: four ulps of the largest logit, rms four ulps, as everywhere."""
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": hidden, "num_hidden_layers": 1, "intermediate_size": inter, "num_attention_heads": heads, "num_key_value_heads": kv, "head_dim": dim,
           "vocab_size": vocab, "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "attention_bias": bias, "mlp_bias": bias, "quantization": {"group_size": 64, "bits": 4}}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=2, dtype=dtype))
    m.enable_paged_kv(num_pages=40, max_blocks=1)
    name = "bfloat16" if dtype == torch.bfloat16 else "float16"
    ids = np.random.default_rng(3).integers(0, vocab, 16).astype(np.int32)
    feed, want = torch.from_numpy(ids).cuda(), []
    for i in range(16):
        c = m.make_cache()
        want.append(m.step(feed[i:i + 1], c)[2].float().cpu().numpy().reshape(-1))
        c[0].page_manager.release()
    for B in (3, 5, 8, 9, 16):
        caches = [m.make_cache() for _ in range(B)]
        got = m.step_batch(feed[:B], caches, graph=False)[2].float().cpu().numpy()
        for i in range(B):
            assert_vec_close(got[i], want[i], name, what=f"B {B} row {i}")
        for c in caches:
            c[0].page_manager.release()
    # a prompt: rotated and appended by the product where q|k|v is not split
    c, p = m.make_cache(), m.make_cache()
    for i in range(12):
        last = m.step(feed[i:i + 1], c)[2].float().cpu().numpy().reshape(-1)
    assert_vec_close(m.step(feed[:12], p)[2].float().cpu().numpy().reshape(-1), last, name, what="prompt")
    for cache in (c, p):
        cache[0].page_manager.release()
