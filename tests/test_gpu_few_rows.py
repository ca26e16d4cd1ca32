"""The Linear of 5 to 64 rows whose operand goes through LDS (k_rows_lds), where it can go wrong: a last chunk of K that is not whole, row blocks that are not full, experts with more rows
than a block, output widths on both sides of every choice of features per workgroup, float16, biases."""
import numpy as np
import pytest
import torch

import taduzen_util as tu
from oracle import taduzen_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [331, 5203, 10259])   # 21, 326 and 642 blocks of 16 features: one, two and four per workgroup
def test_stack_linears_against_the_oracle(vocab):
    """K = 1096 and 1100 (chunks of 256, 512 or 1024 columns), experts with 2 / 3 of the rows each beside a shared one, every wanted row through the head.  bfloat16 storage everywhere: two layers'
    roundings of 2^-9 stay below 0.04 of a row (the bound of the other tests of this design); a dropped or doubled chunk is a quarter of a product and more."""
    from proxy_inference_engine_amd.models.taduzen import Model, ModelArgs
    cfg = tu.config([(tu.latent(heads=9, dim=120, vdim=116, rank=72, window=40), tu.dense(1100)), (tu.latent(heads=2, rank=40), tu.moe(ff=1100, experts=3, top=2, shared=1300))], width=1096, vocab=vocab)
    w = tu.weights(cfg, seed=8)
    m = Model(ModelArgs(**cfg), {k: v.cuda() for k, v in w.items()}, dtype=torch.bfloat16)
    m.enable_paged_kv(num_pages=8)
    wn = tu.as_numpy(w)
    for n in (4, 5, 16, 17, 32, 33, 60):
        ids, c = tu.tokens(cfg, n, seed=n), m.make_cache()
        got = m.step_portions([(ids, c)], [list(range(n))]).cpu().numpy()
        c[0].page_manager.release()
        assert tu.err(got, orc.forward(cfg, wn, ids)) < 0.04, n


def test_mixtures_whose_shared_expert_has_more_rows_than_a_block():
    """64 experts and a shared one, 17 to 64 rows: blocks of 32 rows, in long chunks (17 rows: fewer than 2048 workgroups) and short ones.  The same tokens four at a time take the kernel
    without LDS; bounds as above."""
    from proxy_inference_engine_amd.models.taduzen import Model, ModelArgs
    cfg = tu.config([(tu.latent(heads=2, rank=40), tu.moe(ff=512, experts=64, top=3, shared=640))], width=1096, vocab=200)
    m = Model(ModelArgs(**cfg), {k: v.cuda() for k, v in tu.weights(cfg, seed=9).items()}, dtype=torch.bfloat16)
    m.enable_paged_kv(num_pages=8)
    ids, c = tu.tokens(cfg, 64, seed=3), m.make_cache()
    want = np.concatenate([m.step_portions([(ids[i:i + 4], c)], [list(range(4))]).cpu().numpy() for i in range(0, 64, 4)])
    c[0].page_manager.release()
    for n in (17, 32, 33, 49, 64):
        got = m.step_portions([(ids[:n], c)], [list(range(n))]).cpu().numpy()
        c[0].page_manager.release()
        assert tu.err(got, want[:n]) < 0.04, n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("vocab", [330, 5210, 10260])
def test_dense_llama_step_of_several_rows(dtype, vocab):
    """A step of B sequences against the same tokens fed to single sequences (another kernel: the GEMV).  Two layers, both sides accumulate in fp32 and round to T at the same places: four ulps of the largest
    logit, rms four ulps, as everywhere in this suite."""
    from _util import assert_vec_close
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": 1088, "num_hidden_layers": 2, "intermediate_size": 1472, "num_attention_heads": 16, "num_key_value_heads": 4, "head_dim": 64,
           "vocab_size": vocab, "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "attention_bias": True, "mlp_bias": True, "quantization": None}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=2, dtype=dtype))
    m.enable_paged_kv(num_pages=96, max_blocks=2)
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, vocab, 7 + i % 5).astype(np.int32) for i in range(32)]
    feed = torch.from_numpy(rng.integers(0, vocab, 32).astype(np.int32)).cuda()
    want = []
    for i, p in enumerate(prompts):
        c = m.make_cache()
        m.step(torch.from_numpy(p).cuda(), c)
        want.append(m.step(feed[i:i + 1], c)[2].float().cpu().numpy().reshape(-1))
        c[0].page_manager.release()
    for B in (1, 2, 5, 6, 16, 17, 32):
        caches = [m.make_cache() for _ in range(B)]
        for p, c in zip(prompts, caches):
            m.step(torch.from_numpy(p).cuda(), c)
        for step in range(4):   # eager, captured, replayed; the same position again after every step
            got = m.step_batch(feed[:B], caches)[2].float().cpu().numpy()
            for i in range(B):
                assert_vec_close(got[i], want[i], "bfloat16" if dtype == torch.bfloat16 else "float16", what=f"B {B} row {i} step {step}")
                for layer in caches[i]:
                    layer.trim(1)
        for c in caches:
            c[0].page_manager.release()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("inter,vocab", [(1472, 330), (5632, 16900)])
def test_dense_llama_step_on_both_sides_of_the_choice_of_kernel(dtype, inter, vocab):
    """Rows of 2048 columns, where the number of rows decides between the two kernels: 26 from 256 blocks of features down, 10 or 13 for wider products, and every choice of features per
    workgroup up to 32 rows.  Each sequence's first step alone (the GEMV) is the reference; bounds as above."""
    from _util import assert_vec_close
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": 2048, "num_hidden_layers": 1, "intermediate_size": inter, "num_attention_heads": 16, "num_key_value_heads": 4, "head_dim": 128,
           "vocab_size": vocab, "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "attention_bias": True, "mlp_bias": True, "quantization": None}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=2, dtype=dtype))
    m.enable_paged_kv(num_pages=40, max_blocks=1)
    feed = torch.from_numpy(np.random.default_rng(3).integers(0, vocab, 32).astype(np.int32)).cuda()
    want = []
    for i in range(32):
        c = m.make_cache()
        want.append(m.step(feed[i:i + 1], c)[2].float().cpu().numpy().reshape(-1))
        c[0].page_manager.release()
    for B in (5, 9, 10, 12, 13, 16, 17, 25, 26, 32):
        caches = [m.make_cache() for _ in range(B)]
        got = m.step_batch(feed[:B], caches, graph=False)[2].float().cpu().numpy()
        for i in range(B):
            assert_vec_close(got[i], want[i], "bfloat16" if dtype == torch.bfloat16 else "float16", what=f"B {B} row {i}")
        for c in caches:
            c[0].page_manager.release()


@pytest.mark.parametrize("bits", [None, 8, 4], ids=["dense", "int8", "int4"])
def test_a_head_changed_in_place_is_seen_after_set_globals(bits):
    """The head's tiles stay with the decoder; pie_decoder_set_globals says that the weights behind its pointers are others.  Batch steps, eager and replayed, and prompts with logits
    everywhere, against a decoder that was made with the new head."""
    import ctypes as C

    from proxy_inference_engine_amd import _ffi
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": 512, "num_hidden_layers": 2, "intermediate_size": 512, "num_attention_heads": 8, "num_key_value_heads": 2, "head_dim": 64, "vocab_size": 1024,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "quantization": {"group_size": 64, "bits": bits} if bits else None}
    w = synthetic_checkpoint(cfg, seed=3)
    others = synthetic_checkpoint(cfg, seed=4)
    a, b = Model(ModelArgs(**cfg), dict(w)), Model(ModelArgs(**cfg), dict(w, **{k: v for k, v in others.items() if k.startswith("lm_head")}))
    feed, ids = torch.arange(8, dtype=torch.int32, device="cuda"), torch.arange(40, dtype=torch.int32, device="cuda")
    caches = {}
    for m in (a, b):
        m.enable_paged_kv(num_pages=32, max_blocks=4)
        caches[m] = [m.make_cache() for _ in range(8)]
        for i, c in enumerate(caches[m]):
            m.step(ids[:9 + i], c)

    def steps(m, graph):
        out = []
        for _ in range(3):
            out.append(m.step_batch(feed, caches[m], graph=graph)[2].clone())
            for c in caches[m]:
                for layer in c:
                    layer.trim(1)
        c = m.make_cache()
        out.append(m(ids[None], cache=c).clone())
        c[0].page_manager.release()
        return out
    before = steps(a, True)
    want = steps(b, True)
    assert not torch.equal(before[0], want[0])
    a.lm_head.packed.copy_(b.lm_head.packed)
    _ffi.check(_ffi.load().pie_decoder_set_globals(a._dec, C.byref(a._globals)))
    for graph in (False, True):
        for got, ref in zip(steps(a, graph), want):
            assert torch.equal(got, ref)
