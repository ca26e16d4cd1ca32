"""Few sequences' steps of int4 models have two forms (one launch per product with norms, rotation and sums in it, or the general path on W4M tiles): a captured step keeps the one it was captured in."""
import numpy as np
import pytest
import torch

from _util import assert_vec_close

pytestmark = pytest.mark.gpu

CFG = {"model_type": "llama", "hidden_size": 256, "num_hidden_layers": 2, "intermediate_size": 704, "num_attention_heads": 4, "num_key_value_heads": 2, "rms_norm_eps": 1e-5, "vocab_size": 4096,
       "rope_theta": 10000.0, "max_position_embeddings": 2048, "tie_word_embeddings": False, "quantization": {"group_size": 64, "bits": 4}}


def _model(change=None):
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    w = synthetic_checkpoint(CFG, seed=5, lm_head_gain=4.0)
    if change:
        change(w)
    m = Model(ModelArgs(**CFG), w)
    m.enable_paged_kv(num_pages=32, max_blocks=4)
    return m


def _steps(m, B, steps, before=lambda i: None):
    """Every sequence's steps alone (one-sequence launches, the reference of this suite: four ulps of the largest logit), then together; before(i) runs in front of step i."""
    rng = np.random.default_rng(B)
    feed = torch.from_numpy(rng.integers(0, CFG["vocab_size"], (steps, B)).astype(np.int32)).cuda()
    prompts = [torch.from_numpy(rng.integers(0, CFG["vocab_size"], n).astype(np.int32)).cuda() for n in (9, 70, 23, 61, 40)[:B]]
    want = []
    for b in range(B):
        c = m.make_cache()
        m.step(prompts[b], c)
        want.append([m.step(feed[i, b:b + 1], c)[2].float().cpu().numpy().reshape(-1) for i in range(steps)])
        c[0].page_manager.release()
    caches = [m.make_cache() for _ in range(B)]
    for c, p in zip(caches, prompts):
        m.step(p, c)
    for i in range(steps):
        before(i)
        got = m.step_batch(feed[i], caches)[2].float().cpu().numpy()
        for b in range(B):
            assert_vec_close(got[b], want[b][i], "bfloat16", what=f"B {B} step {i} row {b}")


@pytest.mark.parametrize("first", [None, 0], ids=["tiles", "gemv"])
@pytest.mark.parametrize("B", [3, 5])
def test_a_replayed_step_keeps_the_form_that_was_captured(B, first, knobs):
    """Warm, captured, replayed; then the switch that decides between the forms moves, twice, and the steps are still those of their tokens."""
    m = _model()
    other = 0 if first is None else None

    def before(i):
        if i in (0, 4, 6):
            knobs("w4r", other if i == 4 else first)
    _steps(m, B, 8, before)


@pytest.mark.parametrize("B", [2, 3, 5])
def test_scales_beyond_the_tiles_range(B):
    """The first step finds a matrix that the tiles' product does not take (a scale of 2^101, on codes and a bias of zero), the steps behind it have another form: eager, captured and replayed."""
    def change(w):
        n = "model.layers.1.self_attn.o_proj"
        w[n + ".weight"][3, :8] = 0                 # row 3's first 64 codes
        w[n + ".scales"][3, 0], w[n + ".biases"][3, 0] = 2.0 ** 101, 0.0
    _steps(_model(change), B, 7)
