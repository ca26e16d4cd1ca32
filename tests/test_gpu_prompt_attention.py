"""Prompt attention: the op at the edges of its blocks and masks against float64, and the form split along the keys (rows behind a cached prefix) against the row-by-row kernel."""
import numpy as np
import pytest
import torch

from proxy_inference_engine_amd import _ffi, hip_ops as ops

pytestmark = pytest.mark.gpu
EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("heads", [(2, 2), (3, 1), (4, 2), (8, 2), (5, 1), (8, 1)], ids=str)
@pytest.mark.parametrize("D", [64, 128])
def test_causal_rows_against_float64(heads, D, dtype):
    """Lengths and offsets around the blocks of 32 and 64 keys and the tiles of 32 rows; a scale of either sign, and zero (plain means).  The result is rounded once: one ulp of the largest
    output (values are at most about 4, sums of weights 1, P is split to 16 bits)."""
    Hq, Hkv = heads
    g = torch.Generator().manual_seed(D + Hq)
    for L, off, scale in ((2, 0, 0.3), (31, 1, 0.3), (32, 32, -0.3), (33, 63, 0.3), (64, 0, 0.0), (65, 64, -0.2), (97, 130, 0.3), (150, 7, 0.2)):
        T = off + L
        q, k, v = (torch.randn(1, n, m, D, generator=g).to(dtype) for n, m in ((Hq, L), (Hkv, T), (Hkv, T)))
        got = ops.scaled_dot_product_attention(q.cuda(), k.cuda(), v.cuda(), scale, mask="causal").double().cpu()
        r = Hq // Hkv
        s = q.double() @ k.double().repeat_interleave(r, 1).transpose(-1, -2).contiguous() * scale
        s = s.masked_fill(torch.arange(T)[None] > torch.arange(L)[:, None] + off, -torch.inf)
        want = torch.softmax(s, -1) @ v.double().repeat_interleave(r, 1)
        assert (got - want).abs().max() <= EPS[dtype] * want.abs().max(), (L, off, scale)


@pytest.mark.parametrize("heads", [(4, 1), (8, 2), (5, 1), (8, 1)], ids=str)
@pytest.mark.parametrize("D", [64, 128])
def test_short_prompts_against_float64(heads, D):
    """Up to 56 keys in blocks of 32, 57 in blocks of 64, a second tile of rows, a few cached keys; bound as above."""
    Hq, Hkv = heads
    g = torch.Generator().manual_seed(D + Hq)
    for L, off in ((3, 0), (33, 0), (48, 0), (56, 0), (57, 0), (20, 36), (20, 37), (40, 9)):
        q, k, v = (torch.randn(1, n, m, D, generator=g).to(torch.bfloat16) for n, m in ((Hq, L), (Hkv, off + L), (Hkv, off + L)))
        got = ops.scaled_dot_product_attention(q.cuda(), k.cuda(), v.cuda(), 0.3, mask="causal").double().cpu()
        r = Hq // Hkv
        s = q.double() @ k.double().repeat_interleave(r, 1).transpose(-1, -2).contiguous() * 0.3
        s = s.masked_fill(torch.arange(off + L)[None] > torch.arange(L)[:, None] + off, -torch.inf)
        want = torch.softmax(s, -1) @ v.double().repeat_interleave(r, 1)
        assert (got - want).abs().max() <= EPS[torch.bfloat16] * want.abs().max(), (L, off)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("heads", [(2, 1), (3, 1), (8, 2)], ids=str)
@pytest.mark.parametrize("D", [64, 128])
def test_two_waves_per_tile_against_float64(heads, D, dtype):
    """From 256 keys on, two to four heads a group: block pairs whose second half is empty, masked in part or whole, rows of one and of several tiles; bound as above.  The second half's
    values are much larger in one key each, so that a half that is lost or counted twice shows."""
    Hq, Hkv = heads
    g = torch.Generator().manual_seed(D + Hq)
    for L, off, scale in ((256, 0, 0.3), (257, 0, 0.3), (320, 0, -0.3), (321, 63, 0.3), (7, 249, 0.3), (40, 280, 0.2), (33, 400, 0.0), (450, 1, 0.2)):
        T = off + L
        q, k, v = (torch.randn(1, n, m, D, generator=g).to(dtype) for n, m in ((Hq, L), (Hkv, T), (Hkv, T)))
        v[:, :, 64::128] *= 8
        got = ops.scaled_dot_product_attention(q.cuda(), k.cuda(), v.cuda(), scale, mask="causal").double().cpu()
        r = Hq // Hkv
        s = q.double() @ k.double().repeat_interleave(r, 1).transpose(-1, -2).contiguous() * scale
        s = s.masked_fill(torch.arange(T)[None] > torch.arange(L)[:, None] + off, -torch.inf)
        want = torch.softmax(s, -1) @ v.double().repeat_interleave(r, 1)
        assert (got - want).abs().max() <= EPS[dtype] * want.abs().max(), (L, off, scale)


@pytest.mark.parametrize("paged", [False, True], ids=["contiguous", "paged"])
@pytest.mark.parametrize("geometry", [(8, 2, 64), (8, 1, 128), (2, 2, 128), (6, 2, 128)], ids=str)
def test_rows_behind_a_prefix_split_along_the_keys(geometry, paged):
    """700 cached tokens: 2 to 5 shares, the last ones empty or partly masked.  Two layers against the kernel that takes one query row at a time: both keep fp32 until one rounding, so four ulps of the
    largest logit as everywhere in this suite."""
    from _util import assert_vec_close
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    Hq, Hkv, D = geometry
    cfg = {"model_type": "llama", "hidden_size": 256, "num_hidden_layers": 2, "intermediate_size": 512, "num_attention_heads": Hq, "num_key_value_heads": Hkv, "head_dim": D, "vocab_size": 320,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "quantization": None}
    w = synthetic_checkpoint(cfg, seed=5)
    for n in list(w):
        if "q_proj" in n or "k_proj" in n:
            w[n] = w[n] * 6   # sharp attention: single keys decide
    m = Model(ModelArgs(**cfg), w)
    if paged:
        m.enable_paged_kv(num_pages=40, max_blocks=20)
    ids = torch.from_numpy(np.random.default_rng(1).integers(0, 320, 920).astype(np.int32)).cuda()
    cache = m.make_cache()
    m.step(ids[:700], cache)
    for n in (6, 32, 33, 65, 130, 200):
        got = []
        for valu in (1, None):
            _ffi.set_knob("prefill_attn_valu", valu)
            try:
                got.append(m(ids[None, 700:700 + n], cache=cache).float().cpu().numpy()[0])
            finally:
                _ffi.set_knob("prefill_attn_valu", None)
            for layer in cache:
                layer.trim(n)
        assert _ffi.load().pie_decoder_prompt_shares(m._dec) == (5 if n <= 64 else 3)   # of 700 keys: two blocks of 64 each, three from 65 rows on
        for i in range(n):
            assert_vec_close(got[1][i], got[0][i], "bfloat16", what=f"{n} rows, row {i}")


@pytest.mark.parametrize("paged", [False, True], ids=["contiguous", "paged"])
@pytest.mark.parametrize("geometry,calls", [((4, 2, 64), ((257, 700, 3), (300, 390, 2))), ((3, 1, 128), ((300, 700, 3), (257, 770, 4))), ((8, 2, 128), ((257, 700, 3), (300, 400, 2))),
                                            ((32, 16, 64), ((257, 600, 3), (257, 400, 1))), ((48, 16, 128), ((330, 400, 2),)), ((51, 17, 128), ((500, 500, 1), (490, 736, 1)))], ids=str)
def test_more_than_256_rows_behind_a_prefix(geometry, calls, paged):
    """Two to four heads a group.  Shares of two waves a tile (the first three geometries: the last share empty, its last block's second half empty), shares of one where the chip allows few of two (three of
    144 tiles, two of 176), no shares: two waves a tile, and one where many more keys are cached than rows come and 256 workgroups do not hold the tiles (490
    behind 736).  Against the kernel that takes one query row at a time; pages out of order.  One layer, so that no second layer's sharp scores multiply what one rounding of the first one's rows leaves
    between them: an ulp through o_proj, the MLP and the head, four of the largest logit as everywhere."""
    from _util import assert_vec_close
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    Hq, Hkv, D = geometry
    cfg = {"model_type": "llama", "hidden_size": 256, "num_hidden_layers": 1, "intermediate_size": 512, "num_attention_heads": Hq, "num_key_value_heads": Hkv, "head_dim": D, "vocab_size": 320,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "quantization": None}
    w = synthetic_checkpoint(cfg, seed=5)
    for n in list(w):
        if "q_proj" in n or "k_proj" in n:
            w[n] = w[n] * 6   # sharp attention: single keys decide
    m = Model(ModelArgs(**cfg), w)
    if paged:
        m.enable_paged_kv(num_pages=60, max_blocks=20)
    ids = torch.from_numpy(np.random.default_rng(1).integers(0, 320, 1300).astype(np.int32)).cuda()
    for n, before, shares in calls:
        cache, other = m.make_cache(), m.make_cache()
        for lo in range(0, before, 100):   # (two sequences take their pages in turn)
            m.step(ids[lo:min(lo + 100, before)], cache)
            if paged:
                m.step(ids[lo + 1:lo + 101], other)
        got = []
        for valu in (1, None):
            _ffi.set_knob("prefill_attn_valu", valu)
            try:
                got.append(m(ids[None, before:before + n], cache=cache).float().cpu().numpy()[0])
            finally:
                _ffi.set_knob("prefill_attn_valu", None)
            for layer in cache:
                layer.trim(n)
        assert _ffi.load().pie_decoder_prompt_shares(m._dec) == shares, (n, before)
        for i in range(n):
            assert_vec_close(got[1][i], got[0][i], "bfloat16", what=f"{n} rows behind {before}, row {i}")
        if paged:
            cache[0].page_manager.release(), other[0].page_manager.release()


def test_longer_splits_do_not_allocate():
    """Prompts behind longer and longer prefixes take more and more shares of more rows; the room for their sums is there from the first prompt on."""
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": 256, "num_hidden_layers": 2, "intermediate_size": 512, "num_attention_heads": 32, "num_key_value_heads": 8, "head_dim": 128, "vocab_size": 320,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "quantization": None}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=5))
    m.enable_paged_kv(num_pages=80, max_blocks=40)
    ids = torch.from_numpy(np.random.default_rng(1).integers(0, 320, 2048).astype(np.int32)).cuda()
    cache, other = m.make_cache(), m.make_cache()
    for n in (300, 200, 64, 40):   # every row count once without a prefix: the other buffers have their sizes
        m.step(ids[:n], other)
        other[0].page_manager.release()
    m.step(ids[:300], cache), m.step(ids[300:600], cache), m.step(ids[600:900], cache)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for n in (40, 64, 200, 300):
        m.step(ids[900:900 + n], cache)
        for layer in cache:
            layer.trim(n)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("heads", [(2, 2), (8, 2)], ids=str)
def test_scores_whose_rounding_is_more_than_one(heads, dtype):
    """Scores of 2^24 to 2^36: the largest key takes all the weight, and a score's rounding (up to 2^11) must not reach the exponential.  Sums of 64 products in fp32 are good to 2^-18 of the
    largest score, far below the distance of the two best keys for these draws, so the row is that key's value."""
    Hq, Hkv = heads
    g = torch.Generator().manual_seed(Hq)
    for power in (9, 12, 15):
        gain = 2.0 ** power if dtype == torch.float16 else 2.0 ** (power + 2)   # (float16: up to 4 x 2^15 would overflow, see the clamp)
        q, k, v = (torch.randn(1, n, m, 64, generator=g) for n, m in ((Hq, 70), (Hkv, 130), (Hkv, 130)))
        q, k, v = (q * gain).clamp(-6e4, 6e4).to(dtype), (k * gain).clamp(-6e4, 6e4).to(dtype), v.to(dtype)
        got = ops.scaled_dot_product_attention(q.cuda(), k.cuda(), v.cuda(), 0.5, mask="causal").double().cpu()
        r = Hq // Hkv
        s = q.double() @ k.double().repeat_interleave(r, 1).transpose(-1, -2).contiguous() * 0.5
        s = s.masked_fill(torch.arange(130)[None] > torch.arange(70)[:, None] + 60, -torch.inf)
        want = torch.softmax(s, -1) @ v.double().repeat_interleave(r, 1)
        top = s.topk(2, -1).values
        clear = (top[..., 0] - top[..., 1] > 2.0 ** -16 * s.masked_fill(s == -torch.inf, 0).abs().amax(-1))
        assert clear.float().mean() > 0.95
        assert torch.isfinite(got).all()
        assert ((got - want).abs().amax(-1)[clear] <= EPS[dtype] * want.abs().max()).all(), power


@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("bits", [None, 4, 8], ids=str)
def test_the_last_layer_of_a_prompt_takes_its_last_row_alone(bits, layers):
    """`step` against the pass that returns every position's logits, and `prefill_batch` against both: prompts of a row block, of several chunks (64 rows; the last one of a single row, of a few), fresh
    and behind a prefix.  The rows are multiplied in other blocks: four ulps of the largest logit, as everywhere in this suite."""
    from _util import assert_vec_close
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": 256, "num_hidden_layers": layers, "intermediate_size": 512, "num_attention_heads": 8, "num_key_value_heads": 2, "head_dim": 64, "vocab_size": 320,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "quantization": {"group_size": 64, "bits": bits} if bits else None}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=7))
    ids = torch.from_numpy(np.random.default_rng(3).integers(0, 320, 700).astype(np.int32)).cuda()
    _ffi.set_knob("prefill_chunk", 64)
    try:
        for before, n in ((0, 6), (0, 65), (0, 70), (0, 300), (150, 7), (150, 129)):
            caches = [m.make_cache(), m.make_cache()]
            got = []
            for cache, whole in zip(caches, (True, False)):
                if before:
                    m.step(ids[:before], cache)
                logits = m(ids[None, before:before + n], cache=cache)[0, -1] if whole else m.step(ids[before:before + n], cache)[2]
                got.append((logits.float().cpu().numpy().ravel(), m.hidden.float().cpu().numpy(), m.step(ids[before + n:before + n + 1], cache)[2].float().cpu().numpy().ravel()))
                assert cache[0].offset == before + n + 1
            for a, b, what in zip(got[1], got[0], ("logits", "hidden", "the next step")):
                assert_vec_close(a, b, "bfloat16", what=f"{what}, {n} behind {before}")
    finally:
        _ffi.set_knob("prefill_chunk", None)
    alone = []
    for n in (6, 1, 80):
        alone.append(m(ids[None, :n], cache=m.make_cache())[0, -1].float().cpu().numpy())
    m.enable_paged_kv(num_pages=20, max_blocks=4)
    logits = m.prefill_batch([ids[:n].cpu().numpy() for n in (6, 1, 80)], [m.make_cache() for _ in range(3)])[2].float().cpu().numpy()
    for i in (0, 2):   # (a prompt of one token by itself is a decode step, whose weights are not rounded)
        assert_vec_close(logits[i], alone[i], "bfloat16", what=f"prompt {i} of a batch")


@pytest.mark.parametrize("n", [6, 17, 40, 300])
def test_the_last_row_alone_goes_to_the_gemv(n):
    """Int4 prompts: the products of the row that the last layer goes on with (o_proj, gate|up, down), and the head's, by the kernels' names."""
    from torch.profiler import ProfilerActivity, profile
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": 512, "num_hidden_layers": 1, "intermediate_size": 2048, "num_attention_heads": 8, "num_key_value_heads": 2, "head_dim": 64, "vocab_size": 320,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "quantization": {"group_size": 64, "bits": 4}}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=7))
    ids = torch.from_numpy(np.random.default_rng(3).integers(0, 320, n).astype(np.int32)).cuda()
    m.step(ids, m.make_cache())
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        m.step(ids, m.make_cache())
        torch.cuda.synchronize()
    names = [(e.key, e.count) for e in p.key_averages()]
    assert sum(c for k, c in names if "k_w4s_gemv" in k) == 4 and sum(c for k, c in names if "k_w4a_gemm" in k or "k_w4r_gemm" in k or "k_w4l2_gemm" in k) == 1, names


@pytest.mark.parametrize("n", [40, 150])
@pytest.mark.parametrize("paged", [False, True])
def test_a_prompt_that_fails_leaves_the_sequence_where_it_was(n, paged):
    """The host refuses the last layer's product (a bias at an odd address) behind the launches of everything before it, in one chunk and in three: the prompt again, with its weights, is the prompt."""
    import ctypes as C
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": 256, "num_hidden_layers": 2, "intermediate_size": 512, "num_attention_heads": 8, "num_key_value_heads": 2, "head_dim": 64, "vocab_size": 320,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "quantization": {"group_size": 64, "bits": 4}}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=7))
    ids = torch.from_numpy(np.random.default_rng(3).integers(0, 320, 200).astype(np.int32)).cuda()
    if paged:
        m.enable_paged_kv(num_pages=20, max_blocks=8)
    blk, bias, lib = m.layers[1], torch.zeros(264, dtype=torch.bfloat16, device="cuda"), _ffi.load()

    def layer(o_bias):
        w = _ffi.pie_layer_weights(blk.input_layernorm.data_ptr(), blk.post_attention_layernorm.data_ptr(), blk.wqkv.packed.data_ptr(), blk.wo.packed.data_ptr(), blk.wgateup.packed.data_ptr(),
                                   blk.wdown.packed.data_ptr(), None, o_bias, None, None, *blk.formats)
        _ffi.check(lib.pie_decoder_set_layer(m._dec, 1, C.byref(w)))

    _ffi.set_knob("prefill_chunk", 64)
    try:
        got = []
        for fail in (False, True):
            cache = m.make_cache()
            m.step(ids[:30], cache)
            if fail:
                layer(bias.data_ptr() + 2)
                with pytest.raises(ValueError, match="alignment"):
                    m.step(ids[30:30 + n], cache)
                layer(None)
            got.append([m.step(ids[30:30 + n], cache)[2].clone(), m.step(ids[30 + n:31 + n], cache)[2].clone()])
            assert cache[0].offset == 31 + n
    finally:
        _ffi.set_knob("prefill_chunk", None)
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("power", [120, -124])
@pytest.mark.parametrize("heads", [(2, 2), (8, 2)], ids=str)
@pytest.mark.parametrize("D", [64, 128])
def test_values_near_the_limits_of_bf16(D, heads, power):
    """Scores that rise by seven powers of two over a row's keys and values of 2^120 or 2^-124: up to 60 times a value is what the sums have to hold.  Weights in two halves of bf16 (2^-17), scores
    good to 2^-20 of 8, one rounding to bf16."""
    Hq, Hkv = heads
    g = torch.Generator().manual_seed(D)
    n, rows = 300, 90
    u = torch.randn(D, generator=g)
    q = u.expand(1, Hq, rows, D).to(torch.bfloat16)
    k = (u / u.square().sum() * (torch.arange(n)[:, None] / n * 5) * D ** 0.5).expand(1, Hkv, n, D).to(torch.bfloat16)
    v = ((1 + torch.rand(1, Hkv, n, D, generator=g)) * 2.0 ** power).to(torch.bfloat16)
    got = ops.scaled_dot_product_attention(q.cuda(), k.cuda(), v.cuda(), D ** -0.5, mask="causal").double().cpu()
    r = Hq // Hkv
    s = q.double() @ k.double().repeat_interleave(r, 1).transpose(-1, -2).contiguous() * D ** -0.5
    s = s.masked_fill(torch.arange(n)[None] > torch.arange(rows)[:, None] + n - rows, -torch.inf)
    want = torch.softmax(s, -1) @ v.double().repeat_interleave(r, 1)
    assert torch.isfinite(got).all()
    assert ((got - want).abs() <= want * (2.0 ** -8 + 2.0 ** -15)).all(), float(((got - want).abs() / want).max())
