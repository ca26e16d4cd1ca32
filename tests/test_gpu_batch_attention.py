"""RoPE and the K / V append inside the attention launch of a batch's step (k_attn_step): the new position at every edge of its page and of the split that
ends with it, one split and several, the group sizes in use, both rotary conventions, the projection as T rows (dense, biased) and as K-split slabs
(int4 from six rows).  The reference is each sequence served alone: other kernels append its row and score its cache."""
import numpy as np
import pytest
import torch

from tests._util import assert_vec_close

pytestmark = pytest.mark.gpu

LENS = [1, 2, 31, 63, 64, 65, 128, 257, 520]  # positions cached before the step: the new row opens a page at 64 and 128, lies beyond the first loads in flight at 257 and 520


def _model(hidden, Hq, Hkv, D, traditional, quant, bias):
    from proxy_inference_engine_amd.models.llama import Model, ModelArgs
    from proxy_inference_engine_amd.models.utils import synthetic_checkpoint
    cfg = {"model_type": "llama", "hidden_size": hidden, "num_hidden_layers": 2, "intermediate_size": 512, "num_attention_heads": Hq, "num_key_value_heads": Hkv, "head_dim": D,
           "rms_norm_eps": 1e-5, "vocab_size": 512, "rope_theta": 10000.0, "max_position_embeddings": 2048, "tie_word_embeddings": False, "rope_traditional": traditional,
           "attention_bias": bias}
    if quant:
        cfg["quantization"] = {"group_size": 64, "bits": 4}
    return Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=11, lm_head_gain=4.0))


@pytest.mark.parametrize("hidden,Hq,Hkv,D,traditional,quant,bias", [
    (512, 8, 2, 64, False, False, False), (512, 4, 4, 128, True, False, False), (896, 7, 1, 128, False, False, True),
    (1024, 8, 2, 128, False, True, False), (1024, 16, 2, 64, True, True, False), (768, 6, 2, 128, False, True, True)])
@pytest.mark.parametrize("rows", [9, 2])
def test_batch_step_appends_and_attends_like_each_sequence_alone(hidden, Hq, Hkv, D, traditional, quant, bias, rows):
    model = _model(hidden, Hq, Hkv, D, traditional, quant, bias)
    lens = LENS if rows == len(LENS) else [64, 520]
    rng = np.random.default_rng(rows)
    prompts = [rng.integers(0, 512, n).astype(np.int32) for n in lens]
    pool = model.enable_paged_kv(num_pages=2 * sum(n // 64 + 2 for n in lens), max_blocks=16)
    feed, both = [7 + i for i in range(len(lens))], []
    for batch in (False, True):
        caches = [model.make_cache() for _ in lens]
        for p, c in zip(prompts, caches):
            model.step(torch.from_numpy(p).cuda(), c)
        if batch:
            got = model.step_batch(torch.tensor(feed, dtype=torch.int32, device="cuda"), caches, graph=False)[2].float().cpu().numpy()
        else:
            got = np.stack([model.step(torch.tensor([t], dtype=torch.int32, device="cuda"), c)[2].float().cpu().numpy().reshape(-1) for t, c in zip(feed, caches)])
        rows_of = []
        for c, n in zip(caches, lens):
            page = pool.slab[0].view(torch.bfloat16).view(-1, 2, Hkv, 64, D)[c[0].page_manager.pages[n // 64]]
            rows_of.append(page[:, :, n % 64].clone())
        both.append((got, torch.stack(rows_of)))
    (alone, row_alone), (batched, row_batched) = both
    for i, n in enumerate(lens):
        assert_vec_close(batched[i], alone[i], "bfloat16", what=f"row {i}, {n} positions cached")
        # layer 0's new K / V row, whose inputs are equal.  Per side half an ulp (2^-9) for T(x W^T), for the bias added to it, both up to sqrt 2 larger after the rotation of a
        # pair, and for the rotation: 3.8 x 2^-9; both sides 2^-6.06 of the largest element.  int4 from six rows: weights rounded to T, 2^-9 of each product more, ~2^-9 of an
        # element in the mean.  Under 2^-5 together; another position's row or angle is off by the element itself.
        a, b = row_alone[i].float(), row_batched[i].float()
        assert float((a - b).abs().max()) <= float(a.abs().max()) * 2 ** -5, (i, n)


def _poison(pool, value):
    for slab in pool.slab:
        slab.view(torch.bfloat16).fill_(value)


@pytest.mark.parametrize("hidden,Hq,Hkv,D,quant,rows", [
    (512, 8, 2, 64, False, 3), (512, 8, 2, 64, False, 6), (512, 4, 4, 128, False, 3), (512, 4, 4, 128, False, 6), (1024, 8, 2, 128, True, 6),
    (512, 32, 8, 128, False, 1), (512, 32, 8, 128, True, 1)])
def test_a_step_that_opens_a_page_reads_no_row_that_nobody_wrote(hidden, Hq, Hkv, D, quant, rows):
    """The new position is row 0 of a fresh page (0, 64 and 128 cached): what else lies in the pool -- a recycled page's rows, memory never written -- may be NaN or infinite
    and must not count, not even with weight 0.  The same pool filled with zeros gives the same bits.  Three rows: one split; six: several; one row (32 / 8 heads of 128): the
    attention behind the q|k|v launch."""
    model = _model(hidden, Hq, Hkv, D, False, quant, False)
    cached = [0, 64, 128] * (rows // 3) if rows > 1 else [0, 64, 128]
    prompts = [np.random.default_rng(i).integers(0, 512, n).astype(np.int32) for i, n in enumerate(cached)]
    pool = model.enable_paged_kv(num_pages=2 * sum(n // 64 + 1 for n in cached), max_blocks=4)
    feed = torch.arange(7, 7 + len(cached), dtype=torch.int32, device="cuda")
    got = []
    for fill in (0.0, float("nan"), float("inf")):
        _poison(pool, fill)
        caches = [model.make_cache() for _ in cached]
        for p, c in zip(prompts, caches):
            if len(p):
                model.step(torch.from_numpy(p).cuda(), c)
        if rows > 1:
            got.append(model.step_batch(feed, caches, graph=False)[2].clone())
        else:
            got.append(torch.stack([model.step(feed[i:i + 1], c)[2].clone().reshape(-1) for i, c in enumerate(caches)]))
        for c in caches:
            c[0].page_manager.release()
    assert not torch.isnan(got[0]).any()
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.filterwarnings("ignore:The CUDA Graph is empty")
def test_a_step_of_a_batch_refuses_a_caller_s_capture():
    """A step moves the lengths on the device and the sequences on the host together; in a captured stream only the host's half would happen now."""
    model = _model(512, 8, 2, 64, False, False, False)
    model.enable_paged_kv(num_pages=16, max_blocks=4)
    caches = [model.make_cache() for _ in range(2)]
    for i, c in enumerate(caches):
        model.step(torch.arange(9 + i, dtype=torch.int32, device="cuda"), c)
    feed = torch.tensor([5, 6], dtype=torch.int32, device="cuda")
    want = []
    for _ in range(3):
        want.append(model.step_batch(feed, caches, graph=False)[2].clone())
    for c in caches:
        for layer in c:
            layer.trim(2)
    assert torch.equal(model.step_batch(feed, caches, graph=False)[2], want[1])
    with pytest.raises(RuntimeError, match="captur"):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            model.step_batch(feed, caches, graph=False)
    torch.cuda.synchronize()
    assert torch.equal(model.step_batch(feed, caches, graph=False)[2], want[2])


def test_rows_rotated_by_their_product_take_that_kernel_s_splits():
    """int4 of so few columns that q|k|v is not split: its epilogue rotates and appends, and the attention behind it takes short rows in one piece, whatever the tables have room for.  Tables
    of one page, where there is nothing else, give the same bits -- of sums that cancel, so that their order shows: keys of 0, values of up to 2^30 and their negatives."""
    from proxy_inference_engine_amd import _ffi
    import ctypes as C
    model, B = _model(256, 8, 8, 64, False, True, False), 8
    pool = model.enable_paged_kv(num_pages=2 * B, max_blocks=4)
    caches = [model.make_cache() for _ in range(B)]
    lens = [40 + 3 * i for i in range(B)]
    for n, c in zip(lens, caches):
        model.step(torch.arange(n, dtype=torch.int32, device="cuda"), c)
    gen = torch.Generator().manual_seed(1)
    for n, c in zip(lens, caches):
        half = torch.randn(8, n // 2, 64, generator=gen) * 2.0 ** torch.randint(10, 30, (8, n // 2, 64), generator=gen)
        rows = torch.cat([half, -half[:, torch.randperm(n // 2, generator=gen)], torch.zeros(8, n % 2, 64)], 1).to(torch.bfloat16).cuda()
        page = pool.slab[0].view(torch.bfloat16).view(-1, 2, 8, 64, 64)[c[0].page_manager.pages[0]]
        page[0, :, :n], page[1, :, :n] = 0, rows
    feed, ctx = torch.arange(B, dtype=torch.int32, device="cuda"), torch.tensor(lens, dtype=torch.int32, device="cuda") + 1
    slabs, got = (C.c_void_p * 2)(*[s.data_ptr() for s in pool.slab]), []
    for width in (1, 4):
        table = torch.zeros((B, width), dtype=torch.int32)
        table[:, 0] = torch.tensor([c[0].page_manager.pages[0] for c in caches])
        table, logits, logprobs, token = table.cuda(), torch.empty((B, 512), dtype=torch.bfloat16, device="cuda"), torch.empty((B, 512), device="cuda"), torch.empty(B, dtype=torch.int32, device="cuda")
        _ffi.check(_ffi.load().pie_decoder_step_batch(model._dec, _ffi.p(feed), _ffi.p(ctx), slabs, pool.size(), pool.slab[0].numel() * pool.slab[0].element_size(), _ffi.p(table), width, B,
                                                      _ffi.p(logits), _ffi.p(logprobs), _ffi.p(token), 0, _ffi.stream()))
        got.append(logits.clone())
    assert torch.isfinite(got[0]).all() and torch.equal(*got)
