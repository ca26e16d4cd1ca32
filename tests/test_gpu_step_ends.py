"""The launches at the two ends of a pass: rows, norm and angles in front of the layers; log-probabilities, greedy tokens and the next lengths behind them."""
import numpy as np
import pytest
import torch

from proxy_inference_engine_amd import _ffi, hip_ops as ops
from proxy_inference_engine_amd.models.llama import Model, ModelArgs
from proxy_inference_engine_amd.models.utils import synthetic_checkpoint

pytestmark = pytest.mark.gpu


def check(x, lp, token):
    """Against float64: the sum of a thread's V / 1024 terms and of 1024 threads in fp32, and two roundings of numbers of the log-probabilities' size."""
    x = x.double().cpu()
    V = x.shape[-1]
    assert int(token) == int(torch.argmax((x == x.max()).int()))   # the first one
    want = x - torch.logsumexp(x, -1)
    got, seen = lp.double().cpu(), torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), seen)
    bound = (V / 1024 + 40) * 2.0 ** -24 + 2.0 ** -23 * (want[seen].abs().max() + x[seen].abs().max())
    assert (got - want)[seen].abs().max() <= bound, V


@pytest.mark.parametrize("V", [1, 7, 8, 9, 1000, 8192, 8200, 32768, 33001, 65552])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
def test_log_probabilities_of_a_row(dtype, V):
    """One octet and less, octets of some threads, several rounds; maxima that occur twice, rows that are mostly -inf, large offsets."""
    g = torch.Generator().manual_seed(V)
    x = (torch.randn(V, generator=g) * 4).to(dtype)
    for y in (x, x + 100, torch.where(torch.rand(V, generator=g) < 0.9, torch.tensor(-torch.inf, dtype=dtype), x)):
        y[V // 3] = y[V - 1] = y.max() + 1 if torch.isfinite(y.max()) else 0.0
        token, lp = ops.logprobs_argmax(y.cuda())
        check(y, lp.flatten(), token)


@pytest.mark.parametrize("rows", [1, 3, 17, 40, 300])
def test_log_probabilities_of_many_rows(rows):
    """Sixteen workgroups a row, and one; with and without log-probabilities."""
    V = 4104
    x = torch.randn(rows, V, generator=torch.Generator().manual_seed(rows)).cuda()
    lib = _ffi.load()
    ws = torch.empty(lib.pie_logprobs_argmax_f32_workspace(rows), dtype=torch.uint8, device="cuda")
    for want in (True, False):
        lp, token = torch.zeros_like(x), torch.zeros(rows, dtype=torch.int32, device="cuda")
        _ffi.check(lib.pie_logprobs_argmax_f32(_ffi.p(x), rows, V, _ffi.p(lp) if want else None, _ffi.p(token), _ffi.p(ws), _ffi.stream()))
        assert torch.equal(token.long(), x.argmax(-1))
        for r in range(rows if want else 0):
            check(x[r], lp[r], token[r])


def llama(hidden, layers, quant, dtype="bfloat16"):
    cfg = {"model_type": "llama", "hidden_size": hidden, "num_hidden_layers": layers, "intermediate_size": 256, "num_attention_heads": 4, "num_key_value_heads": 2, "head_dim": 64, "vocab_size": 328,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "quantization": {"bits": quant[0], "group_size": quant[1]} if quant else None}
    return Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=11))


@pytest.mark.parametrize("hidden", [64, 320, 8256])
@pytest.mark.parametrize("quant", [None, (4, 64), (8, 64)], ids=str)
def test_rows_in_front_of_the_layers(hidden, quant):
    """Forms of the embedding table (groups of 32 have their test against the oracle); fewer columns than threads, and more than a thread keeps: a prompt in one pass against the same tokens one by one, and as embeddings.  Few enough
    roundings differ that four ulps of the largest number hold, as everywhere in this suite."""
    from _util import assert_vec_close
    m = llama(hidden, 1, quant)
    ids = torch.from_numpy(np.random.default_rng(hidden).integers(0, 328, 12).astype(np.int32)).cuda()
    cache, one = m.make_cache(), m.make_cache()
    m.step(ids, cache)
    for i in range(12):
        m.step(ids[i:i + 1], one)
    for a, b, what in ((cache[0].keys, one[0].keys, "keys"), (cache[0].values, one[0].values, "values")):
        assert_vec_close(a[0, :, :12].float().cpu().numpy().ravel(), b[0, :, :12].float().cpu().numpy().ravel(), "bfloat16", what=what)
    rows = m.make_cache()
    m.step_embeds(m.embed(ids)[None], rows)
    assert torch.equal(rows[0].keys[0, :, :12], cache[0].keys[0, :, :12])   # the table's rows, whoever fetches them


@pytest.mark.parametrize("B", [3, 7])
def test_batch_steps_take_tokens_where_they_lie_and_move_the_lengths_on(B):
    """Replayed steps with tokens at new addresses, on the host, and in the buffer that the step writes; sequences cut back in between.  Bit for bit the steps as launches."""
    m = llama(320, 2, (4, 64))
    m.enable_paged_kv(num_pages=64, max_blocks=4)
    rng = np.random.default_rng(B)
    prompts = [rng.integers(0, 328, 20 + 7 * i).astype(np.int32) for i in range(B)]
    tokens = torch.from_numpy(rng.integers(0, 328, (9, B)).astype(np.int32))
    device = tokens.cuda()
    runs = []
    for graph in (True, False):
        caches = [m.make_cache() for _ in range(B)]
        nxt = m.prefill_batch(prompts, caches)[0]
        out = []
        for t in range(9):
            step = tokens[t] if t == 3 else nxt if t in (4, 5) else device[t]
            nxt, logprobs, logits = m.step_batch(step, caches, graph=graph)
            out.append((nxt.clone(), logprobs.clone(), logits.clone()))
            if t == 6:   # (one sequence loses a token, another two: lengths from the host again)
                for cache, n in ((caches[0], 1), (caches[1], 2)):
                    for layer in cache:
                        layer.trim(n)
        assert [c[0].offset for c in caches] == [len(p) + 9 - n for p, n in zip(prompts, [1, 2] + [0] * B)]
        runs.append(out)
        for c in caches:
            c[0].page_manager.release()
    for a, b in zip(*runs):
        assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("B", [3, 7])
def test_lengths_move_where_they_were_given_to_be_written(B):
    """pie_decoder_step_batch leaves them, whatever bits its flags have; pie_decoder_step_batch_advance adds one to those of slots in use."""
    import ctypes as C
    m = llama(320, 2, (4, 64))
    pool = m.enable_paged_kv(num_pages=2 * B, max_blocks=4)
    caches = [m.make_cache() for _ in range(B)]
    m.prefill_batch([np.arange(9 + i, dtype=np.int32) for i in range(B)], caches)
    lens = torch.tensor([0] + [10 + i for i in range(1, B)], dtype=torch.int32)
    table = torch.tensor([[c[0].page_manager.pages[0], 0] for c in caches], dtype=torch.int32, device="cuda")
    feed, token = torch.arange(B, dtype=torch.int32, device="cuda"), torch.empty(B, dtype=torch.int32, device="cuda")
    logits, logprobs = torch.empty((B, 328), dtype=torch.bfloat16, device="cuda"), torch.empty((B, 328), device="cuda")
    slabs, lib = (C.c_void_p * 2)(*[s.data_ptr() for s in pool.slab]), _ffi.load()
    for step, flags, moved in ((lib.pie_decoder_step_batch, 0, 0), (lib.pie_decoder_step_batch, 4, 0), (lib.pie_decoder_step_batch_advance, 0, 1)):
        ctx = lens.cuda()
        _ffi.check(step(m._dec, _ffi.p(feed), _ffi.p(ctx), slabs, pool.size(), pool.slab[0].numel() * pool.slab[0].element_size(), _ffi.p(table), 2, B, _ffi.p(logits), _ffi.p(logprobs),
                        _ffi.p(token), flags, _ffi.stream()))
        assert torch.equal(ctx.cpu(), torch.where(lens > 0, lens + moved, lens)), (flags, moved)


@pytest.mark.parametrize("V", [8, 1023, 1024, 8192, 32768, 33001, 131072, 131075])
def test_the_sum_of_a_row_takes_exponentials_to_their_last_bit(V):
    """Rows of one logit of 0 and V - 1 equal ones below it, so that an exponential's error is the sum's, and rows of log-probabilities with a spike of 0: log sum exp is read off the spike, 1
    to 2.5.  In units of 2^-23: an exponential is at most 1 off and its last product half of one, together 1.5 / sqrt 3 = 0.87 rms, all of which equal logits show and random ones do not; a
    logarithm is at most 1 off below 2 and 2 above, 0.82 rms over the range: 1.19 and 0.82, 1.02 over both halves, and a fifth of that for 150 draws' scatter and the sums.  (An exponential of a
    rounded product, half of |x| log2 e off, gives 1.4 to 1.9 over both from 8192 logits on.)"""
    square = 0.0
    for i in range(150):
        if i % 2:
            x = torch.full((V,), 1.0 + i / 100 - np.log(V))
        else:
            x = torch.randn(V, generator=torch.Generator().manual_seed(i)) * 2
            x -= torch.logsumexp(x.double(), 0).float() + i / 150
        x[V // 2] = 0.0
        lp = ops.logprobs_argmax(x.cuda())[1]
        square += float(lp[V // 2].double().cpu() + torch.logsumexp(x.double(), 0)) ** 2
    assert (square / 150) ** 0.5 <= 1.25 * 2.0 ** -23


@pytest.mark.parametrize("V", [33, 32768, 131072])
@pytest.mark.parametrize("rows", [1, 5, 40])
def test_log_probabilities_in_the_logits_place(rows, V):
    x = torch.randn(rows, V, generator=torch.Generator().manual_seed(rows)).cuda()
    lib, got = _ffi.load(), []
    ws = torch.empty(lib.pie_logprobs_argmax_f32_workspace(rows), dtype=torch.uint8, device="cuda")
    for lp, logits in ((torch.empty_like(x), x), (x, x)):
        token = torch.empty(rows, dtype=torch.int32, device="cuda")
        _ffi.check(lib.pie_logprobs_argmax_f32(_ffi.p(logits), rows, V, _ffi.p(lp), _ffi.p(token), _ffi.p(ws), _ffi.stream()))
        got.append((lp.clone(), token))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("rows,V", [(1, 60000), (40, 60000), (41, 60000), (3, 65544), (5, 50257), (46, 50257), (47, 50257), (1, 42859), (2, 131075)])
def test_rows_of_a_large_vocabulary(rows, V):
    """In tiles and not, on both sides of the rule; odd rows, whose tiles lie at any alignment.  The maximum at a tile's first and last place and twice."""
    x = torch.randn(rows, V, generator=torch.Generator().manual_seed(V)) * 3
    x[0, V - 1] = x[0, V // 64 // 8 * 8 + 8] = 20.0
    x[rows - 1, :V // 2] = -torch.inf
    lib, d = _ffi.load(), x.cuda()
    ws = torch.empty(lib.pie_logprobs_argmax_f32_workspace(rows), dtype=torch.uint8, device="cuda")
    lp, token = torch.zeros_like(d), torch.zeros(rows, dtype=torch.int32, device="cuda")
    _ffi.check(lib.pie_logprobs_argmax_f32(_ffi.p(d), rows, V, _ffi.p(lp), _ffi.p(token), _ffi.p(ws), _ffi.stream()))
    for r in {0, rows // 2, rows - 1}:
        check(x[r], lp[r], token[r])


def test_a_16_bit_row_of_a_very_large_vocabulary():
    x = (torch.randn(262144, generator=torch.Generator().manual_seed(1)) * 3).to(torch.bfloat16)
    token, lp = ops.logprobs_argmax(x.cuda())
    check(x, lp, token)


@pytest.mark.parametrize("B", [2, 7, 44])
def test_steps_and_prompts_over_a_large_vocabulary(B):
    """65544 logits, 16 bits: tiles of up to 43 rows; as launches and as a captured step."""
    cfg = {"model_type": "llama", "hidden_size": 64, "num_hidden_layers": 1, "intermediate_size": 64, "num_attention_heads": 1, "num_key_value_heads": 1, "head_dim": 64, "vocab_size": 65544,
           "rms_norm_eps": 1e-5, "tie_word_embeddings": False}
    m = Model(ModelArgs(**cfg), synthetic_checkpoint(cfg, seed=2))
    m.enable_paged_kv(num_pages=2 * B, max_blocks=4)
    caches = [m.make_cache() for _ in range(B)]
    got = [m.prefill_batch([np.arange(5 + i % 3, dtype=np.int32) for i in range(B)], caches)]
    for graph in (False, True, True, True):
        token, logprobs, logits = m.step_batch(got[-1][0], caches, graph=graph)
        got.append((token.clone(), logprobs.clone(), logits.clone()))
    for token, logprobs, logits in got:
        for r in {0, B - 1}:
            check(logits[r], logprobs[r], token[r])
