"""Taduzen without a GPU: configuration, registry, the latent page pool's bookkeeping, and the oracle against itself."""
import json

import numpy as np
import pytest
import torch

import taduzen_util as tu
from oracle import taduzen_oracle as orc
from proxy_inference_engine_amd.cache.kv_cache import LatentPageAllocator, PagedLatentCache, PagedSequence
from proxy_inference_engine_amd.models import utils as mu
from proxy_inference_engine_amd.models.taduzen import ModelArgs


def test_config_is_read_layer_by_layer():
    cfg = tu.config([(tu.latent(window=7), tu.dense(30)), (tu.latent(heads=3, dim=20, vdim=12, window=None), None), (tu.latent(), tu.moe(shared=None))])
    a = ModelArgs(**json.loads(json.dumps(cfg)))
    assert [lay.mixer.heads for lay in a.layers] == [4, 3, 4] and a.layers[0].mixer.mask.size == 7 and a.layers[1].mixer.mask is None
    assert a.layers[1].mlp is None and a.layers[2].mlp.shared is None and a.layers[2].mlp.router.top == 2 and a.norm.eps == 1e-5


def test_registry_refuses_an_unknown_architecture(tmp_path):
    from safetensors.torch import save_file
    save_file({"x": torch.zeros(1)}, str(tmp_path / "model.safetensors"))
    (tmp_path / "config.json").write_text(json.dumps({"architecture": "Nosuch"}))
    with pytest.raises(ValueError, match="Taduzen"):
        mu.load_model(str(tmp_path))


def test_latent_pages_share_ids_over_layers_of_different_widths():
    pool = LatentPageAllocator(4, [24, 8], dtype=torch.float32, device="cpu")
    assert [tuple(s.shape) for s in pool.slabs] == [(4, 64, 24), (4, 64, 8)] and pool.page_bytes == 64 * 32 * 4
    seq = PagedSequence(pool, 1)
    cache = [PagedLatentCache(seq, i) for i in range(2)]
    rows = [torch.randn(1, 1, 70, n) for n in (24, 8)]
    for c, r in zip(cache, rows):
        c.state = (r, None)
    assert seq.offset == 70 and len(seq.pages) == 2 and pool.get_num_free_pages() == 2
    assert all(torch.equal(c.state[0], r) for c, r in zip(cache, rows))
    other = seq.fork()                       # the full page shared, the partly filled one copied
    assert other.pages[0] == seq.pages[0] and other.pages[1] != seq.pages[1]
    assert torch.equal(PagedLatentCache(other, 1).state[0], rows[1])
    cache[0].trim(10)
    assert seq.offset == 60 and len(seq.pages) == 1
    seq.release(), other.release()
    assert pool.get_num_free_pages() == 4


def test_saved_latents_round_trip(tmp_path):
    from proxy_inference_engine_amd.cache.kv_cache import BaseCache, SavedLatentCache
    pool = LatentPageAllocator(2, [16], dtype=torch.bfloat16, device="cpu")
    c = [PagedLatentCache(PagedSequence(pool, 1), 0)]
    c[0].state = (torch.randn(1, 1, 9, 16).to(torch.bfloat16), None)
    BaseCache.save_cache(str(tmp_path / "c.safetensors"), c, {"k": "v"})
    back, meta = BaseCache.load_cache(str(tmp_path / "c.safetensors"), device="cpu")
    assert isinstance(back[0], SavedLatentCache) and back[0].offset == 9 and torch.equal(back[0].rows, c[0].state[0]) and meta == {"k": "v"}


def test_oracle_window_edges_matter():
    """The sharpened weights the device tests use: a window one token off changes the logits of the positions it touches, and only those."""
    cfg = tu.config([(tu.latent(window=9), None)])
    w, ids = tu.as_numpy(tu.weights(cfg, q_gain=6.0)), tu.tokens(cfg, 30)
    a = orc.forward(cfg, w, ids)
    for off in (-1, 1):
        other = json.loads(json.dumps(cfg))
        other["layers"][0]["mixer"]["mask"]["size"] += off
        b = orc.forward(other, w, ids)
        first = 9 if off > 0 else 8
        assert np.allclose(a[:first], b[:first]) and tu.err(b[first:], a[first:]) > 0.1


def test_oracle_absorbed_form_agrees():
    """score and value of latent attention written over the latents alone (what the kernels do) equal the spelled-out keys and values."""
    cfg = tu.config([(tu.latent(heads=2, dim=6, vdim=10, rank=14, window=5), None)])
    w, m = tu.as_numpy(tu.weights(cfg)), cfg["layers"][0]["mixer"]
    h = np.random.default_rng(0).normal(size=(11, cfg["width"]))
    want = orc.latent_attention(h, w, "l0.mix.", 2, 6, 10, m["scale"], 5, 1e-5)
    c = orc.rms(h @ w["l0.mix.dkv"].T, w["l0.mix.dkv.norm"], 1e-5)
    q = (h @ w["l0.mix.q"].T).reshape(11, 2, 6)
    out = []
    for a in range(2):
        ql = q[:, a] @ w["l0.mix.uk"].reshape(2, 6, 14)[a]
        out.append(orc.softmax_rows(ql @ c.T * m["scale"], orc.visible(11, 5)) @ c @ w["l0.mix.uv"].reshape(2, 10, 14)[a].T)
    assert np.allclose(np.concatenate(out, 1) @ w["l0.mix.o"].T, want)


@pytest.mark.parametrize("mistake", ["expert", "share", "gate", "post_norm", "norm_bias", "alpha", "latent_norm", "scale", "logit_scale", "act"])
def test_oracle_mistakes_show(mistake, monkeypatch):
    """With the weights the device tests use, every mechanism left out or replaced moves the logits by far more than those tests allow."""
    cfg = tu.config([(tu.latent(), tu.dense()), (tu.latent(heads=2), tu.moe())])
    w, ids = tu.as_numpy(tu.weights(cfg, seed=3, q_gain=2.0)), tu.tokens(cfg, 60)
    want = orc.forward(cfg, w, ids)
    if mistake == "expert":
        w["l1.mlp.table"] = (w["l1.mlp.table"] + 1) % 5
    elif mistake == "share":
        w["l1.mlp.table"] = w["l1.mlp.table"][:, [0, 0]]
    elif mistake == "gate":
        monkeypatch.setattr(orc, "sigmoid", lambda z: np.ones_like(z))
    elif mistake == "post_norm":
        w["l0.norm1b.alpha"] = w["l0.norm1b.alpha"] * 2
    elif mistake == "norm_bias":
        w["l1.norm2.b"] = np.zeros_like(w["l1.norm2.b"])
    elif mistake == "alpha":
        w["final.norm.alpha"] = np.ones(())
    elif mistake == "latent_norm":
        w["l0.mix.dkv.norm"] = np.ones_like(w["l0.mix.dkv.norm"])
    elif mistake == "scale":
        cfg["layers"][1]["mixer"]["scale"] = 1.0
    elif mistake == "logit_scale":
        cfg["logit_scale"] = 1.0
    elif mistake == "act":
        monkeypatch.setattr(orc, "relu2", lambda z: np.maximum(z, 0.0))
    assert tu.err(orc.forward(cfg, w, ids), want) > 0.05


def test_rows_picked_from_more_than_2_gib_take_the_kernel_with_64_bit_addresses():
    """The head multiplies a few wanted rows of a pass of up to 65535: what counts is where those may lie, not how many they are.  Widths to 32768 are accepted."""
    from proxy_inference_engine_amd import _ffi

    def lds(M, K, ldx, x_rows):
        return _ffi.base().pie_stack_linear_kernel(M, 4000, K, ldx, x_rows)
    for M in (5, 16, 64):
        assert lds(M, 32768, 32768, 0) == 1 and lds(M, 32768, 32768, M) == 1 and lds(M, 32768, 32768, 32767) == 1
        assert lds(M, 32768, 32768, 32768) == 0 and lds(M, 32768, 32896, 32650) == 0 and lds(M, 32768, 32768, 65535) == 0
        assert lds(M, 16384, 16384, 65535) == 1 and lds(M, 16384, 16400, 65535) == 0
        for where in (0, -1):   # 64 rows, one behind the other, of a matrix alone and of one in a list
            assert lds(M, 32768, (1 << 24) - 8, where) == 1 and lds(M, 32768, 1 << 24, where) == 0
    assert _ffi.base().pie_stack_linear_kernel(0, 1, 1, 1, 0) < 0


def test_few_rows_take_the_kernel_that_is_faster_for_their_size():
    """Short rows of x and few of them: both operands straight into the lanes; long ones, more of them, or a chip that the other kernel fills: x through LDS."""
    from proxy_inference_engine_amd import _ffi

    def lds(M, N, K):
        return _ffi.base().pie_stack_linear_kernel(M, N, K, K, 0)
    assert [lds(M, 2048, 2048) for M in (4, 5, 8, 16, 25, 26, 64)] == [0, 0, 0, 0, 0, 1, 1]
    assert [lds(M, 4096, 4096) for M in (5, 12, 13, 32)] == [0, 0, 1, 1]
    assert [lds(M, 3072, 3072) for M in (8, 9, 10)] == [0, 0, 1] and [lds(M, 4096, 14336) for M in (4, 5)] == [0, 1]
    assert [lds(M, 8192, 2048) for M in (9, 10)] == [0, 1] and [lds(M, 6144, 4096) for M in (4, 5)] == [0, 1]
    assert [lds(M, 11264, 2048) for M in (4, 5, 64)] == [0, 1, 1] and [lds(M, 16896, 2048) for M in (12, 13)] == [0, 1]
    assert [lds(M, 28672, 4096) for M in (4, 5)] == [0, 1] and lds(64, 1024, 4096) == 0 and lds(64, 4096, 1000) == 0
