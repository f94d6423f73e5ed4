"""Prompt chunks on the one-call layers: against a float32 stack of the same weights, with the module-by-module path of the same
dtype as the yardstick.  Both round at the same points and differ in the order of their sums, so neither may be further from
float32 than the other by more than that difference; the bounds below are twice the yardstick's own distance."""
import ctypes

import pytest
import torch

from subspec_amd import _lib as L
from subspec_amd import model as M, ops
from subspec_amd.cache import create_kv_cache

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _stack(cfg, w, dtype, rows, cache="static"):
    kv = (create_kv_cache("static", max_cache_len=rows, config=cfg, device=DEV, dtype=dtype) if cache == "static" else
          create_kv_cache("paged", max_cache_len=rows, config=cfg, device=DEV, dtype=dtype))
    return M.Decoder(cfg, w["embed"].to(dtype), [{k: v.to(dtype) for k, v in l.items()} for l in w["layers"]],
                     w["norm"].to(dtype), w["lm_head"].to(dtype), kv)


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


def _cfg(hq, hkv):
    return M.DecoderConfig(num_hidden_layers=2, hidden_size=512, num_attention_heads=hq, num_key_value_heads=hkv, head_dim=128,
                           intermediate_size=1088, vocab_size=1024)


# rows around the tiles of the projections (64, 384) and of the attention (16, 32, 64 rows; one key block, several chunks)
@pytest.mark.parametrize("n,start", [(1, 0), (16, 3), (32, 64), (33, 0), (64, 61), (65, 0), (127, 1), (289, 130), (385, 0),
                                     (700, 64), (256, 1792), (17, 2000), (1, 2047), (1500, 7)])
@pytest.mark.parametrize("dtype,hq,hkv", [(torch.bfloat16, 7, 1), (torch.float16, 4, 2)])
def test_prefill_matches_float32(n, start, dtype, hq, hkv):
    cfg = _cfg(hq, hkv)
    w = M.init_weights(cfg, 3, DEV, dtype)
    w["embed"].mul_(50.0)
    g = torch.Generator(device=DEV).manual_seed(n * 7 + start)
    tokens = torch.randint(0, cfg.vocab_size, (n,), generator=g, device=DEV)
    past = torch.randn((2, 2, 1, hkv, start + n + 9, 128), generator=g, device=DEV).to(dtype)
    out = {}
    with torch.no_grad():
        for name, dt, native in (("exact", torch.float32, False), ("module", dtype, False), ("native", dtype, True)):
            d = _stack(cfg, w, dt, start + n + 9)
            d.use_native_layers = native
            d.kv.cache.data.copy_(past)
            logits = d.prefill(tokens, start, all_logits=True)
            out[name] = (logits, d.kv.cache.data.clone())
            if native:
                assert d._prefill_plan(d.embed[tokens], start) is not None
    for part in (0, 1):
        assert torch.isfinite(out["native"][part]).all()
        module, native = (_rel(out[k][part], out["exact"][part]) for k in ("module", "native"))
        assert native <= 2 * module, (part, native, module)
    rows = out["native"][1]
    assert torch.equal(rows[..., :start, :], past[..., :start, :]) and torch.equal(rows[..., start + n:, :], past[..., start + n:, :])


# more workgroups than compute units and windows of very different length: they start in falling order.  Two chunks at the longest
# windows, and three and more, of which the shorter windows have fewer: every form of the merge over a stride that no window fills
@pytest.mark.parametrize("n,start,hq,hkv,chunks", [(700, 0, 16, 16, 2), (705, 63, 16, 16, 2), (701, 350, 16, 16, 2), (600, 0, 28, 4, 5),
                                                   (1000, 63, 28, 4, 3), (1000, 250, 28, 4, 3), (1100, 1, 32, 8, 3), (1000, 333, 7, 1, 11)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_windows_in_falling_order(n, start, hq, hkv, chunks, dtype):
    order = L.lib().subspec_prefill_attention_order
    entries = (ctypes.c_int32 * 900)()
    assert order(hq, hkv, n, start, entries, 300) <= 300 and -(-(start + n) // entries[2]) == chunks
    assert entries[0] == entries[3] + 1 and entries[1] == entries[4] == 0       # the longest two windows' first chunks
    test_prefill_matches_float32(n, start, dtype, hq, hkv)


@pytest.mark.parametrize("n,start", [(20, 0), (70, 0), (300, 0), (130, 200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prefill_with_scores_far_below_zero(n, start, dtype):
    """Biases that put every score of a prompt's own keys near -1500 before the softmax (softmax over them is the ordinary one:
    they share the shift); with past rows, which lack the bias, ordinary scores lie in front of them and in chunks without any."""
    cfg = _cfg(4, 2)
    w = M.init_weights(cfg, 6, DEV, dtype)
    w["embed"].mul_(50.0)
    slow = torch.tensor([d for d in range(128) if d % 64 >= 60], device=DEV)       # dimensions that the rotation leaves alone
    for layer in w["layers"]:
        heads = layer["qkv_proj.bias"].view(-1, 128)
        heads[:cfg.num_attention_heads, slow] = -14.0
        heads[cfg.num_attention_heads:cfg.num_attention_heads + cfg.num_key_value_heads, slow] = 14.0
    g = torch.Generator(device=DEV).manual_seed(n + start)
    tokens = torch.randint(0, cfg.vocab_size, (n,), generator=g, device=DEV)
    past = torch.randn((2, 2, 1, 2, start + n + 9, 128), generator=g, device=DEV).to(dtype)
    past[:, 0, :, :, :100, 60:64] += 14.0                                          # the first chunk's keys have it too
    past[:, 0, :, :, :100, 124:] += 14.0
    out = {}
    with torch.no_grad():
        for name, dt, native in (("exact", torch.float32, False), ("module", dtype, False), ("native", dtype, True)):
            d = _stack(cfg, w, dt, start + n + 9)
            d.use_native_layers = native
            d.kv.cache.data.copy_(past)
            out[name] = d.prefill(tokens, start, all_logits=True)
    assert torch.isfinite(out["native"]).all()
    module, native = (_rel(out[k], out["exact"]) for k in ("module", "native"))
    assert native <= 2 * module, (native, module)


@pytest.mark.parametrize("chunks", [(70,), (40, 30), (5, 64, 1)])
def test_paged_prefill_equals_contiguous(chunks):
    cfg = _cfg(7, 1)
    w = M.init_weights(cfg, 4, DEV, torch.bfloat16)
    tokens = torch.randint(0, cfg.vocab_size, (sum(chunks),), device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    a, b = _stack(cfg, w, torch.bfloat16, 128), _stack(cfg, w, torch.bfloat16, 128, "paged")
    b.kv.cache.pool.allocate(3)                                      # the request's pages are not the pool's first ones
    with torch.no_grad():
        at = 0
        for n in chunks:
            assert torch.equal(a.prefill(tokens[at:at + n], at), b.prefill(tokens[at:at + n], at))
            at += n
    for i in range(2):
        for x, y in zip(a.kv.cache.prefix_kv(i, at), b.kv.cache.prefix_kv(i, at)):
            assert torch.equal(x, y)


def test_layers_outside_the_one_call_path_keep_running():
    cfg = _cfg(4, 2)
    w = M.init_weights(cfg, 5, DEV, torch.bfloat16)
    tokens = torch.arange(40, device=DEV)
    with torch.no_grad():
        d = _stack(cfg, w, torch.bfloat16, 64)
        want = d.prefill(tokens, 0)
        wide = torch.randn(cfg.hidden_size, cfg.q_size + 8, device=DEV, dtype=torch.bfloat16)
        wide[:, :cfg.q_size] = d.layers[1]["o_proj.weight"]
        d.layers[1]["o_proj.weight"] = wide[:, :cfg.q_size]          # a strided view: that layer goes module by module
        assert _rel(d.prefill(tokens, 0), want) < 0.02               # two bf16 layers: see the distances above


@pytest.mark.parametrize("extra", ["o_proj.bias", "gate_up_proj.bias", "down_proj.bias", "codes"])
def test_layers_that_hold_more_than_the_one_call_form_run_module_by_module(extra):
    """The one-call layer has a bias for q|k|v only and reads dense weights; a layer with other biases, or with int4 codes
    beside its dense matrices (the codes count), keeps its results."""
    cfg = _cfg(4, 2)
    w = M.init_weights(cfg, 7, DEV, torch.bfloat16)
    w["embed"].mul_(50.0)
    layer = w["layers"][1]
    g = torch.Generator(device=DEV).manual_seed(2)
    if extra == "codes":
        layer.update({k: v for k, v in M.quantize_layers([layer])[0].items() if k.startswith("gate_up_proj.")})
        layer["gate_up_proj.weight"] = torch.zeros_like(layer["gate_up_proj.weight"])
    else:
        rows = layer[extra.replace("bias", "weight")].shape[0]
        layer[extra] = torch.randn(rows, generator=g, device=DEV).to(torch.bfloat16)
    tokens = torch.randint(0, cfg.vocab_size, (40,), generator=g, device=DEV)
    out = []
    with torch.no_grad():
        for native in (False, True):
            kv = create_kv_cache("static", max_cache_len=64, config=cfg, device=DEV, dtype=torch.bfloat16)
            d = M.Decoder(cfg, w["embed"], w["layers"], w["norm"], w["lm_head"], kv)
            d.use_native_layers = native
            out.append(d.prefill(tokens, 0, all_logits=True))
    assert _rel(out[1], out[0]) < 0.02                               # one bf16 layer in another order of sums


def test_int4_stacks_allocate_no_workspace_for_layers_that_decline_it():
    """int4 layers of a prompt run module by module; the one-call layers' workspace (69 MB here) is for those that use it."""
    cfg = M.DecoderConfig(num_hidden_layers=1, hidden_size=512, num_attention_heads=4, num_key_value_heads=2, head_dim=128,
                          intermediate_size=11264, vocab_size=1024)
    w = M.init_weights(cfg, 9, DEV, torch.bfloat16)
    tokens = torch.randint(0, cfg.vocab_size, (1500,), generator=torch.Generator(device=DEV).manual_seed(3), device=DEV)
    peak = []
    with torch.no_grad():
        for native in (False, True, False, True):                    # (the first round also sets up what the libraries keep)
            kv = create_kv_cache("static", max_cache_len=1500, config=cfg, device=DEV, dtype=torch.bfloat16)
            d = M.Decoder(cfg, w["embed"], M.quantize_layers(w["layers"]), w["norm"], w["lm_head"], kv)
            d.use_native_layers = native
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats()
            before = torch.cuda.memory_allocated()
            d.prefill(tokens, 0)
            peak.append(torch.cuda.max_memory_allocated() - before)
            del d, kv
    assert peak[3] <= peak[2] + 65536, peak                          # (row numbers and the like)


def test_prefill_layer_refuses_what_it_cannot_hold():
    d = lambda **k: ops.decoder_layer_dims(**{**dict(dtype=torch.bfloat16, n_rows=8, hidden=512, intermediate=1088, n_q_heads=4,
                                                     n_kv_heads=2, head_dim=128, kv_seq_stride=64, prefix_len=0, n_tree_slots=1,
                                                     rms_eps=1e-6, rope_theta=1e4), **k})
    assert ops.prefill_layer_workspace(d()) > 0
    for bad in (dict(prefix_len=57), dict(head_dim=64), dict(hidden=520), dict(n_rows=65537, kv_seq_stride=1 << 20)):
        assert ops.prefill_layer_workspace(d(**bad)) == 0
