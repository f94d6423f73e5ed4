"""A stack in one call against the same layers called one by one: the joined launches sum the same values in the same order, so
the results are equal bit for bit."""
import pytest
import torch

from subspec_amd import model as M, ops
from subspec_amd.cache import create_kv_cache

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows: the int4 kernels of 8, 33 to 64 rows; dense up to 32, 64, more; a prompt.  hidden 4104-wide pieces: one and four per thread
@pytest.mark.parametrize("kind,rows,hidden", [("int4", 8, 512), ("int4", 40, 512), ("int4", 64, 4224), ("dense", 5, 512),
                                              ("dense", 64, 4224), ("dense", 289, 512), ("prefill", 300, 512), ("prefill", 513, 4224)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_stack_equals_layers(kind, rows, hidden, dtype):
    print("stack", kind, rows, hidden, dtype, flush=True)
    cfg = M.DecoderConfig(num_hidden_layers=3, hidden_size=hidden, num_attention_heads=5, num_key_value_heads=1, head_dim=128,
                          intermediate_size=8192, vocab_size=64)
    w = M.init_weights(cfg, rows, DEV, dtype)
    layers = M.quantize_layers(w["layers"]) if kind == "int4" else w["layers"]
    kv = create_kv_cache("static", max_cache_len=rows + 70, config=cfg, device=DEV, dtype=dtype)
    g = torch.Generator(device=DEV).manual_seed(rows)
    kv.cache.data.normal_(generator=g)
    past, prefix = kv.cache.data.clone(), 50
    x0 = torch.randn(rows, hidden, generator=g, device=DEV).to(dtype)
    dims = ops.decoder_layer_dims(dtype, rows, hidden, 8192, 5, 1, 128, rows + 70, prefix, 1 if kind == "prefill" else rows, 1e-6, 1e6)
    pos = torch.arange(prefix, prefix + rows, dtype=torch.int32, device=DEV)
    bits = None if kind == "prefill" else ops.ancestor_bits_tensor([-1] + list(range(rows - 1)), device=DEV)
    make = ops.decoder_layer_weights if kind == "int4" else ops.dense_layer_weights
    tables = [make(l) for l in layers]
    need = ops.prefill_layer_workspace(dims) if kind == "prefill" else ops.decoder_layer_workspace(dims)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    want = x0.clone()
    for i, t in enumerate(tables):
        args = (kv.cache.k(i), kv.cache.v(i), ws)
        if kind == "prefill":
            ops.prefill_layer_(want, dims, t, pos, pos, *args)
        else:
            ops.decoder_layer_(want, dims, t, pos, pos, bits, *args)
    rows_after = kv.cache.data.clone()
    gain = (torch.rand(hidden, generator=g, device=DEV) + 0.5).to(dtype)
    for final_norm in (None, gain):
        kv.cache.data.copy_(past)
        x = x0.clone()
        array = (type(tables[0]) * len(tables))(*tables)
        rest = (kv.cache.data, ws, final_norm)
        h = ops.prefill_stack_(x, dims, array, pos, pos, *rest) if kind == "prefill" else \
            ops.decoder_stack_(x, dims, array, pos, pos, bits, *rest)
        assert torch.isfinite(x).all() and torch.equal(x, want) and torch.equal(kv.cache.data, rows_after)
        assert h is None if final_norm is None else torch.equal(h, ops.rms_norm(want, gain, 1e-6))


# widths at the ends of every number of threads and pieces per thread, row counts on both sides of the line between them
@pytest.mark.parametrize("hidden", [8, 2048, 2056, 4096, 4104, 6144, 6152, 8192, 8200, 12288, 12296, 16384])
@pytest.mark.parametrize("rows", [1, 511, 512])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_norm_at_every_width(dtype, rows, hidden):
    g = torch.Generator(device=DEV).manual_seed(hidden + rows)
    x = torch.randn(rows, hidden, generator=g, device=DEV).to(dtype)
    x[:, -8:] *= 30                                                     # a last piece that counts
    w = (torch.rand(hidden, generator=g, device=DEV) + 0.5).to(dtype)
    got = ops.rms_norm(x, w, 1e-6).double()
    xd = x.double()
    want = w.double() * (xd * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-6))
    # two roundings to 16 bits; the fp32 sum of squares and its root are off by less than 2^-16.  Half-precision values below 2^-14 are
    # spaced 2^-24: the normalized one is off by 2^-25, times a gain of up to 1.5, the product by another 2^-25
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert ((got - want).abs() <= (2.1 * eps + 2.0 ** -16) * want.abs() + 2.5 * 2.0 ** -25).all()


# a stack over a page pool in another order, with the prefix length on the host, on the device, and on the device below the launch's bound
@pytest.mark.parametrize("kind,rows", [("int4", 8), ("int4", 40), ("dense", 64), ("dense", 289)])
@pytest.mark.parametrize("loose", [None, 0, 900])
def test_stack_over_pages(kind, rows, loose):
    print("stack over pages", kind, rows, loose, flush=True)
    prefix, layers, page, hkv = 1350, 2, 16, 4
    bound = prefix + (loose or 0)
    n_pages = (bound + rows + page - 1) // page
    cfg = M.DecoderConfig(num_hidden_layers=layers, hidden_size=512, num_attention_heads=28, num_key_value_heads=hkv, head_dim=128,
                          intermediate_size=512, vocab_size=64)
    w = M.init_weights(cfg, rows, DEV, torch.bfloat16)["layers"]
    w = M.quantize_layers(w) if kind == "int4" else w
    make = ops.decoder_layer_weights if kind == "int4" else ops.dense_layer_weights
    table = ops.layer_table([make(l) for l in w])
    g = torch.Generator(device=DEV).manual_seed(rows)
    cache = torch.randn(layers, 2, 1, hkv, n_pages * page, 128, generator=g, device=DEV).bfloat16()
    order = torch.randperm(n_pages + 3, generator=torch.Generator().manual_seed(1))[:n_pages].to(DEV)
    pool = torch.full((layers, n_pages + 3, 2, page, hkv, 128), float("nan"), device=DEV, dtype=torch.bfloat16)
    for i in range(layers):
        for part in range(2):
            pool[i, order, part] = cache[i, part, 0].transpose(0, 1).reshape(n_pages, page, hkv, 128)
    x0 = torch.randn(rows, 512, generator=g, device=DEV).bfloat16()
    at = torch.arange(prefix, prefix + rows, dtype=torch.int32, device=DEV)
    bits = ops.ancestor_bits_tensor([-1] + [max(0, i - 3) for i in range(rows - 1)], device=DEV)
    gain = torch.ones(512, device=DEV, dtype=torch.bfloat16)
    out = {}
    for name, data, paging, length, dev in (
            ("tight", cache.clone(), {}, prefix, None),
            ("contiguous", cache.clone(), {}, bound, None if loose is None else torch.tensor([prefix], device=DEV)),
            ("paged", pool, dict(page_indices=order.to(torch.int32), max_pages=n_pages + 3, page_len=page), bound,
             None if loose is None else torch.tensor([prefix], device=DEV))):
        dims = ops.decoder_layer_dims(torch.bfloat16, rows, 512, 512, 28, hkv, 128, n_pages * page, length, rows, 1e-6, 1e6,
                                      prefix_len_dev=dev, **paging)
        x, ws = x0.clone(), torch.full((ops.decoder_layer_workspace(dims),), 0xff, dtype=torch.uint8, device=DEV)
        out[name] = (x, ops.decoder_stack_(x, dims, table, at, at, bits, data, ws, gain), data)
    for a, b in zip(out["paged"][:2], out["contiguous"][:2]):
        assert torch.isfinite(a).all() and torch.equal(a, b)
    written = out["paged"][2][:, order].permute(0, 2, 4, 1, 3, 5).reshape(layers, 2, 1, hkv, -1, 128)
    assert torch.equal(written, out["contiguous"][2])
    # another bound cuts the keys into other chunks: averages that differ by 2^-9 of a layer's update (a tenth of x), and with them the
    # rounding of some elements of x, by one unit of at most 2^-7 of the element; together well below 2^-8 of x
    assert (out["paged"][0] - out["tight"][0]).float().norm() <= 2.0 ** -8 * out["tight"][0].float().norm()
