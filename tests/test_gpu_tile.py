"""GPU: the tiled dense kernels (more than 64 rows) at the edges of their tiles: one 64-k chunk, fewer chunks than ring slots,
rows and columns one past a tile, partial last tiles of the SwiGLU pairs.  Every launch shape, with one and with several row
tiles, with K whole and split: at a K of more chunks than the rings have slots, the shape checked against the plan.  Shapes
that only prompts of more than 384 rows take at full size run inside whole layers.  Outputs that are not 16-byte aligned take
the other kernel."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

from subspec_amd import _lib as L
from subspec_amd import model, ops
from subspec_amd.cache import create_kv_cache

DEV = "cuda:0"


def _ref(x, w, b):
    return x.to(DEV).double() @ w.to(DEV).double().T + b.to(DEV).double()


@pytest.mark.parametrize("M,N,K", [(65, 96, 64), (128, 160, 128), (129, 4608, 3584), (257, 1056, 192), (192, 3584, 3584),
                                   (256, 3584, 18944), (289, 3584, 18944), (289, 4608, 3584), (321, 2048, 5632), (384, 32, 320),
                                   (300, 152064, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_linear(M, N, K, dtype):
    print("tile linear", M, N, K, dtype, flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    x, b = torch.randn(M, K, generator=g).to(dtype), torch.randn(N, generator=g).to(dtype)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype)
    got, ref = ops.dense_linear(x.to(DEV), w.to(DEV), b.to(DEV)).double(), _ref(x, w, b)
    # one rounding of the result plus fp32 sums of K products of order K^-1/2 (error below K^1/2 * 2^-24 times that)
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert ((got - ref).abs() <= ulp * ref.abs() + 1e-4).all()


@pytest.mark.parametrize("M,N,K", [(65, 64, 64), (128, 37888, 192), (192, 37888, 64), (256, 37888, 448), (289, 37888, 192),
                                   (384, 11264, 256), (257, 28672, 128), (130, 2112, 320), (289, 11264, 2048)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gate_up_silu(M, N, K, dtype):
    print("tile gate|up", M, N, K, dtype, flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    x, b = torch.randn(M, K, generator=g).to(dtype), torch.randn(N, generator=g).to(dtype)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype)
    act = ops.dense_gate_up_silu(x.to(DEV), w.to(DEV), b.to(DEV)).float()
    gate, up = _ref(x, w, b).to(dtype).float().chunk(2, dim=-1)
    want = torch.nn.functional.silu(gate).to(dtype).float() * up
    # gate and up may each land on the neighbouring value of their type (and silu' < 1.1): three roundings
    ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    assert ((act - want).abs() <= 4 * ulp * want.abs() + 2 * ulp * up.abs() * 1e-1 + 1e-4).all()


@pytest.mark.parametrize("M", [3, 40, 70, 289])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activation_over_its_range(M, dtype):
    """gate = x, up = 1 (one weight per row), so the result is round(silu(gate)): gates from both ends of the exponential, tiny
    and infinite ones, through every dense kernel with the activation in its output stage."""
    K = 128
    g = torch.Generator().manual_seed(M)
    special = torch.tensor([0.0, -0.0, 1e-30, -1e-30, 1.0, -1.0, -16.5, -60.0, -86.5, -87.4, -88.6, -88.8, -92.0, -104.0, -300.0, 88.0, 300.0,
                            60000.0, -60000.0])
    gates = torch.cat([special, torch.linspace(-90.0, 20.0, 1024), torch.randn(M * 64, generator=g) * 3])[: M * 64]
    gates = torch.cat([gates, torch.zeros(M * 64 - gates.numel())]).reshape(M, 64).to(dtype)
    x = torch.cat([gates, torch.ones(M, 1), torch.zeros(M, K - 65)], dim=1).to(dtype)
    w = torch.zeros(128, K)
    w[:64, :64] = torch.eye(64)
    w[64:, 64] = 1.0
    act = ops.dense_gate_up_silu(x.to(DEV), w.to(dtype).to(DEV)).cpu().double()
    exact = gates.double() * torch.sigmoid(gates.double())
    want = exact.to(dtype).double()
    # where the exponential leaves fp32's range the result is zero
    big = gates.double() < -88.0
    assert (act[big].abs() <= 2 * exact[big].abs()).all()
    ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    tiny = 2.0 ** (-133 if dtype == torch.bfloat16 else -24)              # the spacing of subnormal results
    assert ((act - want).abs()[~big] <= ulp * want.abs()[~big] + tiny).all()
    # an fp32 error of |gate| 2^-23 in the exponential (0.69 |gate| ulps) moves one rounding in 2^15 / |gate| (bf16), 2^12 / |gate|
    # (fp16); the values repeat, and |gate| is below 90
    assert (act != want)[~big].double().mean() <= 90 / 2 ** (15 if dtype == torch.bfloat16 else 12)


@pytest.mark.parametrize("M", [3, 40, 70, 289])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activation_of_every_gate_is_the_nearest_value(M, dtype):
    """All finite gates of the type with a normal result (gate = x, up = 1, as above) against silu in float64, rounded once: the
    correctly rounded fp32 quotient of the hardware's exponential misses no bf16 value and one fp16 value (-0.7139)."""
    K, F = 64 + 64, 64
    gates = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype)
    exact = gates.double() * torch.sigmoid(gates.double())
    normal = 2.0 ** (-126 if dtype == torch.bfloat16 else -14)
    gates = gates[gates.isfinite() & (exact.abs() >= normal) & (gates > -80)]
    count = gates.numel()
    rows = -(-count // F)
    rows = -(-rows // M) * M
    gates = torch.cat([gates, torch.ones(rows * F - count, dtype=dtype)]).view(rows, F)
    x = torch.cat([gates, torch.ones(rows, 1, dtype=dtype), torch.zeros(rows, K - F - 1, dtype=dtype)], dim=1).to(DEV)
    w = torch.zeros(2 * F, K)
    w[:F, :F] = torch.eye(F)
    w[F:, F] = 1.0
    w = w.to(dtype).to(DEV)
    got = torch.cat([ops.dense_gate_up_silu(x[i:i + M], w) for i in range(0, rows, M)]).cpu().flatten()[:count]
    gates = gates.flatten()[:count].double()
    want = (gates * torch.sigmoid(gates)).to(dtype)
    assert int((got != want).sum()) <= (0 if dtype == torch.bfloat16 else 1), gates[got != want]


def _plan(M, N, K, gate_up):
    """(tile shape, row tiles, column tiles, K ranges)"""
    plan = (ctypes.c_int32 * 4)()
    L.check(L.lib().subspec_dense_tile_plan(M, N, K, gate_up, plan), "subspec_dense_tile_plan")
    return tuple(plan)


def _tail(M, N, K):
    """(tile shape of a gate|up projection's last columns, row tiles, column tiles, first column); no such columns: (-1, 0, 0, 0)"""
    tail = (ctypes.c_int32 * 4)()
    L.check(L.lib().subspec_dense_tile_tail(M, N, K, tail), "subspec_dense_tile_tail")
    return tuple(tail)


# M, N, K; shape of the last columns, its row and column tiles (the last of them partial), its first column
@pytest.mark.parametrize("M,N,K,tail", [
    (129, 164800, 512, (2, 1, 211, 65536)), (257, 45312, 640, (4, 3, 79, 16384)), (257, 46496, 1024, (5, 2, 108, 16384))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_two_shapes_in_one_launch(M, N, K, tail, dtype):
    assert _tail(M, N, K) == tail
    test_gate_up_silu(M, N, K, dtype)


# M, N, K; tile shape, row tiles, K ranges
@pytest.mark.parametrize("M,N,K,shape,row_tiles,ranges", [
    (129, 41536, 512, 0, 1, 1), (333, 22816, 512, 0, 2, 1), (129, 20736, 5632, 0, 1, 3), (333, 7296, 18944, 0, 2, 4),
    (257, 22816, 512, 1, 1, 1), (257, 7296, 5632, 1, 1, 5), (200, 33216, 512, 2, 1, 1), (200, 16576, 3584, 2, 1, 2),
    (129, 33216, 1024, 3, 1, 1), (129, 4736, 5632, 3, 1, 7), (65, 33216, 3584, 4, 1, 1), (257, 12416, 512, 4, 3, 1),
    (65, 8256, 5632, 4, 1, 4), (300, 5856, 2048, 4, 3, 2), (129, 20736, 512, 5, 1, 1), (257, 14496, 512, 5, 2, 1),
    (129, 4576, 3584, 5, 1, 6), (257, 3616, 3584, 5, 2, 4), (257, 16576, 512, 3, 2, 1), (257, 5536, 2048, 3, 2, 3), (257, 20736, 512, 6, 3, 1), (257, 6816, 2048, 6, 3, 3),
    (65, 16576, 640, 7, 1, 1), (257, 5536, 512, 7, 3, 1), (65, 5536, 5632, 7, 1, 5), (257, 2816, 2048, 7, 3, 3),
    (65, 96, 512, 8, 1, 1), (129, 96, 512, 8, 2, 1), (65, 96, 1024, 8, 1, 2), (129, 96, 1024, 8, 2, 2),
    (300, 4608, 3584, 8, 3, 1), (300, 3584, 18944, 6, 3, 6)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_shape_of_a_linear_layer(M, N, K, shape, row_tiles, ranges, dtype):
    plan = _plan(M, N, K, 0)
    assert (plan[0], plan[1], plan[3]) == (shape, row_tiles, ranges)
    test_dense_linear(M, N, K, dtype)


@pytest.mark.parametrize("M,N,K,shape,row_tiles", [
    (129, 41536, 512, 0, 1), (333, 22816, 512, 0, 2), (333, 28672, 4096, 0, 2), (257, 22816, 512, 1, 1), (300, 37888, 3584, 1, 1),
    (200, 33216, 512, 2, 1), (129, 33216, 1024, 3, 1), (160, 37888, 3584, 3, 1), (100, 37888, 3584, 4, 1), (257, 12416, 512, 4, 3),
    (129, 20736, 512, 5, 1), (257, 14496, 512, 5, 2), (200, 28672, 4096, 5, 1), (257, 16576, 512, 3, 2), (333, 37888, 3584, 3, 2), (257, 20736, 512, 6, 3),
    (65, 16576, 640, 7, 1), (257, 5536, 512, 7, 3), (65, 96, 512, 8, 1), (129, 96, 512, 8, 2), (100, 11264, 2048, 8, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_shape_of_gate_up(M, N, K, shape, row_tiles, dtype):
    plan = _plan(M, N, K, 1)
    assert (plan[0], plan[1], plan[3]) == (shape, row_tiles, 1) and _tail(M, N, K)[0] == -1
    test_gate_up_silu(M, N, K, dtype)


# shapes of q|k|v, o, gate|up (its best alone, which is launched where no last columns follow), down; the K ranges of down; gate|up's last
# columns (behind the largest shape): at the widths of a 7B layer and of a wider one
@pytest.mark.parametrize("rows,widths,shapes,ranges,tail", [
    (2000, (3584, 28, 4, 18944), (2, 5, 0, 0), 2, (2, 8, 32, 16384)), (1000, (3584, 28, 4, 18944), (4, 7, 2, 0), 4, (4, 8, 32, 16384)),
    (1930, (4096, 32, 8, 14336), (0, 5, 0, 5), 1, (5, 8, 32, 12288)), (1590, (4096, 32, 8, 14336), (1, 5, 2, 0), 2, (-1, 0, 0, 0))])
def test_shapes_of_long_prompts(rows, widths, shapes, ranges, tail):
    """One whole layer against float32, the module-by-module path of the same dtype as the yardstick: both round at the same
    points, so neither may be twice as far off as the other, in the 2-norm and in any one element."""
    hidden, hq, hkv, mlp = widths
    sizes = [((hq + 2 * hkv) * 128, hidden, 0), (hidden, hq * 128, 0), (2 * mlp, hidden, 1), (hidden, mlp, 0)]
    plans = [_plan(rows, *s) for s in sizes]
    assert tuple(p[0] for p in plans) == shapes and plans[3][3] == ranges and _tail(rows, 2 * mlp, hidden) == tail
    cfg = model.DecoderConfig(num_hidden_layers=1, hidden_size=hidden, num_attention_heads=hq, num_key_value_heads=hkv, head_dim=128,
                          intermediate_size=mlp, vocab_size=512)
    w = model.init_weights(cfg, 1, DEV, torch.bfloat16)
    w["embed"].mul_(50.0)
    tokens = torch.randint(0, 512, (rows,), generator=torch.Generator(device=DEV).manual_seed(rows), device=DEV)
    out = {}
    with torch.no_grad():
        for name, dt, native in (("exact", torch.float32, False), ("module", torch.bfloat16, False), ("native", torch.bfloat16, True)):
            print("long prompt", rows, hidden, name, flush=True)
            kv = create_kv_cache("static", max_cache_len=rows, config=cfg, device=DEV, dtype=dt)
            layers = [{k: v.to(dt) for k, v in w["layers"][0].items()}]
            d = model.Decoder(cfg, w["embed"].to(dt), layers, w["norm"].to(dt), w["lm_head"].to(dt), kv)
            d.use_native_layers = native
            out[name] = (d.prefill(tokens, 0, all_logits=True).double(), kv.cache.data.double())
    for exact, module, native in zip(out["exact"], out["module"], out["native"]):
        assert (native - exact).norm() <= 2 * (module - exact).norm()
        assert (native - exact).abs().max() <= 2 * (module - exact).abs().max()


@pytest.mark.parametrize("M,N,K", [(70, 96, 256), (200, 96, 2048), (257, 160, 2048), (384, 3584, 3584)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_unaligned_outputs_of_every_row_count(M, N, K, dtype):
    """Two bytes past a 16-byte boundary, as only a direct caller of the library has them: dense_wide_kernel for 65 to 256 and
    for 257 to 384 rows, K whole and split, and its SwiGLU form; nothing outside the output is written."""
    g = torch.Generator().manual_seed(M + N + K)
    x, b = torch.randn(M, K, generator=g).to(dtype).to(DEV), torch.randn(N, generator=g).to(dtype).to(DEV)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype).to(DEV)
    lib, st, code = L.lib(), torch.cuda.current_stream().cuda_stream, L.BF16 if dtype == torch.bfloat16 else L.F16
    ws = torch.empty(lib.subspec_dense_linear_workspace(M, N, K), dtype=torch.uint8, device=DEV)
    ref = _ref(x, w, b)
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    room = torch.zeros(M * N + 16, dtype=dtype, device=DEV)
    L.check(lib.subspec_dense_linear(x.data_ptr(), w.data_ptr(), b.data_ptr(), room[1:].data_ptr(), code, M, N, K, ws.data_ptr(),
                                     ws.numel(), st), "subspec_dense_linear")
    assert room[:1].abs().max() == 0 and room[1 + M * N:].abs().max() == 0
    assert ((room[1:1 + M * N].view(M, N).double() - ref).abs() <= ulp * ref.abs() + 1e-4).all()      # see test_dense_linear
    F = N // 2
    room = torch.zeros(M * F + 16, dtype=dtype, device=DEV)
    L.check(lib.subspec_dense_gate_up_silu(x.data_ptr(), w.data_ptr(), b.data_ptr(), room[1:].data_ptr(), code, M, N, K, st),
            "subspec_dense_gate_up_silu")
    assert room[:1].abs().max() == 0 and room[1 + M * F:].abs().max() == 0
    gate, up = ref.to(dtype).float().chunk(2, dim=-1)
    want = torch.nn.functional.silu(gate).to(dtype).float() * up
    act = room[1:1 + M * F].view(M, F).float()
    assert ((act - want).abs() <= 8 * ulp * want.abs() + 4 * ulp * up.abs() * 1e-1 + 1e-4).all()      # see test_gate_up_silu


def test_unaligned_output_takes_the_other_kernel():
    g = torch.Generator().manual_seed(1)
    M, N, K = 70, 96, 256
    x, w = torch.randn(M, K, generator=g).bfloat16().to(DEV), (torch.randn(N, K, generator=g) / 16).bfloat16().to(DEV)
    lib = L.lib()
    ws = torch.empty(lib.subspec_dense_linear_workspace(M, N, K), dtype=torch.uint8, device=DEV)
    room = torch.zeros(M * N + 16, dtype=torch.bfloat16, device=DEV)
    L.check(lib.subspec_dense_linear(x.data_ptr(), w.data_ptr(), None, room[4:].data_ptr(), L.BF16, M, N, K, ws.data_ptr(),
                                     ws.numel(), torch.cuda.current_stream().cuda_stream), "subspec_dense_linear")
    assert room[:4].abs().max() == 0 and room[4 + M * N:].abs().max() == 0
    want = ops.dense_linear(x, w)
    assert ((room[4:4 + M * N].view(M, N).float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs() + 1e-3).all()


@pytest.mark.parametrize("rows,own", [(65, True), (97, True), (128, True), (129, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_head_over_65_to_128_rows(rows, own, dtype):
    """A head of rows of 4096 elements on the kernel that ``tiled_head`` names, against float64."""
    V, K = 128032, 4096
    assert model.tiled_head(rows, V, K) == own
    g = torch.Generator(device=DEV).manual_seed(rows)
    x = torch.randn(rows, K, generator=g, device=DEV).to(dtype)
    holder = type("Holder", (), {"lm_head": (torch.randn(V, K, generator=g, device=DEV) * K ** -0.5).to(dtype)})()
    with torch.no_grad():
        got = model.Decoder._head(holder, x).double()
    ref = x.double() @ holder.lm_head.double().T
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert ((got - ref).abs() <= ulp * ref.abs() + 1e-4).all()
