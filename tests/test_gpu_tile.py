"""GPU: the tiled dense kernels (more than 64 rows) at the edges of their tiles and for every launch shape the plan can
choose: one 64-k chunk, fewer chunks than ring slots, rows and columns one past a tile, K split over workgroups, partial
last tiles of the SwiGLU pairs, an output that is not 16-byte aligned (which takes the other kernel)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from subspec_amd import _lib as L
from subspec_amd import ops

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
