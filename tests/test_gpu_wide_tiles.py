"""128 x 256 LDS-DMA tiles in several rounds, which shapes run that the ping-pong
kernel does not take: ragged N and K, int8 and int4 weights, against integer
products in float64.
"""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import cider_amd as C

DEV = "cuda"

# more than 256 tiles; ragged N (one column over, one short of 8), K of a part of a
# k-stage, one and a part, many
SHAPES = [(3000, 4097, 160), (2300, 4095, 288), (2100, 4100, 1056), (4096, 4104, 416)]


def ints(shape, lo, hi, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(lo, hi, shape, dtype=torch.int8, device=DEV, generator=g)


def product(a, b):
    return a.double() @ b.double().t().contiguous()


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int8(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(1)
    q, w = ints((M, K), -128, 128, 2), ints((N, K), -128, 128, 3)
    e = product(q, w)
    assert torch.equal(C.int8_matmul_int32(q, w).double(), e)
    sa = torch.rand(M, device=DEV, generator=g) * 0.02 + 1e-3
    sw = torch.rand(N, device=DEV, generator=g) * 1e-2 + 1e-4
    b = torch.randn(N, device=DEV, generator=g).half()
    y = C.perchannel_gemm(q, sa, w, sw, b)
    e = e.float() * sa[:, None]
    e = (e * sw + b.float()).half()
    assert torch.equal(y.view(torch.int16), e.view(torch.int16))


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int4(M, N, K, dtype):
    g = torch.Generator(device=DEV).manual_seed(4)
    x = torch.randn(M, K, device=DEV, generator=g).to(getattr(torch, dtype))
    w = ints((N, K), -8, 8, 5)
    sw = torch.rand(N, device=DEV, generator=g) * 0.1 + 1e-3
    u = w.to(torch.uint8) & 15
    packed = (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous()
    y = C.w4a8_linear_packed(x, packed, sw)
    q, sa = C.quantize_per_token(x.half())
    e = product(q, w).float() * sa[:, None]
    e = (e * sw).half().to(x.dtype)
    assert torch.equal(y.view(torch.int16), e.view(torch.int16))
