"""The ping-pong GEMM (cider_amd/csrc/gemm_pp.hip) at the sizes where its
tiling can go wrong: one, one and a partial, and several rounds of tiles of
each height, tiles moved inside at ragged rows and columns, rows and columns
left to small tiles, even and odd numbers of k-stages, the shortest K.

Bit-exact: the integer accumulators come from float64 products (exact below
2^53), and the epilogue's three binary32 operations are done one by one.
"""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import cider_amd as C

DEV = "cuda"

# (M, N, K); on 256 compute units, tile rows (big, small):
SHAPES = [
    (64, 256, 512),       # the smallest it takes; these three run LDS-DMA tiles
    (100, 520, 640),
    (193, 2056, 1152),
    (1000, 6152, 512),    # 128 rows
    (1334, 6152, 640),    # 192 rows, one round
    (3455, 6152, 512),    # 192 rows, several rounds
    (1000, 12296, 640),   # 256 rows, one round
    (2500, 10248, 1152),  # 256 rows, several rounds
    (4096, 2056, 640),    # 192, then 64 for the last rows
    (1601, 6152, 640),    # 192, then 128
    (1601, 12296, 512),   # the same in two rounds
    (2049, 6152, 640),    # 256, then 64
    (2049, 12296, 512),
    (3455, 12288, 640),   # 256, then 128
    (4096, 12296, 640),   # 256 rows, the last columns in tiles of 128 rows
]

# 64-row tiles: rows moved inside, whole and ragged columns; int8 and int4 weights
# (tests/test_gemm_tiles.py holds which kernel and tiles every shape here selects)
NARROW = [(257, 12288, 512), (319, 12280, 640), (320, 12296, 2048), (129, 18944, 3584),
          (192, 18936, 1152)]

# one, two and three k-stages per tile, several tiles per workgroup: the scales of
# up to four tiles are held at once
SHORT = [(2500, 10248, 128), (4096, 4096, 128), (2049, 12296, 256), (4000, 8200, 384),
         (100, 65544, 256)]


def ints(shape, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(-128, 128, shape, dtype=torch.int8, device=DEV, generator=g)


def exact_product(a, b):
    return a.double() @ b.double().t().contiguous()


@pytest.mark.parametrize("M,N,K", SHAPES + NARROW + SHORT)
def test_int32_product(M, N, K):
    a, b = ints((M, K), 1), ints((N, K), 2)
    a[0], b[-1] = -128, -128  # the largest sums
    out = C.int8_matmul_int32(a, b)
    assert torch.equal(out.double(), exact_product(a, b))


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES + NARROW + SHORT)
def test_perchannel_epilogue(M, N, K, bias):
    g = torch.Generator(device=DEV).manual_seed(3)
    q, w = ints((M, K), 4), ints((N, K), 5)
    sa = torch.rand(M, device=DEV, generator=g) * 0.02 + 1e-3
    sw = torch.rand(N, device=DEV, generator=g) * 1e-2 + 1e-4
    sa[M - 1] = float("inf")  # an infinite row: inf, and NaN where the sum is 0
    b = torch.randn(N, device=DEV, generator=g).half() if bias else None
    y = C.perchannel_gemm(q, sa, w, sw, b)
    e = exact_product(q, w).float() * sa[:, None]
    e = e * sw
    if bias:
        e = e + b.float()
    e = e.half()
    assert torch.equal(y.view(torch.int16)[~e.isnan()], e.view(torch.int16)[~e.isnan()])
    assert torch.equal(y.isnan(), e.isnan())


@pytest.mark.parametrize("M,N,K", SHAPES + NARROW + SHORT + [(65, 256, 512), (777, 4104, 4096)])
def test_int4_weights(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(6)
    x = torch.randn(M, K, device=DEV, generator=g).half()
    x[0] *= 1e-5   # a row of fp16 subnormals: the smallest scales
    x[M - 1] = 0
    w = torch.randint(-8, 8, (N, K), dtype=torch.int8, device=DEV, generator=g)
    w[N - 1] = -8
    sw = torch.rand(N, device=DEV, generator=g) * 0.1 + 1e-3
    u = w.to(torch.uint8) & 15
    packed = (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous()
    y = C.w4a8_linear_packed(x, packed, sw)
    q, sa = C.quantize_per_token(x)  # pinned to the oracle elsewhere
    e = exact_product(q, w).float() * sa[:, None]
    e = (e * sw).half()
    assert torch.equal(y.view(torch.int16), e.view(torch.int16))


# bf16: the fp16 result rounded once more, on every tile height
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K", NARROW + SHORT + SHAPES[3:])
def test_bf16(M, N, K, bias):
    g = torch.Generator(device=DEV).manual_seed(7)
    x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    w = ints((N, K), 8)
    sw = torch.rand(N, device=DEV, generator=g) * 1e-2 + 1e-4
    b = torch.randn(N, device=DEV, generator=g).half() if bias else None
    y = C.perchannel_linear(x, w, sw, b)
    q, sa = C.quantize_per_token(x.half())
    e = exact_product(q, w).float() * sa[:, None]
    e = e * sw
    e = (e + (b.float() if bias else 0.0)).half().bfloat16()
    assert torch.equal(y.view(torch.int16), e.view(torch.int16))
