"""Ragged widths and lengths on the kernels that stream whole 16-byte chunks:
N of any residue (rows of the output at any alignment, a last store that is cut
off) and K that ends inside a 128-k stage (the last stage then begins inside
the one before), for every tile and the few-row kernels; and the M == 1 MV
whose last block is part filled.

Bit-exact: the integer accumulators come from float64 products (exact below
2^53) and the epilogue's binary32 operations are done one by one; the MV is
compared with the oracle's order.
"""

import numpy as np
import pytest

from oracle import cider_oracle as O
from tests.util import assert_bits_equal

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import cider_amd as C

DEV = "cuda"

# (M, N, K): K % 128 of 16, 32, 64, 96, 112 and 0; N % 8 of 1 .. 7
SHAPES = [(2, 37, 144), (3, 509, 1056), (12, 1021, 4160), (16, 5, 960), (24, 4095, 1008),
          (49, 515, 448), (64, 12283, 160), (65, 1, 128), (96, 509, 5952), (100, 1847, 896),
          (129, 3, 608), (300, 2049, 144), (300, 6149, 1120), (700, 4095, 4096),
          (1334, 1023, 1632), (2940, 509, 1088), (1100, 4090, 2016)]


def ints(shape, seed, lo=-128, hi=128):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(lo, hi, shape, dtype=torch.int8, device=DEV, generator=g)


def exact_product(a, b):
    return a.double() @ b.double().t().contiguous()


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int32_product(M, N, K):
    a, b = ints((M, K), 1), ints((N, K), 2)
    a[0], b[-1] = -128, -128  # the largest sums
    assert torch.equal(C.int8_matmul_int32(a, b).double(), exact_product(a, b))


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
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


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int4_weights(M, N, K, dtype):
    g = torch.Generator(device=DEV).manual_seed(6)
    x = torch.randn(M, K, device=DEV, generator=g).to(dtype)
    w = ints((N, K), 7, -8, 8)
    w[N - 1] = -8
    sw = torch.rand(N, device=DEV, generator=g) * 0.1 + 1e-3
    u = w.to(torch.uint8) & 15
    packed = (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous()
    y = C.w4a8_linear_packed(x, packed, sw)
    q, sa = C.quantize_per_token(x.half())  # pinned to the oracle elsewhere
    e = exact_product(q, w).float() * sa[:, None]
    e = (e * sw).half().to(dtype)
    assert torch.equal(y.view(torch.int16), e.view(torch.int16))


# 4, 6, 8 and 16 blocks in flight; a last block of one chunk and of all but one
@pytest.mark.parametrize("gs", [0, 64])
@pytest.mark.parametrize("N,K", [(7, 64), (1001, 320), (4095, 1088), (509, 3008), (2050, 2880),
                                 (33, 4160), (9000, 4032), (130, 16320)])
def test_mv(N, K, gs):
    x = O.synth_activations(1, K, N)
    w = O.synth_weights_i8(N, K, N + 1)
    sw = O.synth_scales((K // gs, N) if gs else N, N + 2)
    b = (np.random.default_rng(N).standard_normal(N) * 0.1).astype(np.float16)
    t = [torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for v in (x, w, sw, b)]
    y = C.pergroup_linear(*t[:3], gs, t[3]) if gs else C.perchannel_linear(*t)
    e = O.mv_pergroup(x, w, sw, b, gs) if gs else O.mv_perchannel(x, w, sw, b)
    assert_bits_equal(y.cpu().numpy().reshape(-1), np.asarray(e).reshape(-1), f"mv {N}x{K} gs {gs}")


@pytest.mark.parametrize("K", [16, 48, 1040, 4112])
def test_mv_few_chunks(K):
    x = O.synth_activations(1, K, K)
    w = O.synth_weights_i8(65, K, K + 1)
    sw = O.synth_scales(65, K + 2)
    t = [torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for v in (x, w, sw)]
    e = O.mv_perchannel(x, w, sw, np.zeros(65, np.float16))
    assert_bits_equal(C.perchannel_linear(*t).cpu().numpy().reshape(-1),
                      np.asarray(e).reshape(-1), f"mv 65x{K}")
