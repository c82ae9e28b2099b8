"""Operands at addresses that are aligned to their element only: the same results,
bit for bit, as aligned ones give (the sums are integers, or taken in the same
order on the same kernel), and nothing written outside the result.
"""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import cider_amd as C

DEV = "cuda"


def off_by_one(t):
    """t's values one element past an aligned address."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
    out = buf[1:].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 == t.element_size()
    return out


def bits(t):
    return t.view(torch.int16)


# int4 kernels that take x in an order of their own, the scalar quantization
# writing it: the ping-pong kernel (with an odd number of row blocks), the one-set
# per-group kernel, its split-K slices; and kernels that take it in order
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("fmt,M,N,K", [
    ("w4", 1334, 6152, 640), ("w4", 257, 12288, 512), ("w4", 100, 520, 640), ("w4", 5, 264, 512),
    ("w4g64", 700, 6144, 1024), ("w4g128", 2051, 2568, 512), ("w4g128", 512, 4096, 12288),
    ("w4g64", 130, 520, 1024), ("w4g128", 7, 264, 512),
    ("pc", 300, 520, 640), ("pc", 3, 264, 512), ("pc", 33, 100, 72)])
def test_x(fmt, M, N, K, dtype):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, device=DEV, generator=g).to(getattr(torch, dtype))
    x[0, 1::2] *= 50.0  # the two halves of a block differ
    if fmt == "pc":
        w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=DEV, generator=g)
        s = torch.rand(N, device=DEV, generator=g) * 1e-2 + 1e-4
        layer = C.CiderLinear(w, s, 0, K, N)
    elif fmt == "w4":
        w = torch.randint(0, 256, (K // 2, N), device=DEV, generator=g).to(torch.uint8)
        layer = C.W4A8Linear(w, torch.rand(N, device=DEV, generator=g) * 0.1 + 1e-3, K)
    else:
        gs = int(fmt[3:])
        w = torch.randint(0, 256, (N, K // 2), device=DEV, generator=g).to(torch.uint8)
        s = (torch.rand(K // gs, N, device=DEV, generator=g) * 0.1 + 1e-3).half()
        layer = C.W4A8GroupLinear(w, s, gs)
    assert torch.equal(bits(layer(off_by_one(x))), bits(layer(x)))
