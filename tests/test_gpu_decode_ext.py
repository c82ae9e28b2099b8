"""The decode step's longer fusions against the launches they replace, bit for
bit: cider_gate_up_mv against the (RMSNorm and) gate + up MV and SwiGLU, and
RMSNorm inside an MV of two rows per wave against the two launches.
"""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import cider_amd as C
    from cider_amd import fused as F

DEV = "cuda"


def linear(N, K, g, bias):
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=DEV, generator=g)
    s = torch.rand(N, device=DEV, generator=g) * 2e-3 + 1e-4
    b = torch.randn(N, device=DEV, generator=g).half() if bias else None
    return C.CiderLinear(w, s, 0, K, N, b)


def bits(t):
    return t.view(torch.int16)


# every K of the table; I of one output, a ragged wave and workgroup, and both
# row counts of K = 4096 (the wider one from 24 outputs per compute unit on)
@pytest.mark.parametrize("mode", ["plain", "norm", "addnorm"])
@pytest.mark.parametrize("I,K", [(1, 1024), (7, 1024), (1037, 2048), (6144, 2048), (9, 3072),
                                 (6143, 4096), (6145, 4096), (12288, 4096), (33, 5120),
                                 (10, 6144), (11, 7168), (500, 8192)])
def test_gate_up_mv(I, K, mode):
    g = torch.Generator(device=DEV).manual_seed(I + K)
    lin = linear(2 * I, K, g, bias=mode != "norm")
    x = torch.randn(1, K, device=DEV, generator=g).half()
    add = torch.randn(1, K, device=DEV, generator=g).half() if mode == "addnorm" else None
    nw = None if mode == "plain" else torch.rand(K, device=DEV, generator=g).half() + 0.5
    h, y = F.gate_up_mv(x, lin, nw, 1e-6, add)
    if nw is None:
        h2, gu = x, lin(x)
    else:
        r = F.rmsnorm_quantize(x, nw, 1e-6, add=add, want_q=False)
        h2, gu = r.h, lin(r.y)
    y2, _, _ = F.silu_mul_quantize(gu, want_q=False) if I % 8 == 0 else (None, None, None)
    if y2 is None:  # the SwiGLU kernel takes multiples of 8
        pad = (-I) % 8
        two = torch.nn.functional.pad(gu.view(2, I), (0, pad)).reshape(1, -1).contiguous()
        y2 = F.silu_mul_quantize(two, want_q=False)[0][:, :I]
    assert torch.equal(bits(h), bits(h2))
    assert torch.equal(bits(y), bits(y2.contiguous()))


def test_gate_up_mv_not_taken():
    g = torch.Generator(device=DEV).manual_seed(1)
    lin = linear(64, 1280, g, False)
    assert F.gate_up_mv(torch.zeros(1, 1280, dtype=torch.float16, device=DEV), lin) is None
    lin = linear(64, 1024, g, False)
    off = torch.zeros(1025, dtype=torch.float16, device=DEV)[1:].view(1, 1024)
    assert F.gate_up_mv(off, lin) is None


@pytest.mark.parametrize("N", [6136, 6144, 6149, 8192])
def test_rmsnorm_mv_rows_per_wave(N):
    g = torch.Generator(device=DEV).manual_seed(N)
    lin = linear(N, 4096, g, True)
    x = torch.randn(1, 4096, device=DEV, generator=g).half()
    nw = torch.rand(4096, device=DEV, generator=g).half() + 0.5
    _, y = F.rmsnorm_mv(x, nw, 1e-6, lin)
    y2 = lin(F.rmsnorm_quantize(x, nw, 1e-6, want_q=False).y)
    assert torch.equal(bits(y), bits(y2))
