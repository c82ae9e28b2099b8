"""Per-group linears at the lines of the dispatch between the two tile kernels,
and the int4 weights' reordered activations on each side of it: just more and
just fewer 128 x 128 tiles than compute units, slices of a split over K, few
rows on wide N, and activations whose alignment rules the reordering out.
Bar: the per-group bar of tests/util.py against the oracle.
"""

import numpy as np
import pytest

from oracle import cider_oracle as O
from tests.util import assert_pergroup_linear_close

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import cider_amd as C

DEV = "cuda"

SHAPES = [(700, 6152, 512),   # 294 tiles
          (640, 6656, 512),   # 260
          (1024, 4096, 512),  # 256: the other side
          (512, 4096, 4096),  # four slices of K in the one-set kernel
          (40, 33032, 256)]   # one tile row, 259 tiles


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def check(y, x, w, sc, b, gs, name):
    M = x.shape[0]
    rows = np.unique(np.r_[0:4, M // 2:M // 2 + 4, M - 4:M])
    with np.errstate(invalid="ignore", over="ignore"):
        exp = O.pergroup_gemm(*O.quantize_per_token(x[rows]), w, sc.astype(np.float32), b, gs)
    assert_pergroup_linear_close(y.cpu().numpy()[rows], x[rows], w, sc, b, gs, exp, name)


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("gs", [64, 128])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int4(M, N, K, gs, special):
    x = O.synth_activations(M, K, M + gs)
    w = np.random.default_rng(M).integers(-8, 8, (N, K), dtype=np.int8)
    sc = O.synth_scales((K // gs, N), N).astype(np.float16)
    if special:  # tiles that take the exact chain
        sc[0, 3], sc[K // gs - 1, N - 2], sc[1, N // 2] = np.inf, np.nan, -np.inf
    b = (np.random.default_rng(5).standard_normal(N) * 0.1).astype(np.float16)
    y = C.w4a8_pergroup_linear(T(x), T(O.pack_w4_lo_first(w)), T(sc), gs, T(b))
    check(y, x, w, sc, b, gs, f"w4g{gs} {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K", [(700, 6152, 512), (512, 4096, 4096)])
def test_int4_unaligned_activations(M, N, K):
    gs = 64
    x = O.synth_activations(M, K, 7)
    w = np.random.default_rng(8).integers(-8, 8, (N, K), dtype=np.int8)
    sc = O.synth_scales((K // gs, N), 9).astype(np.float16)
    buf = torch.empty(M * K + 1, dtype=torch.float16, device=DEV)
    xt = buf[1:].view(M, K)
    xt.copy_(T(x))
    y = C.w4a8_pergroup_linear(xt, T(O.pack_w4_lo_first(w)), T(sc), gs)
    check(y, x, w, sc, None, gs, f"w4g{gs} unaligned {M}x{N}x{K}")


@pytest.mark.parametrize("gs", [64, 128, 256])
@pytest.mark.parametrize("M,N,K", SHAPES[:3])
def test_int8(M, N, K, gs):
    x = O.synth_activations(M, K, M + gs)
    w = O.synth_weights_i8(N, K, 3)
    sc = O.synth_scales((K // gs, N), 4)
    b = (np.random.default_rng(6).standard_normal(N) * 0.1).astype(np.float16)
    y = C.pergroup_linear(T(x), T(w), T(sc), gs, T(b))
    check(y, x, w, sc, b, gs, f"pg{gs} {M}x{N}x{K}")
