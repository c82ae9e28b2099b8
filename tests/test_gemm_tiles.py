"""Which kernel and tiles the shapes of the GEMM tests select, so that a test which
is there for a kernel cannot lose it to a change of the dispatch unseen.  The
dispatch is host code: no GPU is needed.  On 256 compute units, as it assumes
without a GPU."""

import ctypes

import pytest
import torch

import bench
from cider_amd import _lib

from .test_gpu_pp import NARROW, SHAPES, SHORT

PC, W4 = _lib.CIDER_OP_PERCHANNEL, _lib.CIDER_OP_W4A8

# (rows of the ping-pong kernel's tiles, of its small ones), or the LDS-DMA tile
BIG = {(1000, 6152, 512): (128, 0), (1334, 6152, 640): (192, 0), (3455, 6152, 512): (192, 0),
       (1000, 12296, 640): (256, 0), (2500, 10248, 1152): (256, 0), (4096, 2056, 640): (192, 64),
       (1601, 6152, 640): (192, 128), (1601, 12296, 512): (192, 128), (2049, 6152, 640): (256, 64),
       (2049, 12296, 512): (256, 64), (3455, 12288, 640): (256, 128),
       (4096, 12296, 640): (256, 128), **{s: (64, 0) for s in NARROW},
       (2500, 10248, 128): (128, 0), (4096, 4096, 128): (256, 0), (2049, 12296, 256): (128, 0),
       (4000, 8200, 384): (192, 0), (100, 65544, 256): (64, 0)}
LDS_DMA = [(100, 520, 640), (193, 2056, 1152)]


def tiles(op, shape):
    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("another number of compute units")
    out = (ctypes.c_int * 4)()
    rc = _lib.load().cider_gemm_tiles(op, *shape, out)
    return tuple(out) if rc == 0 else rc


@pytest.mark.parametrize("op", [PC, W4])
@pytest.mark.parametrize("shape", [s for s in SHAPES + NARROW + SHORT if s in BIG])
def test_ping_pong(op, shape):
    assert tiles(op, shape) == (1, BIG[shape][0], 256, BIG[shape][1])


def test_every_height_of_the_ping_pong_kernel_is_there():
    # (4, 2), (4, 1), (3, 2), (3, 1): big and small tiles; 2 and 1 alone
    assert set(BIG.values()) == {(256, 128), (256, 64), (256, 0), (192, 128), (192, 64), (192, 0),
                                 (128, 0), (64, 0)}
    assert set(SHAPES + NARROW + SHORT) == set(BIG) | set(LDS_DMA) | {(64, 256, 512)}


@pytest.mark.parametrize("op", [PC, W4])
def test_lds_dma(op):
    for shape in LDS_DMA:
        assert tiles(op, shape)[0] == 0
    assert tiles(op, (64, 256, 512)) == _lib.CIDER_E_UNSUPPORTED


# the headline shape, shapes that the ping-pong kernel does not take, and a short K in
# one round of tiles
@pytest.mark.parametrize("op,shape,expected", [
    (PC, (4096, 10240, 2560), (1, 256, 256, 128)),
    (PC, (4096, 10239, 2560), (0, 128, 256, 0)),
    (PC, (4096, 10240, 2576), (0, 128, 256, 0)),
    (W4, (4096, 10239, 2560), (0, 128, 256, 0)),
    (PC, (1000, 6152, 256), (0, 128, 256, 0)),
])
def test_selected(op, shape, expected):
    assert tiles(op, shape) == expected


# the kernel that bench.py's line names, and the traffic it attaches to that kernel only
@pytest.mark.parametrize("shape,kernel", [
    ((4096, 10240, 2560), "gemm_pp_kernel<4, 2, 1, 0> (256x256 and 128x256 tiles"),
    ((8192, 10240, 2560), "gemm_pp_kernel<4, 2, 1, 0> (256x256 tiles"),
    ((1024, 10240, 2560), "gemm_pp_kernel<3, 1, 1, 0> (192x256 and 64x256 tiles"),
    ((128, 10240, 2560), "gemm_dma_kernel<128, 64, 128, 1, 0, 4, false> (128x64 tiles"),
    ((4096, 10239, 2560), "gemm_dma_kernel<128, 256, 128, 1, 0, 8, true> (128x256 tiles"),
    ((16, 10240, 2560), "per-channel GEMM of few rows"),
])
def test_bench_names_the_kernel(shape, kernel):
    tiles(PC, shape)  # skips on another number of compute units
    name = bench.gemm_kernel_name(*shape)
    assert name.startswith(kernel)
    headline = shape == (4096, 10240, 2560)
    assert (bench.load_traffic(name, *shape) is not None) == headline
    assert bench.load_traffic("gemm_dma_mixed_kernel<1, 0, 8>", *shape) is None
