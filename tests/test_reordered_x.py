"""The order in which quantized activations are written for one int4 kernel (even k
of a block, then odd k) never meets another kernel: every launcher that would hand
such x to a kernel that reads k in order answers an error instead.

The launchers are internal; they are called by their C++ names with made-up
addresses, and only in cases that they have to turn down before any launch."""

import ctypes

import pytest

from cider_amd import _lib

INVALID = 1  # hipErrorInvalidValue
I8, I4 = 0, 1
I32, PC, PG = 0, 1, 2


class GemmArgs(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("x", "w", "sa", "sw", "bias", "y")] + [
        (n, ctypes.c_int) for n in ("M", "N", "K", "x_il")] + [
        (n, ctypes.c_bool) for n in ("y_bf16", "x_bf16")]


def args(M, N, K, il, **off):
    a = {n: 1 << 20 for n in ("x", "w", "sa", "sw", "y")}
    return GemmArgs(**{n: v + off.get(n, 0) for n, v in a.items()}, bias=None, M=M, N=N, K=K,
                    x_il=il)


def call(name, types, a, *rest):
    f = getattr(_lib.load(), name)
    f.restype, f.argtypes = ctypes.c_int, [ctypes.POINTER(GemmArgs), *types]
    return f(ctypes.byref(a), *rest)


_i, _b, _p = ctypes.c_int, ctypes.c_bool, ctypes.c_void_p

BIG = (2048, 12288, 4096)  # the ping-pong kernel, and the one-set per-group kernel


@pytest.mark.parametrize("wf,epi,M,N,K,il,off", [
    (I4, PC, 2, 4096, 4096, 32, {}),         # GEMV
    (I4, PC, 16, 4096, 4096, 32, {}),        # weight streams
    (I4, PC, 40, 4096, 4096, 32, {}),        # few rows
    (I4, PC, 64, 12288, 4096, 32, {}),       # LDS-DMA tiles
    (I4, PC, 100, 520, 640, 32, {}),         # small LDS-DMA tiles ahead of the ping-pong kernel
    (I4, PC, 2048, 12287, 4096, 32, {}),     # ragged
    (I4, PC, 2048, 12288, 416, 32, {}),      # no whole k-stages
    (I4, PC, *BIG, 16, {}),                  # the other kernel's order
    (I4, PC, *BIG, 32, {"y": 2}),
    (I4, PC, *BIG, 32, {"x": 8}),
    (I8, PC, *BIG, 32, {}),                  # int8 weights: in order only
    (I8, I32, *BIG, 32, {}),
    (I4, PG, 2, 4096, 4096, 16, {}),
    (I4, PG, 16, 4096, 4096, 16, {}),
    (I4, PG, 40, 4096, 4096, 16, {}),
    (I4, PG, 256, 4096, 4096, 16, {}),       # the two-set kernel
    (I4, PG, 2048, 12284, 4096, 16, {}),
    (I4, PG, *BIG, 32, {}),
    (I4, PG, *BIG, 16, {"y": 8}),
    (I8, PG, *BIG, 16, {}),
])
def test_launch_gemm_turns_it_down(wf, epi, M, N, K, il, off):
    rc = call("_ZN5cider11launch_gemmERKNS_8GemmArgsEiibiP12ihipStream_t", [_i, _i, _b, _i, _p],
              args(M, N, K, il, **off), wf, epi, wf == I4, 128 if epi == PG else 0, None)
    assert rc == INVALID


@pytest.mark.parametrize("M,N,K,il", [(100, 520, 640, 32), (*BIG, 16)])
def test_lds_dma_tiles_turn_it_down(M, N, K, il):
    rc = call("_ZN5cider15launch_gemm_dmaERKNS_8GemmArgsEiiP12ihipStream_t", [_i, _i, _p],
              args(M, N, K, il), PC, I4, None)
    assert rc == INVALID


@pytest.mark.parametrize("wf,M,N,K,il", [(I4, 256, 4096, 4096, 16), (I4, *BIG, 32), (I8, *BIG, 16)])
def test_per_group_tiles_turn_it_down(wf, M, N, K, il):
    rc = call("_ZN5cider18launch_gemm_dma_pgERKNS_8GemmArgsEibiP12ihipStream_t", [_i, _b, _i, _p],
              args(M, N, K, il), 128, wf == I4, wf, None)
    assert rc == INVALID


# slices of the two-set kernel, and of the one-set kernel in the other order or on
# int8 weights
@pytest.mark.parametrize("wf,M,N,K,il", [(I4, 128, 2560, 10240, 16), (I4, 512, 4096, 12288, 0),
                                         (I4, 512, 4096, 12288, 32), (I8, 512, 4096, 12288, 16)])
def test_split_k_slices_turn_it_down(wf, M, N, K, il):
    rc = call("_ZN5cider21launch_gemm_pg_splitkERKNS_8GemmArgsEibiiPfP12ihipStream_t",
              [_i, _b, _i, _i, _p, _p], args(M, N, K, il), 128, wf == I4, wf, 2, 1 << 21, None)
    assert rc == INVALID
