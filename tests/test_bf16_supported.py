"""Which bf16 linears the library takes is known before anything is allocated."""

import ctypes

import pytest
import torch

from cider_amd import _lib, ops

PC, PG = _lib.CIDER_OP_PERCHANNEL, _lib.CIDER_OP_PERGROUP


def ptr(address):
    return ctypes.c_void_p(address)


# K around the table of the streaming MV; x, w and the scales off their alignment.
# A call that is turned down is turned down before a launch, so no GPU is needed
# (nor any memory read); the others are asked about only.
@pytest.mark.parametrize("op,gs", [(PC, 0), (PG, 64), (PG, 256)])
def test_supported_is_what_the_call_answers(op, gs):
    lib = _lib.load()
    A, seen = 1 << 20, set()
    for K in [64, 256, 512, 768, 1024, 1280, 2560, 3840, 4096, 4160, 4352, 7680, 7936, 16384, 16640]:
        if gs and K % gs:
            continue
        for dx, dw, ds in [(0, 0, 0), (2, 0, 0), (0, 1, 0), (0, 0, 2)]:
            said = lib.cider_linear_bf16_supported(op, ptr(A + dx), ptr(A + dw), ptr(A + ds), 1, K,
                                                   gs)
            seen.add(said)
            if said == 0:
                rc = lib.cider_linear_bf16(op, ptr(A + dx), ptr(A + dw), ptr(A + ds), None, ptr(A),
                                           None, 0, 1, 32, K, gs, None)
                assert rc == _lib.CIDER_E_UNSUPPORTED
            # more tokens, and int4 weights, are always taken
            assert lib.cider_linear_bf16_supported(op, ptr(A + dx), ptr(A + dw), ptr(A + ds), 2, K,
                                                   gs) == 1
            assert lib.cider_linear_bf16_supported(_lib.CIDER_OP_W4A8, ptr(A + dx), ptr(A + dw),
                                                   ptr(A + ds), 1, K, 0) == 1
    assert seen == {0, 1}


def test_nothing_is_allocated_for_a_call_that_is_not_taken(monkeypatch):
    K = 512
    x, w, s = torch.zeros(1, K).bfloat16(), torch.zeros(8, K, dtype=torch.int8), torch.zeros(8)

    def refuse(*a, **k):
        raise AssertionError("allocated")

    monkeypatch.setattr(torch, "empty", refuse)
    monkeypatch.setattr(ops, "_workspace", refuse)
    monkeypatch.setattr(ops, "_stream_ptr", lambda *a: None)
    assert ops._linear_bf16(PC, x, w, s, None, 1, 8, K, 0, "cpu", None) is None
