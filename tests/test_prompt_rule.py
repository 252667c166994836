"""Which calls take the wide products of long prompts (the rules alone: no GPU, nothing launched)."""
import ctypes

import pytest
import torch

from drama3 import _lib, formats, kernels

FMTS = [formats.FMT_I8, formats.FMT_W4, formats.FMT_W6, formats.FMT_F8]
# (T, topk, E, FFN): a shared expert and other few experts, whose wide products would be a few workgroups
FEW = [(34, 1, 1, 768), (256, 1, 1, 768), (1024, 1, 1, 512), (512, 2, 4, 768), (128, 2, 8, 768), (511, 4, 16, 512)]
# few pairs per expert, and none
SHORT = [(256, 8, 128, 768), (33 * 16, 8, 128, 768), (900, 8, 256, 512), (1, 8, 128, 768)]
LONG = [(1000, 8, 128, 768), (2391, 8, 256, 512), (8192, 8, 128, 768), (4096, 1, 1, 768), (512, 4, 16, 512),
        (272, 8, 64, 768)]


def a8_wide(fmt, T, topk, E, inter, **pointers):
    desc = _lib.MoeA8PrefillDesc(format=fmt, T=T, topk=topk, E=E, H=2048, I=inter, **pointers)
    return bool(_lib.lib().d3_moe_a8_prefill_wide(ctypes.byref(desc)))


@pytest.mark.parametrize("fmt", FMTS)
def test_a8_prefill_rule(fmt):
    for call in FEW + SHORT:
        assert not a8_wide(fmt, *call), call
    for call in LONG:
        assert a8_wide(fmt, *call), call
        for pointer in ("gate_up", "down", "workspace"):
            assert a8_wide(fmt, *call, **{pointer: 1024 + 16}) and not a8_wide(fmt, *call, **{pointer: 1024 + 8}), call
    assert not a8_wide(fmt, 2 ** 20, 8, 128, 768)  # hidden rows past 2^32 bytes


@pytest.mark.parametrize("kind", ["int8", "fp8", "w4", "w6"])
def test_resident_prefill_rule(kind):
    weight = "weight" if kind == "fp8" else "_qdata"

    def wide(T, topk, E, inter, offset=0):
        bank = {weight: torch.empty(64, dtype=torch.uint8)[offset:], "scale": torch.empty(4)}
        return kernels.prompt_wide_fits(kind, (bank, bank), (2 * inter, 2048), T * topk, E, 2048)

    for call in FEW + [(256, 8, 128, 768), (900, 8, 256, 512), (1, 8, 128, 768), (0, 8, 128, 768)]:
        assert not wide(*call), call
    for call in LONG:
        assert wide(*call) and not wide(*call, offset=8), call
    assert not wide(1000, 8, 128, 384) and not wide(1000, 8, 32, 200)  # rows not in whole tiles
