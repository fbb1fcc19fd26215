"""Which calls of moe_layer hand the grouped kernels x' pairs (CPU: the launches are stand-ins)."""

from __future__ import annotations

import types

import pytest
import torch

from maple_amd import moe


@pytest.mark.parametrize("inter,n_exp,tokens,expect", [
    (4352, 8, 4, True), (4352, 8, 16, True), (4352, 8, 17, False),  # 16 pairs an expert, and one token past
    (4096, 8, 16, False), (768, 64, 32, False), (5120, 256, 64, True)])
def test_moe_layer_passes_pairs_where_the_kernels_read_them(monkeypatch, inter, n_exp, tokens, expect):
    """Decode batches with rows past a tile (4096 values) run the K-split kernels,
    which otherwise build x's operands in every workgroup; no other form reads
    the pairs."""
    seen = {}

    def route(x, layer, top_k, norm_weight, eps, add=None, *, pairs=False):
        seen["pairs"] = pairs
        return ("h", x, "ids", "wts", "d") + ((("xp", "xc"),) if pairs else ())

    def grouped(x, layer, ids, wts, residual=None, *, dispatch=None, x_pairs=None, combine=True):
        seen.update(x_pairs=x_pairs, residual=residual, dispatch=dispatch, combine=combine)
        return "y"

    monkeypatch.setattr(moe, "moe_route", route)
    monkeypatch.setattr(moe, "moe_grouped", grouped)
    layer = types.SimpleNamespace(gate_weight=torch.empty(n_exp, 2048, dtype=torch.bfloat16), n_experts=n_exp,
                                  hidden=2048, inter=inter)
    x = torch.empty(tokens, 2048, dtype=torch.bfloat16)
    assert moe.moe_layer(x, layer, 8, None, 1e-6, defer_combine=True) == ("y", "ids")
    assert seen == {"pairs": expect, "x_pairs": ("xp", "xc") if expect else None, "residual": "h", "dispatch": "d",
                    "combine": False}
