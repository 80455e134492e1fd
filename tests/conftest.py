"""Test configuration: the ``gpu`` marker and shared helpers."""

from __future__ import annotations

import ctypes
import os
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if REPO not in sys.path:
    sys.path.insert(0, REPO)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built liblastkv_amd.so")


def gpu_available() -> bool:
    import torch

    return torch.cuda.is_available()


@pytest.fixture
def prefill_plans(monkeypatch):
    """The (waves, key splits, halves, decode rows beside the tiles) lkv_prefill_plan gives for every prefill call a
    test makes (in order; the Python body makes the calls)."""

    from lastkv_amd import _lib, ops

    lib, plans = _lib.load(), []
    attn = lib.lkv_prefill_attn

    def planned(args, stream):
        info = _lib.PrefillPlanInfo()
        _lib.check(lib.lkv_prefill_plan(args, ctypes.byref(info)), "lkv_prefill_plan")
        plans.append((info.tile_waves, info.tile_splits, info.key_halves, info.rows_beside_tiles))
        return attn(args, stream)

    monkeypatch.setattr(lib, "lkv_prefill_attn", planned)
    monkeypatch.setattr(ops, "_host", None)
    monkeypatch.setattr(ops, "_host_bound", False)
    return plans


def pytest_collection_modifyitems(config, items):
    if gpu_available():
        return
    skip = pytest.mark.skip(reason="no GPU visible")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)
