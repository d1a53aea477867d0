"""The autotuner's cache file on the CPU: which stored shapes are applied."""

import hashlib
import json

import torch

from blade_amd import autotune

TUNING = {"time_samples_per_lane": 4, "beam_tiles": 1, "chunks_per_item": 8, "workgroups_per_cu": 2}


def _blocks():
    return [(torch.zeros((4, 2, 64, 2, 2), dtype=torch.int8), torch.zeros((3, 4, 2, 1, 2), dtype=torch.complex64), None)]


def _store(path, sig):
    path.write_text(json.dumps({sig: {"tuning": TUNING, "ms": 1.0, "shapes": [[4, 2, 64, 3]], "precision": "f32"}}))


def test_shapes_of_earlier_kernels_are_not_applied(tmp_path, monkeypatch):
    monkeypatch.setenv("BLADE_AMD_CACHE", str(tmp_path))
    shapes = [(4, 2, 64, 3)]
    earlier = hashlib.sha1(json.dumps({"precision": "f32", "shapes": [list(s) for s in shapes]}).encode()).hexdigest()
    _store(tmp_path / "autotune.json", earlier)          # as written before the key named the kernels
    assert autotune.cached_tuning(_blocks(), "f32") is None
    _store(tmp_path / "autotune.json", autotune.signature(shapes, "f32"))
    assert autotune.cached_tuning(_blocks(), "f32") == TUNING
