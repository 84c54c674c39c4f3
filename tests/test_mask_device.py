"""The mask's length kernel runs on the mask's own GPU, which need not be the
current one (its lengths then go to the inputs' device)."""

from __future__ import annotations

import contextlib

import torch

from kda import utils


def test_length_kernel_runs_on_the_masks_device(monkeypatch):
    current, launched = [], []

    @contextlib.contextmanager
    def device(d):
        current.append(d)
        yield
        current.pop()

    class Library:
        @staticmethod
        def kda_mask_lengths(*args):
            launched.append(list(current))
            return 0

    mask = torch.ones(3, 4, dtype=torch.bool)
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(utils._lib, "load", lambda: Library)
    monkeypatch.setattr(utils._lib, "stream_of", lambda d: None)
    assert utils._device_lengths(mask).shape == (3,)
    assert launched == [[mask.device]] and not current
