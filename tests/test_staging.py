"""
The host side of the page-locked transfers (no GPU): a read-only array, as an ordinary step's broadcast mask is, goes
through without a warning and keeps its values.
"""
from __future__ import annotations

import warnings

import numpy as np
import pytest
import torch

from pyocean_amd.staging import Staging


@pytest.mark.parametrize("make", [lambda: np.arange(24.0).reshape(2, 3, 4),
                                  lambda: np.broadcast_to(np.arange(24) % 3 == 0, (24,)).view(np.uint8),
                                  lambda: np.empty((0, 3))])
def test_read_only_arrays_pass_without_a_warning(make):
    a = make()
    a.flags.writeable = False
    torch.set_warn_always(True)                # torch warns of a read-only array once per process otherwise
    try:
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            t = Staging().up(a, torch.device("cpu"))
    finally:
        torch.set_warn_always(False)
    assert t.shape == a.shape and np.array_equal(t.numpy(), a)
