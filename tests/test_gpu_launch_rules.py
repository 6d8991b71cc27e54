"""
GPU tests of the launch shapes that a call's size chooses: each gives the bits of a fixed shape or of the oracle.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from pyocean_amd import batch, ops, synth

pytestmark = pytest.mark.gpu


def _dev(case):
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()        # noqa: E731
    return d(case.C), d(case.V0), d(case.V1), d(case.Qx), d(case.Qy), d(case.ok.astype(np.uint8))


# sizes on both sides of the rule's lines (rows of 2, 4, 8, 16, 32), with a last chunk shorter than the others
@pytest.mark.parametrize("nx,ny,nz,nt", [(64, 7, 2, 1), (96, 81, 8, 2), (130, 129, 20, 2), (127, 130, 60, 2),
                                         (190, 200, 50, 2), (190, 203, 50, 6)])
@pytest.mark.parametrize("precision", ["f64", "split"])
def test_rows_chosen_by_the_size_give_the_bits_of_fixed_rows(gpu, nx, ny, nz, nt, precision):
    print("[gpu case] chunk rows", nx, ny, nz, nt, precision, flush=True)
    case = synth.regional(nx=nx, ny=ny, nz=nz, nt=nt, seed=31)
    a = _dev(case)
    got = ops.advect_fct(*a, case.dt, precision=precision)
    alone = batch.Batch([batch.Domain(*a, case.dt, precision=precision, C_alt=torch.empty_like(a[0]))])
    alone.step()
    try:
        batch.set_tuning(64, 1)
        want = ops.advect_fct(*a, case.dt, precision=precision)
    finally:
        batch.set_tuning(0, 0)
    assert torch.equal(got, want)
    assert torch.equal(alone.state(0), want)
