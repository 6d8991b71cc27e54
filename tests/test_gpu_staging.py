"""
GPU tests of the page-locked transfers: array sizes around the direct limit and the ends of the chunks, both ways, with
the host array changed right after the call, and several threads on one component's buffers.
"""
from __future__ import annotations

import copy
import threading

import numpy as np
import pytest
import torch

from pyocean_amd import staging

pytestmark = pytest.mark.gpu

D, C = staging.DIRECT // 8, staging.CHUNK // 8


@pytest.mark.parametrize("n", [1, D, D + 1, C - 1, C, C + 1, 2 * C, 2 * C + 1, 5 * C + 3])
@pytest.mark.parametrize("dtype", [np.float64, np.uint8])
def test_values_go_there_and_back(gpu, n, dtype):
    print("[gpu case] staging", n, dtype.__name__, flush=True)
    s = copy.deepcopy(staging.Staging())
    a = (np.arange(n) * 7 % 251).astype(dtype)
    want = a.copy()
    t = s.up(a, gpu)
    a[:] = 0                                   # the caller's array is free again
    assert torch.equal(t.cpu(), torch.from_numpy(want))
    back = s.down(t)
    t.zero_()
    assert back.dtype == dtype and np.array_equal(back, want)


def test_threads_take_turns(gpu):
    print("[gpu case] staging threads", flush=True)
    s, bad = staging.Staging(), []

    def work(m):
        with torch.cuda.stream(torch.cuda.Stream()):
            for r in range(4):
                a = np.full(2 * C + 17 * m + r, float(10 * m + r))
                if not np.array_equal(s.down(s.up(a, gpu)), a):
                    bad.append((m, r))
    threads = [threading.Thread(target=work, args=(m,)) for m in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_a_step_takes_read_only_arrays_without_a_warning(gpu):
    import warnings

    from pyocean_amd import synth
    from pyocean_amd.tracers import OpenEdges, TracerAdvection
    print("[gpu case] read-only arrays", flush=True)
    case = synth.regional(nx=70, ny=60, nz=5, nt=2, seed=3)
    adv = TracerAdvection(scheme="weno5", time="ssprk3", dt=case.dt, ob=OpenEdges(()))
    args = [case.C.copy(), case.V0, case.V1, case.Qx, case.Qy, np.ascontiguousarray(case.ok, bool)]
    want = adv.advect_fct(*args)
    args[0].flags.writeable = False
    torch.set_warn_always(True)
    try:
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            got = adv.advect_fct(*args)
    finally:
        torch.set_warn_always(False)
    assert np.array_equal(got, want)
