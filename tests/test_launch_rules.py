"""
The launch shapes that a call's size chooses (host computations, no GPU).
"""
from __future__ import annotations

import pytest

from pyocean_amd import _native
from pyocean_amd._native import OcxDomain


def _domains(*shapes):
    d = (OcxDomain * len(shapes))()
    for q, (nx, ny, nz, nt) in enumerate(shapes):
        d[q].nx, d[q].ny, d[q].nz, d[q].nt = nx, ny, nz, nt
    return d


BASIN, BAY, COAST = (96, 80, 8, 2), (198, 159, 50, 1), (300, 250, 30, 4)


# 64 rows with one tracer a workgroup or a full chip, 32 with two, less while the chip has fewer chunks than units
@pytest.mark.parametrize("shapes,wpg,rows", [
    ([BASIN], 0, 8), ([BASIN] * 4, 0, 16), ([BASIN] * 16, 0, 32), ([BASIN] * 64, 0, 32), ([BASIN] * 8, 1, 64),
    ([BAY], 0, 64), ([BAY] * 2, 0, 64), ([BAY] * 8, 0, 64), ([COAST] * 2, 0, 32), ([COAST] * 2, 1, 64),
    ([(96, 80, 8, 1)] * 4, 0, 16), ([(96, 80, 8, 1), (198, 159, 50, 3)], 0, 32), ([(1024, 1024, 50, 10)], 0, 64),
    ([(1, 1, 1, 1)], 0, 8)])
def test_batch_rows(shapes, wpg, rows):
    assert _native.lib().ocx_batch_rows(_domains(*shapes), len(shapes), wpg) == rows


def test_batch_rows_refuses_what_create_refuses():
    L = _native.lib()
    assert L.ocx_batch_rows(_domains((0, 1, 1, 1)), 1, 0) == _native.OCX_E_ARG
    assert L.ocx_batch_rows(_domains(BASIN), 1, 9) == _native.OCX_E_ARG
    assert L.ocx_batch_rows(None, 0, 0) == _native.OCX_E_ARG


# the history of bundled iterations costs a large grid nothing: every iteration has a launch of its own there
@pytest.mark.parametrize("nx,ny,columns", [(197, 159, 12), (384, 383, 3), (511, 513, 0), (1024, 1024, 0)])
def test_ppm_workspace_holds_the_history_of_one_bundle(nx, ny, columns):
    L = _native.lib()
    for axis, cols in ((0, ny * (nx + 1)), (1, (ny + 1) * nx)):
        size = [int(L.ocx_ppm_transport_workspace_bytes(50, ny, nx, axis, m)) for m in (8, 20)]
        want = columns * cols * 8
        assert abs(size[1] - size[0] - want) <= 512


def test_rows_and_layers_of_a_call():
    L = _native.lib()
    assert [L.ocx_fct_rows(nt, nz, ny, nx) for nx, ny, nz, nt in (BASIN, BAY, (352, 560, 50, 2), (701, 523, 30, 10),
                                                                 (1024, 1024, 50, 10))] == [2, 4, 16, 32, 64]
    assert [L.ocx_rk_layers(2, 20, 128, 128, f) for f in (0, 16, 64, 128, 256)] == [4, 4, 3, 3, 3]
    assert L.ocx_rk_layers(10, 50, 1024, 1024, 0) == L.ocx_rk_layers(10, 50, 1024, 1024, 64) == 50
    assert L.ocx_rk_layers(1, 5, 320, 330, 0) == 5
    assert L.ocx_fct_rows(1, 0, 1, 1) == L.ocx_rk_layers(1, 1, 0, 1, 0) == _native.OCX_E_ARG
