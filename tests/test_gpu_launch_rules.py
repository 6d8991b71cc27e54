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
# (these take 2, 2, 4, 4, 4 and 8 rows; 16 and 32 are asserted further down)
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


# the layer-marching kernel's columns in one piece, in pieces of 1 .. 5 layers and with a shorter last piece, against
# the oracle's unsplit columns: every z face of a piece's first and last layer
# (these take pieces of 1 layer, but for the fourth: 7 of 13 with WENO faces, whole with UP3; longer ones further down)
@pytest.mark.parametrize("nx,ny,nz,nt", [(20, 18, 1, 1), (40, 33, 7, 2), (130, 70, 11, 1), (300, 250, 13, 3),
                                         (70, 66, 23, 1)])
@pytest.mark.parametrize("scheme", ["weno", "js", "up3", "pc"])
def test_columns_cut_into_pieces_match_the_oracle(gpu, nx, ny, nz, nt, scheme):
    from oracle import numpy_ref as R
    print("[gpu case] column pieces", nx, ny, nz, nt, scheme, flush=True)
    case = synth.regional(nx=nx, ny=ny, nz=nz, nt=nt, seed=7, sigma=True)
    Fz = torch.from_numpy(np.ascontiguousarray(case.Fz)).cuda()
    C, V0, V1, Qx, Qy, ok = _dev(case)
    args = (case.C, case.V0, case.V1, case.Qx, case.Qy, case.Fz, case.ok, case.dt)
    if scheme == "pc":
        got = ops.advect_pc(C, V0, V1, Qx, Qy, Fz, ok, case.dt, flags=ops.flags_of(up=3), vert=True)
        want = R.advect_pc(*args, up_order=3)
    else:
        up, js = (3, False) if scheme == "up3" else (0, scheme == "js")
        got = ops.advect_rk3(C, V0, V1, Qx, Qy, Fz, ok, case.dt, flags=ops.flags_of(js=js, up=up), vert=True)
        want = R.advect_rk3(*args, z_variant=not js, up_order=up)
    assert np.array_equal(got.cpu().numpy(), want)


# the along-layer diffusion reads T once where it is Tw, and takes two tracers at a time: odd counts, ragged blocks
@pytest.mark.parametrize("nx,ny,nz,nt", [(1, 1, 1, 1), (63, 5, 2, 2), (64, 4, 3, 3), (65, 9, 2, 1), (130, 17, 5, 5),
                                         (449, 9, 2, 3), (512, 6, 3, 2)])      # rows of a multiple of 8 blocks
def test_diffusion_of_one_and_of_two_arrays_match_the_oracle(gpu, nx, ny, nz, nt):
    from oracle import numpy_ref as R
    print("[gpu case] diffuse_h", nx, ny, nz, nt, flush=True)
    rng = np.random.default_rng(nx)
    T = rng.normal(10.0, 2.0, (nt, nz, ny, nx))
    act = rng.random((ny, nx)) > 0.2
    h = rng.uniform(0.5, 3.0, (nz, ny, nx)) * act
    V = h * 1e6
    cx, cy = rng.uniform(0.9, 1.1, (ny, nx + 1)), rng.uniform(0.9, 1.1, (ny + 1, nx))
    okx, oky = rng.random((ny, nx + 1)) > 0.1, rng.random((ny + 1, nx)) > 0.1
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()                                   # noqa: E731
    m = lambda a: d(a.astype(np.uint8))                                                              # noqa: E731
    args = (d(h), m(act), d(cx), d(cy), m(okx), m(oky), d(V), 100.0, 600.0)
    want = R.diffuse_h_ale(T, T, h, act, cx, cy, okx, oky, V, 100.0, 600.0)
    a, b = d(T), d(T)
    for got in (ops.diffuse_h(a, a, *args), ops.diffuse_h(a, b, *args)):
        assert np.array_equal(got.cpu().numpy(), want)


# both block orders of the along-layer diffusion: rows of one block, of whole lines and of broken ones
@pytest.mark.parametrize("nx,ny,nz,nt", [(40, 37, 3, 2), (64, 50, 5, 3), (72, 33, 4, 3), (136, 21, 7, 1),
                                         (333, 18, 3, 4), (384, 9, 5, 2)])
def test_diffusion_in_both_block_orders_matches_the_oracle(gpu, nx, ny, nz, nt):
    test_diffusion_of_one_and_of_two_arrays_match_the_oracle(gpu, nx, ny, nz, nt)


# chunks of every length that the rule gives, asserted, against chunks of 64 rows
@pytest.mark.parametrize("nx,ny,nz,nt,rows", [(96, 81, 8, 2, 2), (130, 129, 20, 2, 4), (190, 203, 50, 6, 8),
                                              (630, 69, 50, 10, 16), (1260, 70, 50, 10, 32), (1100, 130, 63, 20, 64)])
@pytest.mark.parametrize("precision", ["f64", "split"])
def test_every_chunk_length_gives_the_bits_of_64_rows(gpu, nx, ny, nz, nt, rows, precision):
    from pyocean_amd import _native
    assert _native.lib().ocx_fct_rows(nt, nz, ny, nx) == rows
    print("[gpu case] chunks of", rows, precision, flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows)
    r = lambda *s: torch.rand(*s, device="cuda", dtype=torch.float64, generator=g)                   # noqa: E731
    C, V0, V1 = 10 + r(nt, nz, ny, nx), 1e6 * (0.8 + 0.4 * r(nz, ny, nx)), 1e6 * (0.8 + 0.4 * r(nz, ny, nx))
    Qx, Qy = 2e3 * (r(nz, ny, nx + 1) - 0.5), 2e3 * (r(nz, ny + 1, nx) - 0.5)
    ok = (r(nz, ny, nx) > 0.1).to(torch.uint8)
    got = ops.advect_fct(C, V0, V1, Qx, Qy, ok, 30.0, precision=precision)
    try:
        batch.set_tuning(64, 1)
        assert _native.lib().ocx_fct_rows(nt, nz, ny, nx) == 64
        want = ops.advect_fct(C, V0, V1, Qx, Qy, ok, 30.0, precision=precision)
    finally:
        batch.set_tuning(0, 0)
    assert torch.equal(got, want)


# columns whole and in pieces of 3 and more layers with a shorter last one, with every face scheme, the lengths asserted
@pytest.mark.parametrize("scheme,nx,ny,nz,nt,layers", [
    ("weno", 330, 320, 5, 1, 5), ("weno", 321, 331, 4, 1, 4), ("js", 330, 320, 5, 1, 5), ("weno flat", 330, 320, 5, 1, 5),
    ("weno", 198, 159, 50, 1, 10), ("weno", 128, 128, 20, 2, 4), ("js", 198, 159, 17, 1, 4), ("weno", 260, 250, 9, 1, 5),
    ("weno flat", 198, 159, 17, 1, 4), ("up3", 128, 128, 20, 2, 3), ("up1", 128, 128, 20, 2, 3),
    ("up3", 198, 159, 50, 1, 9), ("up1", 300, 250, 13, 3, 13), ("pc", 128, 128, 20, 2, 3), ("pc", 300, 250, 13, 3, 13),
    ("pc weno", 128, 128, 20, 2, 4), ("pc weno", 330, 320, 5, 1, 5), ("rhs centred", 128, 128, 20, 2, 3),
    ("rhs centred", 300, 250, 13, 3, 13), ("rhs up3", 198, 159, 17, 1, 3), ("rhs", 330, 320, 5, 1, 5),
    ("rhs", 198, 159, 17, 1, 4)])
def test_whole_columns_and_longer_pieces_match_the_oracle(gpu, scheme, nx, ny, nz, nt, layers):
    from oracle import cref
    from oracle import numpy_ref as R
    from pyocean_amd import _native
    flags = ops.flags_of(js=scheme == "js", up=3 if "up3" in scheme or scheme == "pc" else 1 if scheme == "up1" else 0,
                         centred="centred" in scheme)
    assert _native.lib().ocx_rk_layers(nt, nz, ny, nx, flags) == layers
    print("[gpu case] columns", scheme, nx, ny, nz, nt, layers, flush=True)
    case = synth.regional(nx=nx, ny=ny, nz=nz, nt=nt, seed=9, sigma=True)
    vert = "flat" not in scheme
    if not vert:
        case.Fz[...] = 0.0
    Fz = torch.from_numpy(np.ascontiguousarray(case.Fz)).cuda()
    C, V0, V1, Qx, Qy, ok = _dev(case)
    args = (case.C, case.V0, case.V1, case.Qx, case.Qy, case.Fz, case.ok, case.dt)
    if scheme.startswith("pc"):
        got = ops.advect_pc(C, V0, V1, Qx, Qy, Fz, ok, case.dt, flags=flags, vert=True)
        want = R.advect_pc(*args, up_order=3 if scheme == "pc" else 0)
    elif scheme.startswith("rhs"):
        got = ops.rhs(C, Qx, Qy, Fz, ok, ext=C, flags=flags, vert=True)
        rest = (case.C, case.Qx, case.Qy, case.Fz, case.ok, case.C)
        want = cref.rhs(*rest, vert=True) if scheme == "rhs" else \
            R.rhs_up(*rest, order="c" if "centred" in scheme else 3)
    else:
        got = ops.advect_rk3(C, V0, V1, Qx, Qy, Fz, ok, case.dt, flags=flags, vert=vert)
        want = R.advect_rk3(*args, up_order=3 if scheme == "up3" else 1) if scheme[:2] == "up" else \
            cref.advect_rk3(*args, z_variant=scheme != "js")
    assert np.array_equal(got.cpu().numpy(), want)
