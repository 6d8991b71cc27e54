"""
GPU tests of the layer-transport kernels whose layers are shared by a workgroup's wavefronts, at layer and column
counts around the edges of their chunks, and of the outflow limiter's short ways, against the oracle's bits.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import numpy_ref as R
from pyocean_amd import ale, synth

pytestmark = pytest.mark.gpu


def _d(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _bits(got, want, name):
    g = got.cpu().numpy()
    assert np.array_equal(g.view(np.int64), np.ascontiguousarray(want).view(np.int64)), name


# chunks of 16 layers (4 a wavefront), 64 layers a column at most in registers, 64 columns a workgroup
@pytest.mark.parametrize("nx,ny,nz", [(12, 5, 1), (63, 9, 3), (64, 4, 4), (65, 3, 15), (31, 7, 16), (20, 33, 17),
                                      (16, 16, 63), (17, 11, 64), (9, 14, 65)])
def test_transports_at_chunk_edges_match_the_oracle(gpu, nx, ny, nz):
    print("[gpu case] transport chunks", nx, ny, nz, flush=True)
    a = synth.ale_inputs(nx, ny, nz, seed=3)
    act = np.asarray(a.active, bool)
    for u1, u0, wet, w, L, D, dx, ax in ((a.u_new, a.u_old, a.wet_u, a.wu, a.Lu, a.Du, a.dx_t, 0),
                                         (a.v_new, a.v_old, a.wet_v, a.wv, a.Lv, a.Dv, a.dy_t, 1)):
        ut, Qb = ale.transport_velocity(_d(u1), _d(u0), _d(wet), _d(w), _d(L), _d(D), a.theta, a.theta_bc)
        rut, rQb = R.transport_velocity(u1, u0, wet, w, L, D, a.theta, a.theta_bc)
        _bits(ut, rut, "ut")
        _bits(Qb, rQb, "Q_bt")
        qp, qn = ale.face_thickness_axis(_d(a.h), _d(a.H), _d(act), True, ax)
        got, it = ale.ppm_transport(_d(a.h), ut, _d(L), Qb, qp, qn, _d(act), a.dt, _d(dx), ax, return_iterations=True)
        sw = (lambda x: x) if ax == 0 else (lambda x: np.ascontiguousarray(np.swapaxes(x, -1, -2)))
        want, rit = R.ppm_transport_x(sw(a.h), sw(rut), sw(L), sw(rQb), sw(qp.cpu().numpy()), sw(qn.cpu().numpy()),
                                      sw(act), a.dt, sw(dx), return_iterations=True)
        assert it == rit
        _bits(got, sw(want), f"Q axis {ax}")


# iterations with a launch of their own, and bundles of them: stops before, at and after the ends of both, with columns
# that never converge (a flux beyond their bracket), that do after 4, and, a flux just inside its bracket, after 23
@pytest.mark.parametrize("max_iter", [0, 1, 7, 8, 9, 19, 20, 21, 33])
@pytest.mark.parametrize("reach", [1.0, 50.0, 1.672235424598329])
def test_iteration_bundles_stop_where_the_oracle_stops(gpu, max_iter, reach):
    print("[gpu case] newton bundles", max_iter, reach, flush=True)
    a = synth.ale_inputs(40, 13, 6, seed=4)
    act = np.asarray(a.active, bool)
    ut, Qb = R.transport_velocity(a.u_new, a.u_old, a.wet_u, a.wu, a.Lu, a.Du, a.theta, a.theta_bc)
    qe, qw = R.face_transport_thickness(a.h, a.H, act, True)
    Qb = Qb * reach
    want, rit = R.ppm_transport_x(a.h, ut, a.Lu, Qb, qe, qw, act, a.dt, a.dx_t, max_iter, return_iterations=True)
    got, it = ale.ppm_transport(_d(a.h), _d(ut), _d(a.Lu), _d(Qb), _d(qe), _d(qw), _d(act), a.dt, _d(a.dx_t), 0, max_iter,
                                return_iterations=True)
    assert it == rit
    _bits(got, want, "Q")


# faces with no cut (a zero flux may lose its sign there), with a cut that all comes back, and a room0 that is not
# finite (no short way: its product with 0 is a NaN in every layer of the column)
@pytest.mark.parametrize("wild", [None, np.inf])
@pytest.mark.parametrize("n", [1, 8, 9, 17])
def test_limit_outflow_short_ways_match_the_oracle(gpu, n, wild):
    print("[gpu case] limiter short ways", n, wild, flush=True)
    rng = np.random.default_rng(n)
    ny, nx, dt = 9, 13, 100.0
    h = rng.uniform(1.0, 2.0, (n, ny, nx))
    area = np.full((ny, nx), 1e4)
    Qx, Qy = rng.normal(0, 5.0, (n, ny, nx + 1)), rng.normal(0, 5.0, (n, ny + 1, nx))
    Qx[:, :, [0, -1]], Qy[:, [0, -1]] = 0.0, 0.0
    Qx[:, 2], Qx[:, 3, ::2] = -0.0, -0.0
    act = np.ones((ny, nx), bool)
    h[0, 4, 5] = 1e-3
    Qx[0, 4, 6] = 40.0
    if wild is not None:
        h[n - 1, 7, 9] = wild
    args = (_d(h), _d(Qx), _d(Qy), _d(area), dt, _d(act))
    try:
        with np.errstate(all="ignore"):
            rx, ry, nl, status = R.limit_outflow(h, Qx, Qy, area, dt, act)
    except RuntimeError:                       # a column that cannot supply its cut (one layer): refused on both sides
        with pytest.raises(RuntimeError):
            ale.limit_outflow(*args)
        return
    except IndexError:                         # the oracle's search for the emptied layer finds none among NaNs: no answer
        return
    gx, gy, gl = ale.limit_outflow(*args)
    assert gl == nl and status != "noop"
    for g, r in ((gx, rx), (gy, ry)):
        g = g.cpu().numpy()
        assert np.array_equal(np.isnan(g), np.isnan(r))
        assert np.array_equal(np.where(np.isnan(g), 0.0, g).view(np.int64), np.where(np.isnan(r), 0.0, r).view(np.int64))


# a u-face (or a v-face) with nowhere to place its cut ends the call: on a u-face Qy is still the caller's, on either
# the fluxes of that pass are the oracle's at the point where it raises
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 9])
def test_limit_outflow_keeps_the_fluxes_of_the_error(gpu, n, axis):
    import ctypes

    from pyocean_amd import _native, ops
    print("[gpu case] limiter error", n, axis, flush=True)
    rng = np.random.default_rng(5)
    ny, nx, dt = 9, 13, 100.0
    h = rng.uniform(1.0, 2.0, (n, ny, nx))
    area = np.full((ny, nx), 1e4)
    Qx, Qy = rng.normal(0, 5.0, (n, ny, nx + 1)), rng.normal(0, 5.0, (n, ny + 1, nx))
    Qx[:, :, [0, -1]], Qy[:, [0, -1]] = 0.0, 0.0
    act = np.ones((ny, nx), bool)
    h[:, 4, 5] = 0.0                                  # an empty column that a face must carry its cut out of
    h[0, 6, 8] = 1e-3                                 # a layer whose cut across a v-face changes Qy
    Qx[:, 4, 5:7] = Qy[:, 4:6, 5] = 0.0
    if axis == 0:
        Qx[:, 4, 6] = 7.0
    else:
        Qy[:, 5, 5] = 7.0
    Qy[0, 7, 8] = 40.0
    with pytest.raises(RuntimeError):
        R.limit_outflow(h, Qx, Qy, area, dt, act)
    want = (Qx.copy(), Qy.copy())
    dh, dx, dy, da, dm = _d(h), _d(Qx), _d(Qy), _d(area), _d(act.astype(np.uint8))
    L = _native.lib()
    ws = torch.empty(int(L.ocx_limit_outflow_workspace_bytes(n, ny, nx)), dtype=torch.uint8, device="cuda")
    nl, st = ctypes.c_longlong(0), ctypes.c_int(0)
    where, val = (ctypes.c_longlong * 3)(), ctypes.c_double(0.0)
    p = lambda t: ctypes.c_void_p(t.data_ptr())                                                      # noqa: E731
    rc = L.ocx_limit_outflow_f64(p(dh), p(dx), p(dy), p(da), p(dm), n, ny, nx, dt, 2e-10, 50, 0, 0, 0, p(ws), ws.numel(),
                                 ctypes.byref(nl), ctypes.byref(st), where, ctypes.byref(val), ops._stream())
    assert rc == _native.OCX_E_RANGE and st.value == _native.OUTFLOW_EMPTY_DONOR
    assert tuple(where)[:1] == (axis,)
    face = (4, 6) if axis == 0 else None
    if face:
        assert tuple(where)[1:] == face
        _bits(dy, want[1], "Qy")
    assert not np.array_equal(dx.cpu().numpy() if axis == 0 else dy.cpu().numpy(), want[axis])


# grids whose bundles hold 12, 5, 2 and (every iteration alone) 1 iterations
@pytest.mark.parametrize("max_iter", [9, 11, 20])
@pytest.mark.parametrize("nx,ny", [(40, 13), (310, 316), (500, 440), (530, 520)])
def test_bundles_of_every_length_stop_where_the_oracle_stops(gpu, nx, ny, max_iter):
    print("[gpu case] bundle lengths", nx, ny, max_iter, flush=True)
    a = synth.ale_inputs(nx, ny, 2, seed=4)
    act = np.asarray(a.active, bool)
    ut, Qb = R.transport_velocity(a.u_new, a.u_old, a.wet_u, a.wu, a.Lu, a.Du, a.theta, a.theta_bc)
    qe, qw = R.face_transport_thickness(a.h, a.H, act, True)
    for reach in (1.0, 50.0):                 # converges after a few iterations; never
        want, rit = R.ppm_transport_x(a.h, ut, a.Lu, Qb * reach, qe, qw, act, a.dt, a.dx_t, max_iter,
                                      return_iterations=True)
        got, it = ale.ppm_transport(_d(a.h), _d(ut), _d(a.Lu), _d(Qb * reach), _d(qe), _d(qw), _d(act), a.dt, _d(a.dx_t),
                                    0, max_iter, return_iterations=True)
        assert it == rit
        _bits(got, want, "Q")


# layer counts on both sides of the line between columns of one thread and columns of a workgroup, on a grid below and
# on one above the 4096 workgroups at which it moves, with a stop after a few iterations and with none
@pytest.mark.parametrize("nx,ny,nz", [(63, 40, 1), (63, 40, 4), (63, 40, 5), (63, 40, 6), (530, 520, 5), (530, 520, 11),
                                      (530, 520, 12), (530, 520, 13), (530, 520, 17)])
@pytest.mark.parametrize("axis", [0, 1])
def test_walked_and_shared_columns_match_the_oracle(gpu, nx, ny, nz, axis):
    print("[gpu case] walked columns", nx, ny, nz, axis, flush=True)
    a = synth.ale_inputs(nx, ny, nz, seed=6)
    act = np.asarray(a.active, bool)
    u1, u0, wet, w, Lf, D, d = ((a.u_new, a.u_old, a.wet_u, a.wu, a.Lu, a.Du, a.dx_t) if axis == 0 else
                                (a.v_new, a.v_old, a.wet_v, a.wv, a.Lv, a.Dv, a.dy_t))
    ut, Qb = R.transport_velocity(u1, u0, wet, w, Lf, D, a.theta, a.theta_bc)
    qp, qn = ale.face_thickness_axis(_d(a.h), _d(a.H), _d(act), True, axis)
    sw = (lambda x: x) if axis == 0 else (lambda x: np.ascontiguousarray(np.swapaxes(x, -1, -2)))
    for reach, max_iter in ((1.0, 20), (50.0, 3)):
        want, rit = R.ppm_transport_x(sw(a.h), sw(ut), sw(Lf), sw(Qb * reach), sw(qp.cpu().numpy()),
                                      sw(qn.cpu().numpy()), sw(act), a.dt, sw(d), max_iter, return_iterations=True)
        got, it = ale.ppm_transport(_d(a.h), _d(ut), _d(Lf), _d(Qb * reach), qp, qn, _d(act), a.dt, _d(d), axis, max_iter,
                                    return_iterations=True)
        assert it == rit
        _bits(got, sw(want), f"Q reach {reach}")


# the transport velocity's columns of one thread below 10 and above 64 layers
@pytest.mark.parametrize("n", [1, 2, 9, 10, 11, 64, 65])
@pytest.mark.parametrize("nx,ny", [(1, 1), (63, 5), (300, 41)])
def test_transport_velocity_on_both_sides_of_its_lines(gpu, nx, ny, n):
    print("[gpu case] transport velocity", nx, ny, n, flush=True)
    rng = np.random.default_rng(n)
    u1, u0, w = (rng.normal(0, 0.3, (n, ny, nx)) for _ in range(3))
    wet, Lf, D = rng.random((ny, nx)) > 0.2, rng.uniform(900, 1100, (ny, nx)), rng.uniform(1, 50, (ny, nx))
    ut, Qb = ale.transport_velocity(_d(u1), _d(u0), _d(wet), _d(w), _d(Lf), _d(D), 0.6, 0.5)
    rut, rQb = R.transport_velocity(u1, u0, wet, w, Lf, D, 0.6, 0.5)
    _bits(ut, rut, "ut")
    _bits(Qb, rQb, "Q_bt")


# the transport thicknesses of few layers, taken one by one, and of more, KB = 8 in flight
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("axis", [0, 1])
def test_face_thickness_of_few_layers_matches_the_oracle(gpu, n, axis):
    print("[gpu case] face thickness", n, axis, flush=True)
    rng = np.random.default_rng(n)
    ny, nx = 37, 70
    H = rng.uniform(5.0, 50.0, (ny, nx))
    h = rng.dirichlet(np.ones(n), (ny, nx)).transpose(2, 0, 1) * H
    h[rng.random(h.shape) < 0.02] = np.nan
    act = rng.random((ny, nx)) > 0.1
    got = ale.face_thickness_axis(_d(h), _d(H), _d(act), True, axis)
    sw = (lambda x: x) if axis == 0 else (lambda x: np.ascontiguousarray(np.swapaxes(x, -1, -2)))
    for g, w, nm in zip(got, R.face_transport_thickness(sw(h), sw(H), sw(act), True), ("q_pos", "q_neg")):
        _bits(g, sw(w), nm)


# the edges' layers in one slice, in some and in slices of 4: planes on both sides of the line, ragged last slices
@pytest.mark.parametrize("nx,ny,n", [(70, 37, 1), (70, 37, 9), (700, 760, 3), (512, 512, 21), (1030, 1020, 6)])
@pytest.mark.parametrize("axis", [0, 1])
def test_ppm_edges_of_every_slicing_match_the_oracle(gpu, nx, ny, n, axis):
    print("[gpu case] edge slices", nx, ny, n, axis, flush=True)
    rng = np.random.default_rng(n)
    h = rng.uniform(0.0, 3.0, (n, ny, nx))
    act = rng.random((ny, nx)) > 0.1
    got = ale.ppm_edges_axis(_d(h), _d(act), axis)
    sw = (lambda x: x) if axis == 0 else (lambda x: np.ascontiguousarray(np.swapaxes(x, -1, -2)))
    for g, w, nm in zip(got, R.ppm_edges(sw(np.where(act, h, 0.0)), sw(act)), ("low", "high")):
        _bits(g, sw(w), nm)
