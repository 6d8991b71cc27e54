"""
GPU tests of launches whose blocks fill more than one grid dimension, against the same kernels on parts of the work
that stay below that.
"""
from __future__ import annotations

import gc

import pytest
import torch

from pyocean_amd import ale, ops

pytestmark = pytest.mark.gpu


def _need_memory(gib):
    gc.collect()
    torch.cuda.empty_cache()                           # what earlier tests left with torch's allocator
    if torch.cuda.mem_get_info()[0] < gib << 30:
        pytest.skip(f"needs {gib} GiB of device memory")


# one block holds 64 x 4 cells, so a plane of one column has the most blocks for its cells: 2^22 blocks and one more
# layer, and beyond the 2^26 at which the threads of one dimension no longer count in 32 bits
@pytest.mark.parametrize("ny,nz,gib", [(1 << 20, 17, 2), (1 << 21, 129, 16)])
@pytest.mark.parametrize("same", [True, False])
def test_diffusion_of_many_blocks(gpu, ny, nz, gib, same):
    print("[gpu case] wide diffuse_h", ny, nz, same, flush=True)
    _need_memory(gib)
    g = torch.Generator(device="cuda").manual_seed(1)
    r = lambda *s: torch.rand(*s, device="cuda", dtype=torch.float64, generator=g)                   # noqa: E731
    m = lambda *s: (r(*s) > 0.1).to(torch.uint8)                                                     # noqa: E731
    T, h, V = r(1, nz, ny, 1), r(nz, ny, 1), 1e6 + r(nz, ny, 1)
    Tw = T if same else T.clone()
    act, cx, cy, okx, oky = m(ny, 1), r(ny, 2), r(ny + 1, 1), m(ny, 2), m(ny + 1, 1)
    got = ops.diffuse_h(T, Tw, h, act, cx, cy, okx, oky, V, 100.0, 600.0)
    for k in range(0, nz, 8):                          # the layers are independent
        e = min(k + 8, nz)
        t = T[:, k:e].contiguous()
        want = ops.diffuse_h(t, t if same else t.clone(), h[k:e].contiguous(), act, cx, cy, okx, oky,
                             V[k:e].contiguous(), 100.0, 600.0)
        assert torch.equal(got[:, k:e], want), k


# four threads a column: from 2^30 columns on, the threads of one dimension no longer count in 32 bits
def test_transport_velocity_of_many_columns(gpu):
    print("[gpu case] wide transport velocity", flush=True)
    _need_memory(60)
    rows, cols = 1 << 20, 1088
    g = torch.Generator(device="cuda").manual_seed(2)
    u = torch.rand(1, rows, cols, device="cuda", dtype=torch.float64, generator=g)
    wet = torch.ones(rows, cols, dtype=torch.uint8, device="cuda")
    ut, Qb = ale.transport_velocity(u, u, wet, u, u[0], u[0], 0.6, 0.5)
    q = rows // 4
    for a in range(0, rows, q):                        # the columns are independent
        x = u[:, a:a + q]
        w0, w1 = ale.transport_velocity(x, x, wet[a:a + q], x, x[0], x[0], 0.6, 0.5)
        assert torch.equal(ut[:, a:a + q], w0) and torch.equal(Qb[a:a + q], w1), a
    del u, ut, Qb, wet, x, w0, w1
    torch.cuda.empty_cache()


def test_ppm_transport_of_many_columns(gpu):
    print("[gpu case] wide ppm transport", flush=True)
    _need_memory(120)
    rows, nx = 1 << 20, 1087
    g = torch.Generator(device="cuda").manual_seed(3)
    h = 0.5 + torch.rand(1, rows, nx, device="cuda", dtype=torch.float64, generator=g)
    u = 0.5 + torch.rand(1, rows, nx + 1, device="cuda", dtype=torch.float64, generator=g)
    act = torch.ones(rows, nx, dtype=torch.uint8, device="cuda")
    ws = ops.Workspace()
    call = lambda h, u, act: ale.ppm_transport(h, u, u[0], u[0], u, u, act, 0.1, h[0], 0, 1,        # noqa: E731
                                               workspace=ws)
    out = call(h, u, act)
    q = rows // 4
    for a in range(0, rows, q):                        # so are the rows, but for the stop of all columns' iterations
        part = call(h[:, a:a + q], u[:, a:a + q], act[a:a + q])
        assert torch.equal(out[:, a:a + q], part), a
    del h, u, act, ws, out, part
    torch.cuda.empty_cache()
