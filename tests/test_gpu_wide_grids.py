"""
GPU tests of launches whose blocks fill more than one grid dimension, against the same kernels on parts of the work
that stay below that.
"""
from __future__ import annotations

import pytest
import torch

from pyocean_amd import ops

pytestmark = pytest.mark.gpu


def _need_memory(gib):
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
