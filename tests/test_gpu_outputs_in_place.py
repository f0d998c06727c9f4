"""Products and forces written over one of their inputs: the launches that write
the outputs (the one-launch kernels and the reduces of the others) read inputs
while other workgroups write outputs, so such a call goes through the workspace
and must give the same bits as one with its own output.
"""
import ctypes

import numpy as np
import pytest
import torch

from rigidmultiblobswall_amd import _lib, forces, wall_rpy
from rigidmultiblobswall_amd._lib import RMW_UF

pytestmark = pytest.mark.gpu


def _blobs(n, seed):
    rng = np.random.default_rng(seed)
    r = torch.from_numpy(np.column_stack([rng.uniform(0, 1.5 * np.sqrt(n), (n, 2)), rng.uniform(0.2, 3.0, n)])).cuda()
    return r, torch.from_numpy(rng.standard_normal((n, 3))).cuda()


@pytest.mark.parametrize("n", [5, 700, 2304, 3000])
def test_product_over_its_forces(gpu, n):
    print(f"case product in place n={n}", flush=True)
    r, f = _blobs(n, n)
    want = wall_rpy.apply(RMW_UF, r, force=f, eta=0.9, a=0.4)[0]
    wall_rpy.apply(RMW_UF, r, force=f, eta=0.9, a=0.4, out_velocity=f)
    assert torch.equal(f.reshape(-1), want.reshape(-1))
    f2 = torch.stack([_blobs(n, n + s)[1] for s in (1, 2, 3)])   # right-hand sides
    t2 = f2.flip(0).contiguous()
    want = wall_rpy.apply(15, r, force=f2, torque=t2, eta=0.9, a=0.4, k=3)
    wall_rpy.apply(15, r, force=f2, torque=t2, eta=0.9, a=0.4, k=3, out_velocity=f2, out_omega=t2)
    assert torch.equal(f2.reshape(-1), want[0].reshape(-1)) and torch.equal(t2.reshape(-1), want[1].reshape(-1))


@pytest.mark.parametrize("n", [5, 700, 2304, 3000])
def test_radii_product_over_its_forces(gpu, n):
    print(f"case radii in place n={n}", flush=True)
    r, f = _blobs(n, n)
    rad = torch.linspace(0.2, 0.5, n, dtype=torch.float64, device="cuda")
    want = wall_rpy.apply_radii_self(r, f, rad, 0.9)
    g = f.clone()
    wall_rpy.apply_radii_self(r, g, rad, 0.9, out=g)
    assert torch.equal(g, want)
    want = wall_rpy.apply_radii(r, r, f, rad, rad, 0.9)
    wall_rpy.apply_radii(r, r, f, rad, rad, 0.9, out=f)
    assert torch.equal(f, want)


@pytest.mark.parametrize("n", [5, 700, 3000, 6000, 9000])
def test_forces_over_the_positions(gpu, n):
    print(f"case forces in place n={n}", flush=True)
    r, _ = _blobs(n, n)
    want = forces.blob_forces(r, 0.3, 0.05, 0.4, precision="fp64")
    forces.blob_forces(r, 0.3, 0.05, 0.4, precision="fp64", out=r)
    # (another order of the sums where cells would have been taken)
    assert torch.linalg.vector_norm(r - want) <= 1e-13 * torch.linalg.vector_norm(want)


ROUTES = {"direct": (700, None), "blocks": (5000, None), "tiles": (20000, None), "ordered": (9000, dict(symmetric=-1))}


@pytest.mark.parametrize("route", sorted(ROUTES))
def test_product_over_every_input(gpu, route):
    """Five right-hand sides (a pass of four and one of one), outputs over the
    forces and torques, crossed, and the velocity of one over the positions,
    which the second pass reads again."""
    n, tuning = ROUTES[route]
    print(f"case product over its inputs, {route} n={n}", flush=True)
    r, _ = _blobs(n, n)
    k = 5
    f, t = (torch.stack([_blobs(n, n + 10 * q + s)[1] for s in range(k)]) for q in (1, 2))
    kw = dict(eta=0.9, a=0.4, k=k, tuning=tuning)
    want = wall_rpy.apply(15, r, force=f, torque=t, **kw)
    for crossed in (False, True):
        g, s = f.clone(), t.clone()
        wall_rpy.apply(15, r, force=g, torque=s, out_velocity=s if crossed else g, out_omega=g if crossed else s, **kw)
        u, w = (s, g) if crossed else (g, s)
        assert torch.equal(u.reshape(-1), want[0].reshape(-1)) and torch.equal(w.reshape(-1), want[1].reshape(-1))
    # rows of a block: [positions, room], the velocities from the positions on
    block = torch.zeros((k, n, 3), dtype=torch.float64, device=gpu)
    block[0] = r
    wall_rpy.apply(15, block[0], force=f, torque=t, out_velocity=block, **kw)
    assert torch.equal(block.reshape(-1), want[0].reshape(-1))


def test_product_without_a_workspace_over_its_forces(gpu):
    lib = _lib.load()
    for n, k in ((700, 1), (3000, 4), (12000, 1), (9000, 4), (30000, 1)):
        print(f"case product without a workspace in place n={n} k={k}", flush=True)
        r, _ = _blobs(n, n)
        f, t = (torch.stack([_blobs(n, n + 10 * q + s)[1] for s in range(k)]) for q in (1, 2))

        def call(u, w, g, s):
            _lib.check(lib.rmw_wall_rpy_apply_noalloc(15, _lib.precision_code("fp32"), r.data_ptr(), g.data_ptr(),
                                                      s.data_ptr(), u.data_ptr(), w.data_ptr(), n, k, 0, 0.9, 0.4,
                                                      (ctypes.c_double * 3)(0, 0, 0), None,
                                                      torch.cuda.current_stream().cuda_stream))
        u, w = torch.empty_like(f), torch.empty_like(f)
        call(u, w, f, t)
        call(f, t, f, t)
        # (the array may hold another layout's sums beside the outputs)
        assert float(torch.linalg.vector_norm(f - u)) <= 1e-6 * float(torch.linalg.vector_norm(u))
        assert float(torch.linalg.vector_norm(t - w)) <= 1e-6 * float(torch.linalg.vector_norm(w))


@pytest.mark.parametrize("n,tuning", [(700, None), (3000, None), (20000, None), (9000, dict(symmetric=-1))],
                         ids=["direct", "blocks", "tiles", "ordered"])
def test_radii_product_over_the_positions(gpu, n, tuning):
    print(f"case radii over positions n={n}", flush=True)
    r, f = _blobs(n, n)
    rad = torch.linspace(0.2, 0.5, n, dtype=torch.float64, device="cuda")
    want = wall_rpy.apply_radii_self(r, f, rad, 0.9, tuning=tuning)
    x = r.clone()
    wall_rpy.apply_radii_self(x, f, rad, 0.9, out=x, tuning=tuning)
    assert torch.equal(x, want)
    x = torch.cat([rad, torch.zeros(2 * n, dtype=torch.float64, device="cuda")])   # over the radii
    wall_rpy.apply_radii_self(r, f, x[:n], 0.9, out=x.view(n, 3), tuning=tuning)
    assert torch.equal(x.view(n, 3), want)
    want = wall_rpy.apply_radii(r, r, f, rad, rad, 0.9, tuning=tuning)
    wall_rpy.apply_radii(r, r, f, rad, rad, 0.9, out=r, tuning=tuning)
    assert torch.equal(r, want)
