"""Products and forces written over one of their inputs: the one-launch
kernels read inputs while other workgroups write outputs, so such a call goes
through the workspace and must give the same bits as one with its own output.
"""
import numpy as np
import pytest
import torch

from rigidmultiblobswall_amd import forces, wall_rpy
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
