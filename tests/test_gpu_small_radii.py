"""Different radii: the one-launch kernel of few blobs and the symmetric kernel
on 64-blob blocks, at the edges of their tiles and of the rules that choose
them, against the ordered kernel (which the other tests hold to the oracle)
and the oracle itself.

Tolerances: FP32 pair terms 1e-6, as everywhere in these tests; FP64 1e-12.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from rigidmultiblobswall_amd import _lib, wall_rpy

pytestmark = pytest.mark.gpu

ETA = 0.9
TOL = {"fp64": 1e-12, "fp32": 1e-6, "fp32_blocked": 1e-6, "fp32_kahan": 1e-6}
ORDERED = _lib.Tuning(256, 0, 0, -1, 0)


def rel(a, b):
    return float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))


def _system(n, seed):
    rng = np.random.default_rng(seed)
    side = 1.3 * np.sqrt(n) + 1.0
    # some blobs overlap the wall, each other, and some hold smaller ones
    r = np.column_stack([rng.uniform(0, side, n), rng.uniform(0, side, n), rng.uniform(0.1, 2.5, n)])
    return r, rng.standard_normal((n, 3)), rng.uniform(0.05, 0.9, n)


@pytest.mark.parametrize("prec", ["fp32_blocked", "fp64"])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 63, 64, 65, 257, 1600, 1601, 1664, 4033, 10001, 18432, 18433])
def test_self_sizes(gpu, n, prec):
    print(f"case radii self n={n} {prec}", flush=True)
    r, f, rad = _system(n, n)
    got = wall_rpy.apply_radii_self(r, f, rad, ETA, precision=prec)
    ref = wall_rpy.apply_radii_self(r, f, rad, ETA, precision=prec, tuning=ORDERED)
    assert rel(got, ref) <= TOL[prec], rel(got, ref)
    kernel = wall_rpy.describe_radii_self(n, prec)["kernel"]
    assert kernel == ("ordered" if n <= 1600 else "symmetric")


@pytest.mark.parametrize("n", [90, 2500])
@pytest.mark.parametrize("prec", ["fp32", "fp32_blocked", "fp32_kahan", "fp64"])
@pytest.mark.parametrize("boundary", ["wall", "unbounded", "free_surface"])
def test_boundaries_and_precisions(gpu, boundary, prec, n):
    print(f"case radii {boundary} {prec} n={n}", flush=True)
    r, f, rad = _system(n, 3)
    for L in (None, (40.0, 0.0, 0.0), (30.0, 25.0, 0.0)) if n < 100 else (None,):
        kw = dict(periodic_length=L, precision=prec, boundary=boundary)
        got = wall_rpy.apply_radii_self(r, f, rad, ETA, **kw)
        assert rel(got, wall_rpy.apply_radii_self(r, f, rad, ETA, tuning=ORDERED, **kw)) <= TOL[prec]
    if n < 100 and boundary != "free_surface":
        want = O.radii_apply(r, r, f, rad, rad, ETA, wall=boundary == "wall")
        got = wall_rpy.apply_radii_self(r, f, rad, ETA, precision=prec, boundary=boundary)
        assert rel(got, torch.as_tensor(np.asarray(want).reshape(n, 3)).to(got)) <= TOL[prec]


@pytest.mark.parametrize("ns,nt", [(1, 1), (1, 70), (70, 1), (255, 31), (257, 4097), (3000, 9), (8193, 9), (10, 6000)])
def test_source_to_target(gpu, ns, nt):
    print(f"case radii source {ns} target {nt}", flush=True)
    (s, f, rs), (t, _, rt) = _system(ns, 5), _system(nt, 6)
    for prec in ("fp32_blocked", "fp64"):
        for L in (None, (30.0, 25.0, 0.0)):
            kw = dict(periodic_length=L, precision=prec)
            got = wall_rpy.apply_radii(s, t, f, rs, rt, ETA, **kw)
            ref = wall_rpy.apply_radii(s, t, f, rs, rt, ETA, tuning=_lib.Tuning(256, 0, 0, -1, 0), **kw)
            assert rel(got, ref) <= TOL[prec]


def test_coincident_blobs(gpu):
    """Blobs at one point are in the inner regime of the tensor, not an error."""
    for n in (70, 2500):
        r, f, rad = _system(n, 8)
        r[1] = r[0]
        got = wall_rpy.apply_radii_self(r, f, rad, ETA, precision="fp64")
        assert rel(got, wall_rpy.apply_radii_self(r, f, rad, ETA, precision="fp64", tuning=ORDERED)) <= 1e-12
