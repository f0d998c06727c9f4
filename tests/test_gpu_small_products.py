"""The direct kernel (few blobs, one launch) and the symmetric kernel on
64-blob blocks, at the edges of their tiles and of the rule that chooses
them, against the ordered kernel (which the other tests hold to the oracle)
and the oracle itself.

Tolerances: FP32 pair terms 1e-6, as everywhere in these tests; FP64 1e-12.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from rigidmultiblobswall_amd import _lib, wall_rpy
from rigidmultiblobswall_amd._lib import RMW_UF, RMW_UT, RMW_WF, RMW_WT

pytestmark = pytest.mark.gpu

GRAND = 15
ETA, A = 0.9, 0.4
TOL = {"fp64": 1e-12, "fp32": 1e-6, "fp32_blocked": 1e-6, "fp32_kahan": 1e-6}
ORDERED = _lib.Tuning(256, 0, 0, -1, 0)


def rel(a, b):
    return float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))


def _system(n, seed, k=1):
    rng = np.random.default_rng(seed)
    side = 1.2 * np.sqrt(n) + 1.0
    # some blobs overlap the wall (z < a) and each other
    r = np.column_stack([rng.uniform(0, side, n), rng.uniform(0, side, n), rng.uniform(0.2, 2.5, n)])
    return r, rng.standard_normal((k, n, 3)), rng.standard_normal((k, n, 3))


def _both(mask, prec, n, seed, k=1, L=None, domain="single_wall"):
    r, f, t = _system(n, seed, k)
    kw = dict(force=f, torque=t, eta=ETA, a=A, precision=prec, k=k, periodic_length=L, domain=domain)
    got = wall_rpy.apply(mask, r, tuning="heuristic", **kw)
    ref = wall_rpy.apply(mask, r, tuning=ORDERED, **kw)
    return [(g, x) for g, x in zip(got, ref) if g is not None]


@pytest.mark.parametrize("prec", ["fp32_blocked", "fp64"])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 63, 64, 65, 255, 257, 513, 2303, 2304, 2305, 2433])
def test_sizes_around_the_tiles(gpu, n, prec):
    print(f"case small product n={n} {prec}", flush=True)
    for mask in (RMW_UF, GRAND):
        for g, ref in _both(mask, prec, n, n):
            assert rel(g, ref) <= TOL[prec], (mask, rel(g, ref))
    plan = wall_rpy.describe(RMW_UF, n, 1, prec, tuning="heuristic")
    assert plan["kernel"] == ("ordered" if n <= 2304 else "symmetric")


@pytest.mark.parametrize("n", [70, 2400])
@pytest.mark.parametrize("mask", [RMW_UF, RMW_UT, RMW_WF, RMW_WT, RMW_UF | RMW_UT, RMW_UF | RMW_WF, RMW_UT | RMW_WT,
                                  RMW_WF | RMW_WT, GRAND])
def test_every_mask_precision_and_boundary(gpu, mask, n):
    domains = {"single_wall": 15, "no_wall": 15, "in_plane": 3, "free_surface": 1}
    boxes = [None, (30.0, 25.0, 0.0)] + ([(30.0, 0.0, 9.0)] if n < 100 else [])
    for prec in TOL:
        print(f"case small product mask={mask} n={n} {prec}", flush=True)
        for dom, served in domains.items():
            if mask & ~served:
                continue
            for L in boxes:
                for g, ref in _both(mask, prec, n, mask, L=L, domain=dom):
                    assert rel(g, ref) <= TOL[prec], (dom, L, prec, rel(g, ref))


@pytest.mark.parametrize("k", [2, 3, 4, 5])
@pytest.mark.parametrize("n", [90, 2500])
def test_several_right_hand_sides(gpu, n, k):
    print(f"case small product n={n} k={k}", flush=True)
    for prec in ("fp32_blocked", "fp64"):
        for mask in (RMW_UF, GRAND, RMW_UF | RMW_UT):
            for g, ref in _both(mask, prec, n, k, k=k):
                assert rel(g, ref) <= TOL[prec]
    # rows further apart than they are long
    r, f, t = _system(n, k, k)
    rd = torch.from_numpy(r).to(gpu)
    X = torch.full((k, 6 * n + 10), 7.0, dtype=torch.float64, device=gpu)
    X[:, : 6 * n] = torch.from_numpy(np.concatenate([f.reshape(k, -1), t.reshape(k, -1)], axis=1))
    Y, Yr = torch.full_like(X, 5.0), torch.full_like(X, 5.0)
    wall_rpy.apply_strided(GRAND, rd, n, X, Y, ETA, A, precision="fp64", tuning="heuristic")
    wall_rpy.apply_strided(GRAND, rd, n, X, Yr, ETA, A, precision="fp64", tuning=ORDERED)
    assert rel(Y[:, : 6 * n], Yr[:, : 6 * n]) <= 1e-12
    assert bool((Y[:, 6 * n:] == 5.0).all())


@pytest.mark.parametrize("sizes", [[0, 1, 70, 0, 300, 64, 5], [2500, 0, 130, 2305, 1]], ids=["direct", "blocks"])
def test_batches_with_empty_and_odd_systems(gpu, sizes):
    off = np.concatenate([[0], np.cumsum(sizes)])
    n = int(off[-1])
    for k in (1, 3):
        r, f, t = _system(n, 11, k)
        for prec in ("fp32_blocked", "fp64"):
            print(f"case small batch {sizes} k={k} {prec}", flush=True)
            got = wall_rpy.apply_ragged(GRAND, r, off, f, t, ETA, A, precision=prec, k=k, tuning="heuristic")
            ref = wall_rpy.apply_ragged(GRAND, r, off, f, t, ETA, A, precision=prec, k=k, tuning=ORDERED)
            for g, x in zip(got, ref):
                assert rel(g, x) <= TOL[prec]


@pytest.mark.parametrize("n", [130, 2330])
def test_against_the_oracle(gpu, n):
    r, f, t = _system(n, 5)
    rows = (0, min(n, 200))
    for L in (None, (20.0, 22.0, 0.0)):
        print(f"case small product oracle n={n} L={L}", flush=True)
        b = lambda blk, v: O.block_apply(blk, r, v[0], ETA, A, L, rows=rows).reshape(n, 3)[rows[0]:rows[1]]  # noqa: E731
        u, w = wall_rpy.apply(GRAND, r, f, t, ETA, A, periodic_length=L, precision="fp64", tuning="heuristic")
        for got, ref in ((u, b(O.UF, f) + b(O.UT, t)), (w, b(O.WF, f) + b(O.WT, t))):
            assert rel(got[rows[0]:rows[1]].cpu(), torch.from_numpy(ref)) <= 1e-12


@pytest.mark.parametrize("n", [200, 2500])
@pytest.mark.parametrize("prec", ["fp32", "fp32_blocked", "fp64"])
def test_coincident_blobs_stay_non_finite(gpu, n, prec):
    r, f, _ = _system(n, 8)
    r[n - 1] = r[3]
    print(f"case small product coincident n={n} {prec}", flush=True)
    u, _ = wall_rpy.apply(RMW_UF, r, f, eta=ETA, a=A, precision=prec, tuning="heuristic")
    bad = ~torch.isfinite(u).all(dim=1)
    assert bool(bad[3]) and bool(bad[n - 1]) and int(bad.sum()) == 2


@pytest.mark.parametrize("n", [90, 2433])
def test_minimum_images_at_ties(gpu, n):
    """Blobs on a lattice of half the box, many boxes apart: d / L + 1/2 is a
    whole number, where the count of boxes must be that of the division."""
    rng = np.random.default_rng(n)
    L = np.array([16.0, 24.0, 0.0])
    boxes = rng.integers(-3, 4, (n, 2)) * np.where(rng.random((n, 1)) < 0.2, 1e5, 1.0)
    r = np.column_stack([rng.integers(0, 2, (n, 2)) * (L[:2] / 2) + boxes * L[:2], 0.75 * np.arange(1, n + 1)])
    f, t = rng.standard_normal((1, n, 3)), rng.standard_normal((1, n, 3))
    rows = (0, 90)
    want = [O.block_apply(blk, r, v[0], ETA, 0.5, L, rows=rows).reshape(n, 3)[:90] for blk, v in ((O.UF, f), (O.UT, t))]
    for prec in ("fp64", "fp32_blocked"):
        for tuning in ("heuristic", ORDERED, _lib.Tuning(256, 0, 0, 1, 0)):
            u, _ = wall_rpy.apply(RMW_UF | RMW_UT, r, force=f, torque=t, eta=ETA, a=0.5, precision=prec,
                                  periodic_length=L, tuning=tuning)
            ref = torch.as_tensor(want[0] + want[1]).to(u)
            assert rel(u.reshape(n, 3)[:90], ref) <= TOL[prec], (prec, tuning)
