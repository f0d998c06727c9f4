"""The blob forces by cells and in one launch, against the kernels over all
pairs (which the other tests hold to the oracle): open and periodic boxes, the
cutoff, different radii, boxes of few cells, blobs outside the box, dense
suspensions, which fall back to all pairs, and positions that do not fit the
cell arithmetic.

Each test names the route that its calls must take, read from the counters the
cells leave in the workspace.

Tolerances: the terms are the same, only the order of FP64 sums differs:
1e-12; the FP32 exponential does not change that.
"""
import numpy as np
import pytest
import torch

from rigidmultiblobswall_amd import _lib, forces, wall_rpy

pytestmark = pytest.mark.gpu

ALL_PAIRS = _lib.Tuning(256, 0, 0, -1, 0)
EPS, B, A = 0.3, 0.07, 0.6


def _layout(n, seed, spread=1.6, flat=True):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (0.5 if flat else 1 / 3)))
    idx = rng.permutation(m ** (2 if flat else 3))[:n]
    g = np.stack([idx % m, (idx // m) % m, idx // m ** 2 if not flat else 0 * idx], axis=1) * spread
    return g + rng.uniform(-0.5, 0.5, (n, 3)) - 0.3 * m * spread      # about a third below zero


def _rel(a, b):
    return float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))


def _route(r, prec, **kw):
    """The route of one call: 'cells' gave the forces, 'all pairs' the launches
    after the cells' counts, 'no cells' without any (one launch, or the host
    knew).  The counters lie behind the partial sums of the kernel over all
    pairs, symmetric from 23 tiles of 256 blobs on."""
    n = r.shape[0]
    call = lambda: forces.blob_forces(r, EPS, kw["b"], A, precision=prec,   # noqa: E731
                                      **{k: v for k, v in kw.items() if k != "b"})
    call()      # sizes the workspace
    ws = wall_rpy.workspace(1, slot="forces")
    off = forces.describe(n, prec, _lib.Tuning(0, 0, 0, 1 if -(-n // 256) >= 23 else -1, 0))["workspace_bytes"]
    if off + 16 > ws.numel():
        return "no cells"
    ws.fill_(0xFF)
    call()
    cursor, unfit = ws[off:off + 8].view(torch.int32).tolist()
    pairs = ws[off + 8:off + 16].view(torch.int64).item()
    if cursor == -1 and unfit == -1 and pairs == -1:
        return "no cells"
    return "cells" if unfit == 0 and pairs <= n * n // 4 else "all pairs"


def _check(r, what, L=None, cutoff=0.0, radii=None, b=B, tol=1e-12, route=None):
    for prec in ("fp32", "fp64"):
        print(f"case forces {what} n={r.shape[0]} L={L} cutoff={cutoff:.3g} {prec}", flush=True)
        kw = dict(periodic_length=L, cutoff=cutoff, radius_blobs=radii, precision=prec)
        got = forces.blob_forces(r, EPS, b, A, **kw)
        ref = forces.blob_forces(r, EPS, b, A, tuning=ALL_PAIRS, **kw)
        assert _rel(got, ref) <= tol, (what, prec, _rel(got, ref))
        assert torch.equal(got, forces.blob_forces(r, EPS, b, A, **kw))   # the same sums every time
        if route is not None:
            assert _route(r, kw.pop("precision"), b=b, **kw) == route, (what, prec)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 255, 257, 1000, 4096, 4097, 5003])
def test_sizes(gpu, n):
    if n > 1:
        _check(_layout(n, n), "open")
        _check(_layout(n, n, flat=False), "open 3d", cutoff=2 * A + 30 * B)
    else:
        assert bool((forces.blob_forces(_layout(1, 1), EPS, B, A) == 0).all())


@pytest.mark.parametrize("n", [700, 6001])
def test_periodic_boxes(gpu, n):
    r = _layout(n, 3)
    side = 1.6 * np.ceil(np.sqrt(n))
    cut = 2 * A + 30 * B
    # whole numbers of cells from 1 up, sides below and just above the range
    for L in [(side, side, 0), (side, 0, 0), (0, side, 3.0), (3 * cut * 1.001, side, 0), (2.9 * cut, 4.05 * cut, 0),
              (1.5 * cut, side, 2 * cut), (0, 0, 7 * cut)]:
        _check(r, "periodic", L=np.array(L, dtype=float), cutoff=cut)
    _check(r, "periodic, no cutoff", L=np.array([side, side, 0.0]))
    shifted = r + np.random.default_rng(1).integers(-3, 4, r.shape) * np.array([side, side, 0.0])
    _check(shifted, "outside the box", L=np.array([side, side, 0.0]), cutoff=cut)


def test_radii_with_a_cutoff_and_without(gpu):
    r = _layout(6301, 5)
    rad = np.random.default_rng(6).uniform(0.3, 0.8, 6301)
    _check(r, "radii, cutoff", cutoff=3.5, radii=rad, route="cells")
    _check(r, "radii", radii=rad, route="no cells")


@pytest.mark.parametrize("n", [6301, 9001])
def test_cells_that_pay(gpu, n):
    """Up to and beyond the size at which the kernel over all pairs changes;
    without the cutoff the range of the FP64 exponential, 746 b, is short
    enough for small b."""
    r = _layout(n, n + 1)
    _check(r, "cutoff", cutoff=2 * A + 30 * B, route="cells")
    _check(r, "short range", b=0.01, route="cells")
    side = 1.6 * np.ceil(np.sqrt(n))
    _check(r, "short range, periodic", b=0.01, L=np.array([side, side, 0.0]), route="cells")
    _check(r, "cutoff, periodic", cutoff=2 * A + 30 * B, L=np.array([side, side, 0.0]), route="cells")


@pytest.mark.parametrize("n", [6301, 9001])
def test_dense_suspensions_take_all_pairs(gpu, n):
    r = _layout(n, 7, spread=0.05)
    _check(r, "dense", b=1.0, route="all pairs")
    _check(np.vstack([r, r[:3]]), "dense with coincident blobs", b=1.0, route="all pairs")
    L = np.array([5.0, 5.0, 0.0])
    _check(r, "dense periodic", L=L, b=1.0, route="no cells")
    _check(r, "dense periodic in one direction", L=np.array([5.0, 0.0, 0.0]), b=1.0, route="all pairs")


@pytest.mark.parametrize("n", [6400, 9002])
def test_clusters_in_few_cells(gpu, n):
    """Two clusters far apart: every blob in one of two cells (half of all
    pairs), next to an otherwise empty suspension; then every second blob in
    a dilute one (waves with blobs of one cell and of many); then clusters of
    a few blobs (waves with a few blobs to a cell)."""
    rng = np.random.default_rng(8)
    r = np.vstack([rng.uniform(0, 1.0, (n // 2, 3)), rng.uniform(0, 1.0, (n // 2, 3)) + 500.0])
    _check(r, "two clusters", cutoff=3.0, route="all pairs")
    r[1::2] = _layout(n // 2, 9, spread=40.0)
    _check(r, "cluster and dilute", cutoff=3.0, route="cells")
    r = np.repeat(_layout(n // 10 + 1, 10, spread=40.0), 10, axis=0)[:n] + rng.uniform(0, 1.0, (n, 3))
    _check(r, "clusters of ten in order", cutoff=3.0, route="cells")
    _check(r[rng.permutation(n)], "clusters of ten", cutoff=3.0, route="cells")


@pytest.mark.parametrize("n", [6301, 9001])
def test_positions_that_do_not_fit(gpu, n):
    r = _layout(n, 10)
    far = r.copy()
    far[17] = [1e12, -3e9, 5.0]
    _check(far, "far blob", route="all pairs")
    _check(far, "far blob, periodic", L=np.array([200.0, 200.0, 0.0]), cutoff=3.3, tol=1e-9, route="all pairs")
    for bad in (np.nan, np.inf):
        x = r.copy()
        x[4321, 1] = bad
        for prec in ("fp32", "fp64"):
            print(f"case forces {bad} n={n} {prec}", flush=True)
            got = forces.blob_forces(x, EPS, B, A, precision=prec)
            ref = forces.blob_forces(x, EPS, B, A, precision=prec, tuning=ALL_PAIRS)
            assert bool((torch.isfinite(got) == torch.isfinite(ref)).all())
            assert _route(x, prec, b=B) == "all pairs"
