"""The fused Arnoldi step (k bases per launch), the Lanczos step's square root
and the body preconditioner at the edges of their launch forms, against plain
FP64.

Tolerances: 1e-12 relative where sums of n products are compared, 1e-13 for the
coefficients of the square root (condition numbers up to 1e4), 1e-9 for the
inverse blocks as in the other preconditioner tests.
"""
import ctypes

import numpy as np
import pytest
import torch

from rigidmultiblobswall_amd import _lib, krylov, rigid

pytestmark = pytest.mark.gpu


def _stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("n,k,m", [(1, 1, 1), (255, 3, 2), (257, 2, 9), (5000, 4, 70), (140001, 2, 5), (300001, 3, 3),
                                   (1200007, 1, 2)])
def test_batched_arnoldi_step(gpu, n, k, m):
    """m orthonormal vectors per basis (fewer when n is smaller), one step, two
    workspaces: the one the query asks for and the one of a single set of
    partial sums, which takes the separate launches."""
    m = min(m, n)
    print(f"case arnoldi batch n={n} k={k} m={m}", flush=True)
    lib = _lib.load()
    g = torch.Generator(device="cpu").manual_seed(n + k)
    V0 = torch.zeros((m + 1, k, n), dtype=torch.float64)
    for r in range(k):
        V0[:m, r] = torch.linalg.qr(torch.randn((n, m), generator=g, dtype=torch.float64))[0].T
    w0 = torch.randn((k, n), generator=g, dtype=torch.float64)
    ops = krylov.KrylovOps(n, m + 1, gpu)
    short = torch.empty(512 * (m + 1) * 8, dtype=torch.uint8, device=gpu)
    for ws in (ops.ws, short):
        V, w = V0.to(gpu), w0.to(gpu)
        H = torch.full((k, m + 3), -5.0, dtype=torch.float64, device=gpu)
        hs = torch.empty(m + 2, dtype=torch.float64, device=gpu)
        _lib.check(lib.rmw_arnoldi_cgs2_batch(V.data_ptr(), k * n, n, m - 1, k, w.data_ptr(), n, n, H.data_ptr(), m + 3,
                                              hs.data_ptr(), ws.data_ptr(), ws.numel(), _stream()))
        for r in range(k):
            rec = V[:, r].T @ H[r, : m + 1]
            scale = float(torch.linalg.norm(w0[r]))
            assert float(torch.linalg.norm(rec.cpu() - w0[r])) <= 1e-12 * scale
            assert float((V[:m, r] @ V[m, r]).abs().max()) <= 1e-12 or n == m
            assert float(H[r, m + 1]) == -5.0 and float(H[r, m + 2]) == -5.0
            assert abs(float(torch.linalg.norm(V[m, r])) - 1.0) <= 1e-12


@pytest.mark.parametrize("m", [1, 2, 3, 7, 33, 63, 64, 65, 130])
def test_lanczos_square_root(gpu, m):
    lib = _lib.load()
    rng = np.random.default_rng(m)
    kinds = {"wide": (rng.uniform(1, 5, m), rng.uniform(0, 0.5, m)), "indefinite": (rng.standard_normal(m), rng.uniform(0, 1, m)),
             "nearly diagonal": (rng.uniform(1, 5, m), 1e-14 * rng.uniform(0, 1, m)),
             "split": (rng.uniform(1, 5, m), rng.uniform(0, 0.5, m) * (np.arange(m) % 3 > 0)),
             "large": (1e160 * rng.uniform(1, 5, m), 1e160 * rng.uniform(0, 0.5, m)),
             "equal": (np.full(m, 2.0), np.zeros(m))}
    H = torch.zeros((len(kinds), m, m + 1), dtype=torch.float64)
    ref = []
    for q, (d, e) in enumerate(kinds.values()):
        for i in range(m):
            H[q, i, i], H[q, i, i + 1] = d[i], e[i]
        T = np.diag(d) + np.diag(e[: m - 1], 1) + np.diag(e[: m - 1], -1)
        lam, Q = np.linalg.eigh(T)
        ref.append(2.0 * Q @ (np.sqrt(np.clip(lam, 0, None)) * Q[0]))
    k = len(kinds)
    H = H.to(gpu)
    sc = torch.full((k,), 2.0, dtype=torch.float64, device=gpu)
    C = torch.zeros((k, m + 2), dtype=torch.float64, device=gpu)
    if m > 1:
        C[:, : m - 1] = 0.25
    z = torch.empty(k * m * m, dtype=torch.float64, device=gpu)
    test = torch.empty((k, 3), dtype=torch.float64, device=gpu)
    print(f"case lanczos square root m={m}", flush=True)
    _lib.check(lib.rmw_lanczos_step_coeffs(H.data_ptr(), H.stride(0), H.stride(1), m, k, sc.data_ptr(), C.data_ptr(),
                                           C.stride(0), z.data_ptr(), z.numel(), test.data_ptr(), _stream()))
    got, t = C.cpu().numpy(), test.cpu().numpy()
    old = np.zeros(m)
    old[: m - 1] = 0.25
    for q, name in enumerate(kinds):
        n = np.linalg.norm(ref[q])
        assert np.linalg.norm(got[q, :m] - ref[q]) <= 1e-13 * max(n, 1e-300) * np.sqrt(m), name
        assert abs(t[q, 0] - np.linalg.norm(ref[q] - old)) <= 1e-12 * max(n, 1.0), name
        assert abs(t[q, 1] - np.linalg.norm(old)) <= 1e-14 and t[q, 2] == 0.0, name
        assert (got[q, m:] == 0).all()


@pytest.mark.parametrize("sizes", [[1], [2, 1, 5], [11, 16, 6, 21], [42, 45, 40], [45, 50, 1]])
def test_preconditioner_of_bodies_of_every_block_size(gpu, sizes):
    """Bodies whose blocks end inside and at the edges of the threads' element
    blocks; one blob and two blobs have a singular K^T M^-1 K (pseudo-inverse
    by rotations)."""
    rng = np.random.default_rng(sum(sizes))
    refs = []
    for nb in sizes:
        i = np.arange(nb) + 0.5
        z = 1 - 2 * i / nb
        ph = 2.4 * i
        s = np.sqrt(1 - z * z)
        refs.append(np.column_stack([s * np.cos(ph), s * np.sin(ph), z]) if nb > 2 else
                    np.column_stack([np.zeros(nb), np.zeros(nb), np.arange(nb) * 1.0]))
    B = len(sizes)
    loc = np.column_stack([4.0 * np.arange(B), np.zeros(B), np.full(B, 2.2)])
    q = rng.standard_normal((B, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    print(f"case preconditioner bodies {sizes}", flush=True)
    S = rigid.RigidSuspension(loc, q, refs, 1.0, 0.24)
    S.build_preconditioner()
    r, rel = S.r_blobs.cpu().numpy(), S.r_rel.cpu().numpy()
    x = torch.from_numpy(rng.standard_normal(S.size)).to(gpu)
    y = torch.empty_like(x)
    S.pc_apply(x, y)
    xs, ys, off, moff = x.cpu().numpy(), y.cpu().numpy(), 0, 0
    minv, nbody = S.minv.cpu().numpy(), S.nbody.cpu().numpy()
    from oracle import oracle as O
    for b, nb in enumerate(sizes):
        n = 3 * nb
        M = O.single_wall_fluid_mobility(r[off:off + nb], 1.0, 0.24)
        K = O.K_matrix(rel[off:off + nb])
        Mi = np.linalg.inv(M)
        N = np.linalg.pinv(K.T @ Mi @ K)
        got = minv[moff:moff + n * n].reshape(n, n)
        assert np.abs(got - Mi).max() <= 1e-9 * np.abs(Mi).max()
        assert np.abs(nbody[b] - N).max() <= 1e-9 * np.abs(N).max()
        s, F = xs[3 * off:3 * off + n], xs[3 * S.Nblobs + 6 * b:3 * S.Nblobs + 6 * b + 6]
        Y = N @ (-F - K.T @ (Mi @ s))
        assert np.abs(ys[3 * S.Nblobs + 6 * b:3 * S.Nblobs + 6 * b + 6] - Y).max() <= 1e-9 * np.abs(Y).max()
        lam = Mi @ (s + K @ Y)
        assert np.abs(ys[3 * off:3 * off + n] - lam).max() <= 1e-9 * np.abs(Mi @ s).max()
        off += nb
        moff += n * n


@pytest.mark.parametrize("m", [1, 59, 60, 61, 78, 79, 156, 157, 267, 268, 269, 327, 328, 400])
def test_square_root_storage_edges(gpu, m):
    """Sizes at which fewer nodes fit into LDS at a time, or none, for a
    positive definite T and one with a negative eigenvalue."""
    print(f"case square root m={m}", flush=True)
    lib = _lib.load()
    rng = np.random.default_rng(m)
    k = 2
    a, b = rng.uniform(2.5, 30.0, (k, m)), rng.uniform(0.0, 1.2, (k, m))
    a[1, m // 2] = -4.0
    H = torch.zeros((k, m, m + 1), dtype=torch.float64)
    want = []
    for r in range(k):
        T = np.diag(a[r]) + np.diag(b[r, :-1], 1) + np.diag(b[r, :-1], -1)
        lam, Q = np.linalg.eigh(T)
        want.append(Q @ (np.sqrt(np.maximum(lam, 0)) * Q[0]))
        H[r, np.arange(m), np.arange(m)] = torch.from_numpy(a[r])
        H[r, np.arange(m), np.arange(m) + 1] = torch.from_numpy(b[r])
    H = H.to(gpu)
    C = torch.zeros((k, m), dtype=torch.float64, device=gpu)
    sc = torch.ones(k, dtype=torch.float64, device=gpu)
    status = torch.full((k,), 7, dtype=torch.int32, device=gpu)
    scr = torch.empty(k * m * m, dtype=torch.float64, device=gpu)
    _lib.check(lib.rmw_lanczos_sqrt_coeffs(H.data_ptr(), H.stride(0), H.stride(1), m, k, sc.data_ptr(), C.data_ptr(), m,
                                           scr.data_ptr(), scr.numel(), status.data_ptr(), _stream()))
    assert status.tolist() == [0, 0]
    for r in range(k):
        assert np.linalg.norm(C[r].cpu().numpy() - want[r]) <= 1e-13 * max(np.linalg.norm(want[r]), 1.0)
