"""Layouts of the symmetric wall products next to the limits of their partial
sums (2 GiB for a workspace, 64 MiB for the library's own array): the tiles take
over where the blocks' sums do not fit, all right-hand sides of a pass are kept
while a layout has room for them, and the ordered kernel comes last.

The layout is read from the workspace that a call asks for.  Tolerance of the
products: 1e-6 as between all routes in the blocked mode (the pair terms are
FP32, the order of their sums differs).
"""
import ctypes
import re

import numpy as np
import pytest
import torch

from rigidmultiblobswall_amd import _lib, wall_rpy

pytestmark = pytest.mark.gpu

CU = 256
GRAND = 15


def _slots(sizes, bs, run):
    """Target-side and source-side slots: rows of m tiles in runs of `run`
    64-source blocks (of tiles for bs = 64, as one is a block)."""
    per = bs // 64
    total = 0
    for n in sizes:
        nt = -(-n // bs)
        total += sum(-(-(m * per) // run) for m in range(1, nt + 1)) + nt * (nt + 1) // 2
    return total


def _ragged_bytes(sizes, k, mask=GRAND):
    """What a call without images asks for when it gets no workspace (the size
    query also covers the layout with images); nothing is launched."""
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    lib = _lib.load()
    rc = lib.rmw_wall_rpy_ragged_apply(mask, _lib.precision_code("fp32_blocked"), None, None, None, None, None,
                                       off.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), len(sizes), k, 0, 1.0, 0.5,
                                       None, None, None, 0, None)
    assert rc == _lib.RMW_E_ARG
    return int(re.search(r"need (\d+) bytes", lib.rmw_last_error().decode()).group(1))


MIXED = list(np.random.default_rng(5).integers(128, 4097, 512))


@pytest.mark.parametrize("sizes,k,kpass,bs,run", [
    ([4096] * 64, 4, 4, 64, 4),         # the blocks' sums fit: 1.9 GiB
    ([4096] * 96, 4, 4, 256, 4),        # blocks 2.9 GiB, tiles 1.2
    ([4096] * 192, 2, 2, 256, 8),       # blocks 2.9, tiles 0.9
    ([4096] * 192, 4, 4, 256, 8),       # blocks 5.8, tiles 1.8
    ([4096] * 236, 4, 4, 256, 28),      # tiles in short runs 2.2, in long ones 1.8
    ([4096] * 300, 4, 2, 256, 12),      # four right-hand sides 2.2 at least
    ([4096] * 300, 1, 1, 256, 12),      # blocks 2.3, tiles 0.6
    (MIXED, 4, 4, 256, 8),
], ids=["64x4096k4", "96x4096k4", "192x4096k2", "192x4096k4", "236x4096k4", "300x4096k4", "300x4096k1", "512mixedk4"])
def test_batches_keep_a_symmetric_layout(gpu, sizes, k, kpass, bs, run):
    assert wall_rpy.device_info()["cu_count"] == CU
    got, want = _ragged_bytes(sizes, k), _slots(sizes, bs, run) * kpass * bs * 6 * 8
    print(f"case {len(sizes)} systems k={k}: {got} bytes, layout {want}", flush=True)
    # beside the sums: the table of the systems and room for the outputs
    assert want <= got <= want + 64 * len(sizes) + 48 * k * sum(sizes) + 4096
    assert want <= 2 << 30


def test_batch_by_tiles_equals_its_systems(gpu):
    """96 systems of 4096 blobs, four right-hand sides: three of the systems
    by themselves (blocks)."""
    n, S, k = 4096, 96, 4
    g = torch.Generator(device="cpu").manual_seed(3)
    r = torch.rand((S * n, 3), generator=g, dtype=torch.float64) * torch.tensor([106.0, 106.0, 1.2], dtype=torch.float64)
    r = (r + torch.tensor([0.0, 0.0, 0.8], dtype=torch.float64)).to(gpu)
    f = torch.randn((k, S * n, 3), generator=g, dtype=torch.float64).to(gpu)
    t = torch.randn((k, S * n, 3), generator=g, dtype=torch.float64).to(gpu)
    kw = dict(eta=1e-3, a=0.656, k=k, precision="fp32_blocked")
    u, w = wall_rpy.apply_ragged(GRAND, r, np.arange(S + 1) * n, force=f, torque=t, **kw)
    for s in (0, 41, 95):
        sl = slice(s * n, (s + 1) * n)
        us, ws = wall_rpy.apply(GRAND, r[sl].contiguous(), force=f[:, sl].contiguous(), torque=t[:, sl].contiguous(), **kw)
        assert float(torch.linalg.norm(u[:, sl] - us) / torch.linalg.norm(us)) <= 1e-6
        assert float(torch.linalg.norm(w[:, sl] - ws) / torch.linalg.norm(ws)) <= 1e-6


@pytest.mark.parametrize("mask,k,n", [(1, 1, 22500), (1, 1, 26000), (15, 1, 15000), (15, 4, 7000)])
def test_products_without_a_workspace_stay_symmetric(gpu, mask, k, n):
    """Sizes whose preferred tiles do not fit the library's array while longer
    runs do: the same bits as the product with a workspace whose tuning asks
    for the symmetric kernel in those runs."""
    lib = _lib.load()
    rng = np.random.default_rng(n)
    side = 300.0 * np.sqrt(n / 32768.0)
    r = torch.from_numpy(np.column_stack([rng.uniform(0, side, (n, 2)), rng.uniform(0.8, 2.0, n)])).to(gpu)
    f, t = (torch.from_numpy(rng.standard_normal((k, n, 3))).to(gpu) for _ in range(2))
    u, w = torch.empty_like(f), torch.empty_like(f)
    _lib.check(lib.rmw_wall_rpy_apply_noalloc(mask, _lib.precision_code("fp32_blocked"), r.data_ptr(), f.data_ptr(),
                                              t.data_ptr(), u.data_ptr(), w.data_ptr(), n, k, 0, 1e-3, 0.656,
                                              (ctypes.c_double * 3)(0, 0, 0), None,
                                              torch.cuda.current_stream().cuda_stream))
    nt = -(-n // 256)
    run = 256 * max(1, nt * (nt + 1) // 2 // (16 * CU))
    us, ws = wall_rpy.apply(mask, r, force=f, torque=t, eta=1e-3, a=0.656, k=k, precision="fp32_blocked",
                            tuning=dict(symmetric=1, chunk_len=run))
    assert torch.equal(u.reshape(-1), us.reshape(-1))
    if mask == GRAND:
        assert torch.equal(w.reshape(-1), ws.reshape(-1))
