"""Drop-in products on numpy arrays that go through one pinned buffer, against
the same products on device tensors: the same launches, so the same bits; and
the inputs that this way does not take, which the general one must still serve
or refuse."""
import threading

import numpy as np
import pytest
import torch

from rigidmultiblobswall_amd import mobility, wall_rpy

pytestmark = pytest.mark.gpu

UF = mobility.single_wall_mobility_trans_times_force_hip
ONE = [UF, mobility.single_wall_mobility_trans_times_torque_hip, mobility.single_wall_mobility_rot_times_force_hip,
       mobility.single_wall_mobility_rot_times_torque_hip, mobility.no_wall_mobility_trans_times_force_hip,
       mobility.no_wall_mobility_trans_times_torque_hip, mobility.no_wall_mobility_rot_times_force_hip,
       mobility.no_wall_mobility_rot_times_torque_hip, mobility.in_plane_mobility_trans_times_force_hip,
       mobility.in_plane_mobility_trans_times_torque_hip, mobility.free_surface_mobility_trans_times_force_hip]
TWO = [mobility.single_wall_mobility_trans_times_force_torque_hip,
       mobility.no_wall_mobility_trans_times_force_torque_hip]


def _system(n, seed=0):
    rng = np.random.default_rng(seed + n)
    r = np.column_stack([rng.uniform(0, 2 * np.sqrt(n), (n, 2)), rng.uniform(0.3, 4.0, n)])
    return r, rng.standard_normal((n, 3)), rng.standard_normal(3 * n)


def _tensor(*xs):
    return [torch.as_tensor(x).cuda() for x in xs]


@pytest.mark.parametrize("n", [1, 172, 1024, 1025, 2400, 8738, 14563, 14564])
def test_same_bits_as_device_tensors(gpu, n):
    print(f"case host product n={n}", flush=True)
    r, f, t = _system(n)
    for fn in ONE if n < 2000 else ONE[:1]:
        assert np.array_equal(fn(r, t, 0.9, 0.4), fn(*_tensor(r, t), 0.9, 0.4)), fn.__name__
    for fn in TWO:
        assert np.array_equal(fn(r, f, t, 0.9, 0.4), fn(*_tensor(r, f, t), 0.9, 0.4)), fn.__name__
    ft = np.concatenate([f.reshape(-1), t])
    for prec in ("fp32", "fp64"):
        for L in (np.zeros(3), np.array([30.0, 0.0, 0.0])) if n < 2000 else (np.zeros(3),):
            kw = dict(precision=prec, periodic_length=L)
            want = mobility.single_wall_grand_mobility_hip(*_tensor(r, ft), 0.9, 0.4, **kw)
            got = mobility.single_wall_grand_mobility_hip(r, ft, 0.9, 0.4, **kw)
            assert np.array_equal(got, want) and got.flags.writeable and got.flags.owndata


def test_inputs_of_other_forms(gpu):
    n = 60
    r, f, _ = _system(n)
    want = UF(r, f, 0.9, 0.4)
    wide = np.zeros((n, 6))
    wide[:, ::2] = f
    for g in (f.astype(np.float32).astype(np.float64), f.reshape(-1), np.asfortranarray(f), wide[:, ::2], f.tolist(),
              torch.from_numpy(f)):
        ref = UF(*_tensor(r, g), 0.9, 0.4)   # (torch takes a list as float32)
        assert np.array_equal(UF(r, g, 0.9, 0.4), ref)
    assert np.array_equal(UF(r, f, 0.9, 0.4, check_finite=True), want)
    assert UF(np.zeros((0, 3)), np.zeros(0), 0.9, 0.4).shape == (0,)
    for bad in (f[:-1], f.reshape(-1)[:-1], np.zeros((n + 1, 3))):
        with pytest.raises(ValueError):
            UF(r, bad, 0.9, 0.4)
    for kw in (dict(eta=-1.0, a=0.4), dict(eta=1.0, a=0.0)):
        with pytest.raises(Exception):
            UF(r, f, **kw)
    assert np.array_equal(UF(r, f, 0.9, 0.4), want)


@pytest.mark.parametrize("own_stream", [True, False])
def test_threads_and_streams(gpu, own_stream):
    systems = [_system(n) for n in (50, 300, 2500, 1500)]
    want = [UF(r, f, 0.9, 0.4) for r, f, _ in systems]
    wrong = []

    def work(q):
        with torch.cuda.stream(torch.cuda.Stream() if own_stream else torch.cuda.default_stream()):
            for _ in range(20):
                if not np.array_equal(UF(*systems[q][:2], 0.9, 0.4), want[q]):
                    wrong.append(q)

    threads = [threading.Thread(target=work, args=(q,)) for q in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not wrong and len(wall_rpy._stages) <= wall_rpy._STAGES
