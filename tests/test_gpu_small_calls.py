"""The single-species operator on both sides of the lines by (function, task,
direction, radius) count: the form of the Nyquist planes (256 or 512) and the
loads in flight of the gain's staging (1024), f = g and f != g, the twofold
residue split, and the reference-state form, against the FP64 oracle.

States carry 5 % noise, so that the Nyquist planes hold as much as the rest.
Tolerances as the direct form's everywhere: 1e-11 (FP64) and 3e-5 (FP32) of
max|Q|; 1e-6 in the reference-state form, which is as exact as its FP32 result
(2^-24 of the terms added: Q0, G and L of a 1 % deviation)."""
import numpy as np
import pytest

from oracle import collision as OC
from oracle import velocitymesh as OVM

pytestmark = pytest.mark.gpu

M, NRHO = 6, 3                                       # 18 (direction, radius) per function


def _setup(N):
    vm = OVM.VelocityMesh(1e-3, 273.0, 2.3e-4, 39.96e-3, N, NRHO, 0.0, 273.0, 5.0, M)
    gamma = 2 * (1 - 0.81)
    rng = np.random.default_rng(N)
    u = np.stack([np.exp(-((vm.cv - rng.uniform(-0.4, 0.4, (3, 1))) ** 2).sum(0) /
                         rng.uniform(0.8, 1.3)) * (1 + 0.05 * rng.uniform(-1, 1, N ** 3))
                  for _ in range(3)])
    return vm, gamma, u, OC.Precomp(N, vm.L, vm.qz, vm.qw, vm.sz, vm.sw, gamma)


def _plan(cuda, vm, gamma, N, code, ntask):
    from dgfs1d_gpu_amd import _lib
    from dgfs1d_gpu_amd.collision import CollisionPlan
    return CollisionPlan(N, M, NRHO, vm.L, vm.qz, vm.qw, vm.sz, vm.sw, gamma, 0.7, code,
                         _lib.VHS, ntask, device=cuda)


@pytest.mark.parametrize('N,dtype', [(12, 'F32'), (12, 'F64'), (16, 'F64'), (20, 'F32'),
                                     (20, 'F64'), (24, 'F32'), (24, 'F64'), (32, 'F32'),
                                     (32, 'F64'), (48, 'F32')])
@pytest.mark.parametrize('functions', [1, 2])
def test_counts(cuda, monkeypatch, N, dtype, functions):
    """functions = 2: f != g, so that a task counts twice."""
    import torch
    from dgfs1d_gpu_amd import _lib, collision
    monkeypatch.setattr(collision, 'PAIR_WORK', 1 << 62)       # tasks repeat three slices
    vm, gamma, u, pre = _setup(N)
    td = torch.float64 if dtype == 'F64' else torch.float32
    pairs = [(0, 0), (1, 1), (2, 2)] if functions == 1 else [(0, 1), (1, 2), (2, 0)]
    ref = np.stack([OC.q_vhs(pre, u[a], u[b], 0.7) for a, b in pairs])
    tol = (1e-11 if dtype == 'F64' else 3e-5) * np.abs(ref).max()
    for line in (256, 512, 1024):
        below = (line - 1) // (18 * functions)
        for nt in (below, below + 1):
            plan = _plan(cuda, vm, gamma, N, getattr(_lib, dtype), nt)
            plan.set_tasks(nt, 1, [(o, [(pairs[o % 3][0], 1.0)], [(pairs[o % 3][1], 1.0)])
                                   for o in range(nt)])
            d = torch.zeros(nt, N ** 3, dtype=td, device=cuda)
            d[:3] = torch.tensor(u, dtype=td, device=cuda)
            for split in (1, 2) if functions == 1 else (1,):
                plan.set_schedule(split, 1)
                Q = torch.zeros_like(d)
                plan(d, Q)
                got = Q.double().cpu().numpy()
                err = max(np.abs(got[o] - ref[o % 3]).max() for o in range(nt))
                print(N, dtype, functions, nt * 18 * functions, split, err / np.abs(ref).max(),
                      flush=True)
                assert err < tol
            plan.close()


@pytest.mark.parametrize('N', [16, 24, 32])
def test_reference_counts(cuda, N):
    import torch
    from dgfs1d_gpu_amd import _lib
    vm, gamma, u, pre = _setup(N)
    u0 = u.astype(np.float32)
    u1 = (0.99 * u0 + 0.01 * np.roll(u0, 1, 0)).astype(np.float32)
    q = [OC.q_vhs(pre, f.astype(np.float64), f.astype(np.float64), 0.7) for f in u1]
    q0 = np.stack([OC.q_vhs(pre, f.astype(np.float64), f.astype(np.float64), 0.7) for f in u0])
    most = max(np.abs(x).max() for x in q)
    for line in (256, 512, 1024):
        for nt in ((line - 1) // 18, (line - 1) // 18 + 1):
            plan = _plan(cuda, vm, gamma, N, _lib.F32, nt)
            plan.set_tasks(nt, 1, [(s, [(s, 1.0)], [(s, 1.0)]) for s in range(nt)])
            at = [s % 3 for s in range(nt)]
            d0 = torch.tensor(u0[at], device=cuda)
            d1 = torch.tensor(u1[at], device=cuda)
            Q0 = torch.tensor(q0[at], device=cuda)
            Q = torch.zeros_like(d1)
            plan.reference_set(d0)
            plan.reference(d1, d0, Q0, Q)
            got = Q.double().cpu().numpy()
            err = max(np.abs(got[s] - q[s % 3]).max() for s in range(nt)) / most
            print('reference', N, nt * 18, err, flush=True)
            assert err < 1e-6
            plan.close()
