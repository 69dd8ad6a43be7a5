"""The mixture operator's streaming kernels (packed real transforms, Hermitian
half of the products, paired directions) against the FP64 oracle and against
each other, at the forms they accept: N = 20, 24, 32 with one and two lanes per
plane row, rules with and without opposite directions, the like-species call,
task chunks and several group and x-range splits.

States carry 5 % noise, so that the Nyquist planes hold as much as the rest.
Tolerances as tests/test_gpu_bivss.py: 1e-11 (FP64) and 3e-5 (FP32) of
max|Q|; results that only differ in the order of sums agree to 1e-13."""
import numpy as np
import pytest

from oracle import bivss as OB
from oracle.velocitymesh import load_design
from test_gpu_bivss import TASKS, _fields, _mesh

pytestmark = pytest.mark.gpu


def _rule(M, antipodal):
    if antipodal:
        return load_design('womersley', M)
    p = np.random.default_rng(M).standard_normal((M, 3))
    return p / np.linalg.norm(p, axis=1)[:, None]


def _call(cuda, N, M, antipodal, dtype, p, q, ntask_max, tasks=TASKS, masses=None, like=False,
          Nrho=3, oracle=True):
    """Q of one call, its error against the oracle, and the plan's query."""
    import torch
    from dgfs1d_gpu_amd import _lib
    from dgfs1d_gpu_amd.collision import BiCollisionPlan
    vm = _mesh(N, 6, Nrho)
    sz, szpre = _rule(M, antipodal), load_design('womersley', 32)
    m = masses or vm.masses
    u = _fields(vm, 2, 2, 11)
    plan = BiCollisionPlan(N, M, Nrho, vm.L, vm.qz, vm.qw, sz, vm.sw, szpre, m[p], m[q], 1.36,
                           0.8, 0.41, dtype, ntask_max, device=cuda)
    plan.set_tasks(2, 2, tasks)
    td = torch.float64 if dtype == _lib.F64 else torch.float32
    up = torch.tensor(u[p], dtype=td, device=cuda)
    uq = up if like else torch.tensor(u[q], dtype=td, device=cuda)
    Q = torch.full((4, N ** 3), 0.25, dtype=td, device=cuda)
    plan(up, uq, Q)
    got = Q.double().cpu().numpy() - 0.25
    info = plan.query()
    plan.close()
    err = None
    if oracle:
        pre = OB.BiPrecomp(N, vm.L, vm.qz, vm.qw, sz, vm.sw, szpre, m[p], m[q], 1.36, 0.8)
        ref = np.zeros_like(got)
        for out, ft, gt in tasks:
            ref[out] += OB.q_pq(pre, sum(c * u[p][s] for s, c in ft),
                                sum(c * u[q][s] for s, c in gt), 0.41)
        err = np.abs(got - ref).max() / np.abs(ref).max()
    return got, err, info


@pytest.mark.parametrize('N,dtype', [(20, 'F64'), (20, 'F32'), (24, 'F64'), (24, 'F32'),
                                     (32, 'F64'), (32, 'F32')])
@pytest.mark.parametrize('M,antipodal', [(6, True), (5, False), (1, False)])
def test_rules(cuda, N, dtype, M, antipodal):
    from dgfs1d_gpu_amd import _lib
    # a task capacity whose product cubes exceed the streaming line at N = 20, 24
    got, err, info = _call(cuda, N, M, antipodal, getattr(_lib, dtype), 0, 1, 400 // M)
    print(N, dtype, M, antipodal, err, info, flush=True)
    assert err < (1e-11 if dtype == 'F64' else 3e-5)


# singular triplets of symmetric 2 x 2 couplings (degenerate and not), and a
# single-slice task with unequal coefficients
TRIPLETS = [(0, [(0, 1.0)], [(1, 0.7)]), (0, [(1, 1.0)], [(0, 0.7)]),
            (1, [(0, 0.8), (1, 0.6)], [(0, 0.8), (1, 0.6)]),
            (1, [(0, -0.6), (1, 0.8)], [(0, 0.3), (1, -0.4)]), (3, [(2, 0.5)], [(2, 3.0)])]
SAME = [(0, [(0, 1.0)], [(0, 1.0)]), (1, [(1, 0.5), (3, 0.25)], [(1, 0.5), (3, 0.25)]),
        (1, [(2, -1.0)], [(2, -1.0)])]


@pytest.mark.parametrize('N,dtype', [(20, 'F64'), (24, 'F32'), (32, 'F64')])
@pytest.mark.parametrize('M,antipodal', [(6, True), (5, False)])
@pytest.mark.parametrize('tasks', ['same', 'triplets'])
def test_like_species(cuda, N, dtype, M, antipodal, tasks):
    """up is uq and the tasks of each output symmetric in f and g: one product
    per opposite pair; the same table with another array takes the general
    form."""
    from dgfs1d_gpu_amd import _lib
    d = getattr(_lib, dtype)
    todo = SAME if tasks == 'same' else TRIPLETS
    a, err, _ = _call(cuda, N, M, antipodal, d, 1, 1, 400 // M, todo, like=True)
    b, _, _ = _call(cuda, N, M, antipodal, d, 1, 1, 400 // M, todo, oracle=False)
    diff = np.abs(a - b).max() / np.abs(b).max()
    print(N, dtype, M, err, diff, flush=True)
    assert err < (1e-11 if dtype == 'F64' else 3e-5)
    assert diff < (1e-13 if dtype == 'F64' else 3e-5)


def test_one_species_with_unsymmetric_tasks(cuda):
    """up is uq, but f and g do not exchange: the general form."""
    from dgfs1d_gpu_amd import _lib
    a, err, _ = _call(cuda, 20, 6, True, _lib.F64, 0, 0, 70, TASKS, like=True)
    assert err < 1e-11


def test_like_call_of_unequal_masses(cuda):
    """The like form needs equal masses: with others the call is the general one."""
    from dgfs1d_gpu_amd import _lib
    a, err, _ = _call(cuda, 20, 6, True, _lib.F64, 0, 0, 70, SAME, masses=[1.0, 2.0], like=True)
    assert err < 1e-11


@pytest.mark.parametrize('N,dtype', [(20, 'F64'), (24, 'F32'), (16, 'F64')])
def test_engine_and_streaming_agree(cuda, N, dtype):
    """The same call from a plan below and one above the line between the two
    forms (N <= 16: always the engine)."""
    from dgfs1d_gpu_amd import _lib
    d = getattr(_lib, dtype)
    a, ea, ia = _call(cuda, N, 6, True, d, 0, 1, len(TASKS))
    b, eb, ib = _call(cuda, N, 6, True, d, 0, 1, 80)
    diff = np.abs(a - b).max() / np.abs(a).max()
    print(N, dtype, ea, eb, diff, ia, ib, flush=True)
    assert max(ea, eb) < (1e-11 if dtype == 'F64' else 3e-5)
    assert diff < (1e-13 if dtype == 'F64' else 3e-5)


@pytest.mark.parametrize('ratio', [1e-6, 1e5])
def test_trace_species(cuda, ratio):
    """Species of very different densities share a transform: each keeps its own
    relative precision (FP32; the oracle is bilinear in the densities)."""
    import torch
    from dgfs1d_gpu_amd import _lib
    from dgfs1d_gpu_amd.collision import BiCollisionPlan
    N, M, Nrho = 32, 6, 3
    vm = _mesh(N, M, Nrho)
    sz, szpre, m = load_design('womersley', M), load_design('womersley', 32), vm.masses
    u = _fields(vm, 2, 2, 11)
    plan = BiCollisionPlan(N, M, Nrho, vm.L, vm.qz, vm.qw, sz, vm.sw, szpre, m[0], m[1], 1.36,
                           0.8, 0.41, _lib.F32, 1, device=cuda)
    plan.set_tasks(2, 2, [(0, [(0, 1.0)], [(1, 1.0)])])
    up = torch.tensor(u[0] * ratio, dtype=torch.float32, device=cuda)
    uq = torch.tensor(u[1], dtype=torch.float32, device=cuda)
    Q = torch.zeros_like(up)
    plan(up, uq, Q)
    pre = OB.BiPrecomp(N, vm.L, vm.qz, vm.qw, sz, vm.sw, szpre, m[0], m[1], 1.36, 0.8)
    ref = OB.q_pq(pre, u[0][0] * ratio, u[1][1], 0.41)
    err = np.abs(Q[0].double().cpu().numpy() - ref).max() / np.abs(ref).max()
    print('trace species', ratio, err, flush=True)
    assert err < 3e-5


@pytest.mark.parametrize('like', [False, True])
def test_chunks(cuda, monkeypatch, like):
    """One and two tasks per chunk (twice that where a call shares products;
    other group and x-range splits) change nothing but the order of sums."""
    from dgfs1d_gpu_amd import _lib
    todo = SAME * 2 if like else TASKS                # 10.5 MB of scratch per task
    q = 0 if like else 1

    def call(oracle):
        return _call(cuda, 32, 6, True, _lib.F64, 0, q, len(todo), todo, like=like, oracle=oracle)
    ref, err, info = call(True)
    assert err < 1e-11
    seen = {info['chunk']}
    for mb in ('1', '22'):
        monkeypatch.setenv('DGFS_BI_SCRATCH_MB', mb)
        got, _, info = call(False)
        seen.add(info['chunk'])
        assert np.abs(got - ref).max() < 1e-13 * np.abs(ref).max()
    assert seen == {1, 2, len(todo)}, seen
