"""The mixture operator's streaming kernels (packed real transforms, Hermitian
half of the products, paired directions) against the FP64 oracle and against
each other, at the forms they accept: N = 20, 24, 32, 48 with one and two lanes
per plane row, rules with and without opposite directions, the like-species
call, task chunks and several group and x-range splits.

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


def _call(cuda, N, M, antipodal, dtype, p, q, ntask_max, tasks=TASKS, like=False, Nrho=3,
          oracle=True):
    """Q of one call, its error against the oracle, and the plan's query."""
    import torch
    from dgfs1d_gpu_amd import _lib
    from dgfs1d_gpu_amd.collision import BiCollisionPlan
    vm = _mesh(N, 6, Nrho)
    sz, szpre = _rule(M, antipodal), load_design('womersley', 32)
    m = vm.masses
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
                                     (32, 'F64'), (32, 'F32'), (48, 'F32')])
@pytest.mark.parametrize('M,antipodal', [(6, True), (5, False), (1, False)])
def test_rules(cuda, N, dtype, M, antipodal):
    from dgfs1d_gpu_amd import _lib
    # a task capacity whose product cubes exceed the streaming line at N = 20, 24
    got, err, info = _call(cuda, N, M, antipodal, getattr(_lib, dtype), 0, 1, 400 // M)
    print(N, dtype, M, antipodal, err, info, flush=True)
    assert info['streaming'] and not info['like_chunk']       # unequal masses
    assert err < (1e-11 if dtype == 'F64' else 3e-5)


# singular triplets of symmetric 2 x 2 couplings (degenerate and not), and a
# single-slice task with unequal coefficients
TRIPLETS = [(0, [(0, 1.0)], [(1, 0.7)]), (0, [(1, 1.0)], [(0, 0.7)]),
            (1, [(0, 0.8), (1, 0.6)], [(0, 0.8), (1, 0.6)]),
            (1, [(0, -0.6), (1, 0.8)], [(0, 0.3), (1, -0.4)]), (3, [(2, 0.5)], [(2, 3.0)])]
SAME = [(0, [(0, 1.0)], [(0, 1.0)]), (1, [(1, 0.5), (3, 0.25)], [(1, 0.5), (3, 0.25)]),
        (1, [(2, -1.0)], [(2, -1.0)])]


@pytest.mark.parametrize('N,dtype', [(20, 'F64'), (24, 'F32'), (32, 'F64'), (48, 'F32')])
@pytest.mark.parametrize('M,antipodal', [(6, True), (5, False)])
@pytest.mark.parametrize('tasks', ['same', 'triplets'])
def test_like_species(cuda, N, dtype, M, antipodal, tasks):
    """up is uq and the tasks of each output symmetric in f and g: one product
    per opposite pair; the same table with another array takes the general
    form."""
    from dgfs1d_gpu_amd import _lib
    d = getattr(_lib, dtype)
    todo = SAME if tasks == 'same' else TRIPLETS
    a, err, info = _call(cuda, N, M, antipodal, d, 1, 1, 400 // M, todo, like=True)
    assert info['streaming'] and (info['like_chunk'] > 0) == antipodal
    b, _, _ = _call(cuda, N, M, antipodal, d, 1, 1, 400 // M, todo, oracle=False)
    diff = np.abs(a - b).max() / np.abs(b).max()
    print(N, dtype, M, err, diff, flush=True)
    assert err < (1e-11 if dtype == 'F64' else 3e-5)
    assert diff < (1e-13 if dtype == 'F64' else 3e-5)


def test_one_species_with_unsymmetric_tasks(cuda):
    """up is uq, but f and g do not exchange: the general form."""
    from dgfs1d_gpu_amd import _lib
    a, err, info = _call(cuda, 20, 6, True, _lib.F64, 0, 0, 70, TASKS, like=True)
    assert info['streaming'] and info['like_chunk']
    assert err < 1e-11


def test_like_call_of_unequal_masses(cuda):
    """The like form needs equal masses: with others the call is the general one."""
    import torch
    from dgfs1d_gpu_amd import _lib
    from dgfs1d_gpu_amd.collision import BiCollisionPlan
    N, M = 20, 6
    vm = _mesh(N, M, 3)
    sz, szpre, u = load_design('womersley', M), load_design('womersley', 32), _fields(vm, 2, 2, 11)[0]
    d = torch.tensor(u, device=cuda)
    for mp, mq in ((vm.masses[0], vm.masses[1]), (vm.masses[1], vm.masses[1])):
        plan = BiCollisionPlan(N, M, 3, vm.L, vm.qz, vm.qw, sz, vm.sw, szpre, mp, mq, 1.36, 0.8,
                               0.41, _lib.F64, 70, device=cuda)
        info = plan.query()
        assert info['streaming'] and (info['like_chunk'] > 0) == (mp == mq)
        plan.set_tasks(2, 2, SAME)
        Q = torch.zeros_like(d)
        plan(d, d, Q)
        plan.close()
        pre = OB.BiPrecomp(N, vm.L, vm.qz, vm.qw, sz, vm.sw, szpre, mp, mq, 1.36, 0.8)
        ref = np.zeros_like(u)
        for out, ft, gt in SAME:
            ref[out] += OB.q_pq(pre, sum(c * u[s] for s, c in ft), sum(c * u[s] for s, c in gt),
                                0.41)
        assert np.abs(Q.cpu().numpy() - ref).max() < 1e-11 * np.abs(ref).max()


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
    assert not ia['streaming'] and ib['streaming'] == (N > 16)
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


# (streaming) plans of one pair, with the task capacity that takes them over the
# line between the forms at N = 20, 24
ABSENT = [(20, 'F64'), (20, 'F32'), (24, 'F64'), (24, 'F32'), (32, 'F64'), (32, 'F32'),
          (48, 'F32')]


def _plan(cuda, N, dtype, p, q, Nrho=3, M=6):
    from dgfs1d_gpu_amd import _lib
    from dgfs1d_gpu_amd.collision import BiCollisionPlan
    vm = _mesh(N, M, Nrho)
    m = vm.masses
    sz, szpre = load_design('womersley', M), load_design('womersley', 32)
    plan = BiCollisionPlan(N, M, Nrho, vm.L, vm.qz, vm.qw, sz, vm.sw, szpre, m[p], m[q], 1.36,
                           0.8, 0.41, getattr(_lib, dtype), 80, device=cuda)
    pre = OB.BiPrecomp(N, vm.L, vm.qz, vm.qw, sz, vm.sw, szpre, m[p], m[q], 1.36, 0.8)
    return vm, plan, pre


@pytest.mark.parametrize('N,dtype', ABSENT)
def test_absent_species(cuda, N, dtype):
    """Where a species is absent the pair's term is exactly zero, beside nodes
    that hold both; where the present side is not finite the term is not
    either.  The like-species form too."""
    import torch
    td = torch.float64 if dtype == 'F64' else torch.float32
    tasks = [(s, [(s, 1.0)], [(s, 1.0)]) for s in range(4)]
    for p, q in ((0, 1), (1, 1)):
        vm, plan, _ = _plan(cuda, N, dtype, p, q)
        u = _fields(vm, 2, 2, 11)
        plan.set_tasks(2, 2, tasks)
        full = [torch.tensor(u[s], dtype=td, device=cuda) for s in (p, q)]
        if p == q:
            full[1] = full[0]

        def call(f, g):
            Q = torch.full((4, N ** 3), 0.25, dtype=td, device=cuda)
            plan(f, g, Q)
            return Q

        base = call(*full)
        f, g = full[0].clone(), full[1].clone()
        f[1], g[2] = 0.0, 0.0
        if p == q:
            g[1] = f[2] = 0.0
        f[3], g[3] = 0.0, 0.0
        got = call(f, f if p == q else g)
        assert torch.equal(got[0], base[0]) and not torch.equal(base[0], torch.full_like(base[0], 0.25))
        for s in (1, 2, 3):
            assert torch.equal(got[s], torch.full_like(got[s], 0.25)), (p, q, s)
        if p != q:
            g[1] = float('nan')
            f[2] = float('inf')
            bad = call(f, g)
            assert torch.equal(bad[0], base[0])
            assert bool(bad[1].isnan().all()) and bool(bad[2].isnan().all())
        plan.close()


@pytest.mark.parametrize('N,dtype,a,b', [
    (32, 'F32', 1e-18, 1.0), (24, 'F32', 1e18, 1.0), (20, 'F32', 1e-30, 1e25),
    (32, 'F32', 1e20, 1e-25), (20, 'F64', 1e-200, 1e150), (24, 'F64', 1e160, 1e-170),
    (32, 'F64', 1e-40, 1.0)])
def test_density_range(cuda, N, dtype, a, b):
    """Densities from end to end of the type's range: the sides of a shared
    transform keep the precision that each has alone.  The oracle is bilinear in
    the densities, so it is taken at 1 and scaled."""
    import torch
    td = torch.float64 if dtype == 'F64' else torch.float32
    vm, plan, pre = _plan(cuda, N, dtype, 0, 1)
    u = _fields(vm, 2, 2, 11)
    plan.set_tasks(2, 2, [(0, [(0, 1.0)], [(1, 1.0)])])
    up = torch.tensor(u[0] * a, dtype=td, device=cuda)
    uq = torch.tensor(u[1] * b, dtype=td, device=cuda)
    Q = torch.zeros_like(up)
    plan(up, uq, Q)
    ref = OB.q_pq(pre, u[0][0], u[1][1], 0.41)
    err = np.abs(Q[0].double().cpu().numpy() / (a * b) - ref).max() / np.abs(ref).max()
    plan.close()
    print('densities', N, dtype, a, b, err, flush=True)
    assert err < (1e-11 if dtype == 'F64' else 3e-5)


@pytest.mark.parametrize('N,dtype', ABSENT + [(16, 'F64')])
def test_empty_groups(cuda, N, dtype):
    """Groups without tasks, first and last, beside others in a work-group:
    their outputs stay, the others are those of the table without them."""
    import torch
    td = torch.float64 if dtype == 'F64' else torch.float32
    vm, plan, _ = _plan(cuda, N, dtype, 0, 1)
    u = _fields(vm, 2, 2, 11)
    up, uq = (torch.tensor(x, dtype=td, device=cuda) for x in u)
    t = plan.set_tasks(2, 2, [(1, [(0, 1.0)], [(1, 1.0)]), (1, [(2, 0.5)], [(3, 1.0)]),
                              (2, [(1, 1.0)], [(0, 2.0)]), (2, [(3, 1.0)], [(3, 1.0)]),
                              (2, [(2, 1.0)], [(2, 1.0)])])
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=cuda)
    assert t['gstart'].tolist() == [0, 2, 5] and t['gslice'].tolist() == [1, 2]
    gaps = dict(t, ngroup=4, gstart=ints([0, 0, 2, 5, 5]), gslice=ints([0, 1, 2, 3]))
    got = []
    for table in (t, gaps):
        Q = torch.full((4, N ** 3), 0.25, dtype=td, device=cuda)
        plan(up, uq, Q, tasks=table)
        got.append(Q)
    assert torch.equal(got[0], got[1])
    for s in (0, 3):
        assert torch.equal(got[1][s], torch.full_like(got[1][s], 0.25))
    plan.close()


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
    assert info['streaming'] and (info['like_chunk'] > 0) == like
    assert err < 1e-11
    seen = {info['chunk']}
    for mb in ('1', '22'):
        monkeypatch.setenv('DGFS_BI_SCRATCH_MB', mb)
        got, _, info = call(False)
        seen.add(info['chunk'])
        assert info['like_chunk'] == (min(2 * info['chunk'], len(todo)) if like else 0)
        assert np.abs(got - ref).max() < 1e-13 * np.abs(ref).max()
    assert seen == {1, 2, len(todo)}, seen
