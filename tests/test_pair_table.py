"""The pair form of mode-coupling task tables (collision.pair_table) on the
host: the gain and loss coefficients add up to the tasks' bilinear form over
every accepted table, and tables that gain nothing keep their tasks."""
import numpy as np
import pytest

from dgfs1d_gpu_amd.collision import pair_table


def _forms(p, nsl):
    """(symmetric gain form, loss form) per output from the tables."""
    import torch
    v = {k: (x.numpy() if isinstance(x, torch.Tensor) else x) for k, x in p.items()}
    first = v['slice'][:, 0, 0], v['slice'][:, 1, 0]
    assert (v['nterm'] == 1).all() and (v['coef'][:, :, 0] == 1.0).all()
    assert (first[0][:v['ndiag']] == first[1][:v['ndiag']]).all()
    assert (first[0][v['ndiag']:] != first[1][v['ndiag']:]).all()
    out = {}
    for o in range(v['nout']):
        G, L = np.zeros((nsl, nsl)), np.zeros((nsl, nsl))
        for j in range(v['gstart'][o], v['gstart'][o + 1]):
            a, b = first[0][v['gpair'][j]], first[1][v['gpair'][j]]
            G[a, b] += v['gcoef'][j] / 2
            G[b, a] += v['gcoef'][j] / 2
        last = []
        for j in range(v['lstart'][o], v['lstart'][o + 1]):
            t = v['lpair'][j]
            assert t < v['ndiag']
            if not last or last[-1] != t:
                assert t not in last           # one task's entries are consecutive
                last.append(t)
            L[v['lslice'][j], first[1][t]] += v['lcoef'][j]
        out[int(v['oslice'][o])] = G, L
    return out


def _check(K, Ne, tasks):
    import torch
    p = pair_table(K, Ne, tasks, torch.float64, 'cpu')
    assert p is not None
    nsl = K * Ne
    ref = {}
    for o, f, g in tasks:
        T = ref.setdefault(o, np.zeros((nsl, nsl)))
        for a, ca in f:
            for b, cb in g:
                T[a, b] += ca * cb
    got = _forms(p, nsl)
    assert set(got) == set(ref)
    for o, T in ref.items():
        tol = 1e-14 * np.abs(T).max()
        assert np.abs(got[o][1] - T).max() <= tol
        assert np.abs(got[o][0] - (T + T.T) / 2).max() <= tol
    return p


@pytest.mark.parametrize('K', [2, 3, 4, 5, 7])
@pytest.mark.parametrize('kind', ['modal-orthonormal-legendre', 'modal-modified-karniadakis'])
def test_modal_bases(K, kind):
    from dgfs1d_gpu_amd.basis import Basis
    from dgfs1d_gpu_amd.dictionary import Dictionary
    from dgfs1d_gpu_amd.nputil import subclass_where
    cfg = Dictionary('[basis]\nkind = %s\nK = %d\nNqr = 4\n' % (kind, K))
    tasks = subclass_where(Basis, basis_kind=kind)(cfg).collision_tasks(3)
    p = _check(K, 3, tasks)
    assert p['ndiag'] == 3 * K and p['npair'] <= len(tasks)


def test_unsymmetric_and_repeated_terms():
    """f and g of different slices, repeated slices in a task, outputs that
    share pairs, an output whose terms cancel."""
    tasks = [(0, [(0, 1.0), (1, -2.0)], [(1, 0.5), (0, 1.5)]), (0, [(1, 1.0)], [(0, 3.0)]),
             (2, [(0, 1.0), (0, 1.0)], [(1, 1.0)]), (2, [(1, 0.25)], [(0, 1.0)]),
             (1, [(0, 1.0)], [(0, 1.0)]), (3, [(1, 1.0)], [(1, 1.0)]),
             (3, [(1, -1.0)], [(1, 1.0)])]
    _check(2, 2, tasks)


def test_tables_without_gain_keep_their_tasks():
    import torch
    nodal = [(s, [(s, 1.0)], [(s, 1.0)]) for s in range(6)]
    assert pair_table(3, 2, nodal, torch.float64, 'cpu') is None
    cross = [(0, [(0, 1.0)], [(1, 1.0)]), (1, [(2, 1.0)], [(3, 1.0)])]
    assert pair_table(2, 2, cross, torch.float64, 'cpu') is None
    assert pair_table(2, 2, [], torch.float64, 'cpu') is None


@pytest.mark.parametrize('bad,dtype', [(float('inf'), 'float64'), (float('nan'), 'float64'),
                                       (1e200, 'float64'), (1e30, 'float32'), (1e-30, 'float32'),
                                       (1e-170, 'float64')])
def test_coefficients_out_of_range_keep_their_tasks(bad, dtype):
    """Products of coefficients that are not finite or no normal numbers of the
    type: the tasks give what they always gave for them, no output is dropped."""
    import torch
    td = getattr(torch, dtype)
    good = [(o, [(0, 1.0), (1, 0.5)], [(0, c), (1, 2.0)]) for o in range(4) for c in (1.0, 3.0)]
    assert pair_table(4, 1, good, td, 'cpu') is not None
    for at in range(2):
        worse = list(good)
        worse[5] = (2, [(at, bad)], [(0, bad)])
        assert pair_table(4, 1, worse, td, 'cpu') is None


def test_small_coefficients_stay():
    """A coefficient far below its output's largest belongs to a slice that may be
    as much larger: only products that cancel are left out."""
    tasks = [(o, [(0, 1.0), (1, 1e-9)], [(0, c), (1, 2e-9)]) for o in range(4) for c in (1.0, 3.0)]
    got = _forms(_check(4, 1, tasks), 4)
    for o in range(4):
        assert abs(got[o][1][1, 1] - 4e-18) <= 1e-32
    zero = [(o, [(0, 1.0), (1, c)], [(0, 0.3), (1, 0.7 * c)]) for o in range(4) for c in (1.0, -1.0)]
    p = _check(4, 1, zero)                     # (0, 1) and (1, 0) cancel
    assert p['npair'] == p['ndiag'] == 2


def test_symmetric_flag():
    """task_table marks exactly the tables whose outputs are symmetric in f and g."""
    import torch
    from dgfs1d_gpu_amd.basis import Basis
    from dgfs1d_gpu_amd.collision import task_table
    from dgfs1d_gpu_amd.dictionary import Dictionary
    from dgfs1d_gpu_amd.nputil import subclass_where
    flag = lambda K, Ne, t: task_table(K, Ne, t, torch.float64, 'cpu')['symmetric']
    kind = 'modal-orthonormal-legendre'
    for K in (2, 3, 5):
        cfg = Dictionary('[basis]\nkind = %s\nK = %d\nNqr = 4\n' % (kind, K))
        assert flag(K, 2, subclass_where(Basis, basis_kind=kind)(cfg).collision_tasks(2))
    assert flag(2, 1, [(0, [(1, 0.5)], [(1, 2.0)])])
    assert not flag(2, 1, [(0, [(0, 1.0)], [(1, 1.0)])])
    both = [(0, [(0, 1.0)], [(1, 1.0)]), (0, [(1, 1.0)], [(0, 1.0)])]
    assert flag(2, 1, both)
    assert not flag(2, 1, [both[0], (1,) + both[1][1:]])
    assert not flag(2, 1, [(0, [(0, float('nan'))], [(1, 1.0)])])
