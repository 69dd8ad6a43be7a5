"""Weight and bias gradients of the closure network at the sizes where their
partial sums are split differently: fewer tile tasks than work-groups (one
16^3 grid: 32 partials, each thread of the reduction sums one or none),
several tasks per work-group, and the 48^3 tile, all of one plane per task,
against the oracle; and batches whose tasks march through two, four and eight
planes against their grids one by one.

Both sides round to bf16 at the same points; a flip of one rounding (2^-8 of a
value) in a fraction of the activations gives the 2e-2 relative bound used for
every gradient tensor against the oracle."""
import numpy as np
import pytest

from test_gpu_closure import _rel, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('G,B', [(16, 1), (16, 20), (32, 1), (48, 1)])
def test_gradients(cuda, G, B):
    import torch
    net, onet, eng, u, src, sc, fs = _setup(cuda, G, B, seed=4)
    rng = np.random.default_rng(5)
    dout = rng.standard_normal((B, G, G, G)).astype(np.float32)
    eng.forward(u, src, sc, mode=0)
    d = torch.tensor(dout.reshape(-1), device=cuda)
    got = {k: v.cpu().numpy().copy() for k, v in eng.backward(u, src, sc, d).items()}
    again = eng.backward(u, src, sc, d)
    for k, v in again.items():
        assert np.array_equal(v.cpu().numpy(), got[k]), k
    _, cache = onet.forward(fs, bf=True)
    ref = onet.backward(dout.astype(np.float64), cache, bf=True)
    for k in got:
        r = np.asarray(ref[k]).reshape(got[k].shape)
        assert _rel(got[k], r) < 2e-2, (k, _rel(got[k], r))


# grids per batch whose 32 -> 32 weight-gradient tasks hold two, four and eight
# planes: as many as leave 512 work-groups a task each, from eight down
@pytest.mark.parametrize('G,B,planes', [(16, 32, 2), (16, 64, 4), (16, 128, 8), (32, 4, 2),
                                        (32, 5, 2), (32, 8, 4), (32, 16, 8), (32, 17, 8),
                                        (48, 2, 2), (48, 4, 4), (48, 8, 8)])
def test_batches_add_up(cuda, G, B, planes):
    """The gradients of a batch are the sums of its grids': the same products and
    roundings to bf16, FP32 sums in another order.  Terms of random sign add up to
    sqrt(n) of one, and m additions round by 2^-24 sqrt(m / 2) of that: 2e-6 for
    the 2000 additions of a chain of matrix instructions and partials; 1e-5.  A
    tensor's norm is that sqrt(n) but for the one value of b4, the sum of dOut
    (unit variance), which may be anywhere about 0."""
    import torch
    from dgfs1d_gpu_amd.learned import ClosureEngine
    rows = {16: 8, 32: 4, 48: 4}[G]
    tasks = lambda p: B * (G // rows) * (G // p)
    if torch.cuda.get_device_properties(cuda).multi_processor_count >= 256:
        assert tasks(planes) >= 512 and (planes == 8 or tasks(2 * planes) < 512)
    net, onet, eng, u, src, sc, fs = _setup(cuda, G, B, seed=4)
    d = torch.randn(B * G ** 3, device=cuda, generator=torch.Generator(cuda).manual_seed(5))
    eng.forward(u, src, sc, mode=0)
    got = {k: v.double().clone() for k, v in eng.backward(u, src, sc, d).items()}
    one = ClosureEngine(net, G, 1)
    n = G ** 3
    total = {k: torch.zeros_like(v) for k, v in got.items()}
    for b in range(B):
        ub = u[b * n:(b + 1) * n].contiguous()
        one.forward(ub, src[:1], sc[b:b + 1].contiguous(), mode=0)
        g = one.backward(ub, src[:1], sc[b:b + 1].contiguous(), d[b * n:(b + 1) * n].contiguous())
        for k, v in g.items():
            total[k] += v.double()
    for k, v in got.items():
        err = float((v - total[k]).norm()) / ((B * n) ** 0.5 if k == 'b4' else float(total[k].norm()))
        print(G, B, planes, k, '%.1e' % err, flush=True)
        assert err < 1e-5, k
