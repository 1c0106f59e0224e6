"""GPU: calls of several contexts and networks in turn, and of one context on
its two streams, with nothing waiting in between.

torch hands a tensor that was dropped to the next call at once, so outputs of
different contexts share memory; every result equals that of a call of its
own, bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def systems():
    from gimic_amd import synth
    made = [synth.sheet30(), synth.ring12()]
    ctxs = [s.context(screening=1e-8) for s in made]
    yield ctxs
    for ctx in ctxs:
        ctx.close()


def _points(n, seed):
    import torch
    return torch.tensor(np.random.default_rng(seed).uniform(-6.0, 6.0, (n, 3)),
                        dtype=torch.float64, device="cuda")


def test_contexts_share_one_stream_for_callers_on_the_null_stream(systems):
    import torch
    dev = torch.device("cuda")
    own = [ctx._stream(dev, None).value for ctx in systems]
    assert own[0] and own[0] == own[1]
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert systems[0]._stream(dev, None).value == side.cuda_stream
    assert systems[0]._stream(dev, side.cuda_stream).value == side.cuda_stream
    assert systems[0]._stream(dev, 0).value == own[0]


@pytest.mark.parametrize("n", [100, 20000])
def test_contexts_that_share_an_output_buffer(systems, n):
    import torch
    a, b = systems
    pa, pb = _points(n, 1), _points(n, 2)
    ref = torch.tensor(a.jtensor(pa.cpu().numpy()), device="cuda")
    other = torch.tensor(b.jtensor(pb.cpu().numpy()), device="cuda")
    torch.cuda.synchronize()
    for rep in range(8):
        print("case shared output", n, rep, flush=True)
        a.jtensor_device(pa)  # the longer call first, its output dropped
        got_b = b.jtensor_device(pb)
        got = a.jtensor_device(pa)
        b.jtensor_multi_device(pb, ["total", "total"])
        torch.cuda.synchronize()
        assert torch.equal(got, ref) and torch.equal(got_b, other)


def test_device_and_host_calls_of_one_context(systems):
    """the shared stream and the context's own take turns on one workspace"""
    import torch
    ctx = systems[0]
    pa, pb = _points(20000, 3), _points(17000, 4)
    ha, hb = pa.cpu().numpy(), pb.cpu().numpy()
    ref_a, ref_b = ctx.jtensor(ha), ctx.jtensor(hb)
    planes = [dict(points=hb[:3000], weights=np.ones(3000), normal=[0.0, 0.0, 1.0],
                   bfield=[0.0, 0.0, 1.0], center=[0.0, 0.0, 0.0])]
    flux = ctx.flux_planes(planes)
    for rep in range(4):
        print("case device and host calls", rep, flush=True)
        got = ctx.jtensor_device(pa)
        assert np.array_equal(ctx.jtensor(hb), ref_b)
        more = ctx.jtensor_device(pb)
        assert np.array_equal(ctx.flux_planes(planes), flux)
        last = ctx.jtensor_device(pa)
        torch.cuda.synchronize()
        assert np.array_equal(got.cpu().numpy(), ref_a)
        assert np.array_equal(more.cpu().numpy(), ref_b)
        assert np.array_equal(last.cpu().numpy(), ref_a)


def test_context_and_network_that_share_an_output_buffer(systems):
    import torch
    from gimic_amd.surrogate import Network
    ctx = systems[0]
    net = Network(1.5, np.array([0.0, 0.0, 0.0, 6.0]), np.linspace(0.5, 2.0, 9), seed=1)
    p, q = _points(20000, 5), _points(20000, 6)
    ref = ctx.jtensor(q.cpu().numpy())
    want = net.predict(p, unfused=True)
    torch.cuda.synchronize()
    for rep in range(4):
        print("case context and network", rep, flush=True)
        ctx.jtensor_device(q)
        got = net.predict(p)
        J = ctx.jtensor_device(q)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and np.array_equal(J.cpu().numpy(), ref)
    net.close()
