"""Value scatters and captured graphs: a captured one depends on no context
scratch, and an eager one touches none that a captured graph addresses."""
import numpy as np
import pytest
import torch

from oracle import pm as opm

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def in_tiles(monkeypatch):
    """Contexts that scatter values in tiles at any particle count."""
    from pmwd_amd import _lib
    monkeypatch.setenv('PMX_VALUES_MIN', '0')
    monkeypatch.setattr(_lib, '_ctx_cache', {})


def _state(dev, shape, copies, seed):
    import pmwd_amd as pa
    conf = pa.Configuration(1.7, shape, mesh_shape=1)
    pmid, disp = opm.gen_grid(shape, conf.mesh_shape, conf.cell_size)
    rng = np.random.default_rng(seed)
    pmid, disp = np.tile(pmid, (copies, 1)), np.tile(disp, (copies, 1))
    disp = (disp + 2 * conf.cell_size * rng.standard_normal(disp.shape)).astype(np.float32)
    val = rng.standard_normal((len(pmid), 3)).astype(np.float32)
    t = lambda a: torch.as_tensor(a, device=dev)
    return conf, pa.Particles(conf, t(pmid), t(disp)), t(val)


def _captured(dev, ctx, work):
    from pmwd_amd import _lib
    side = torch.cuda.Stream(device=dev)
    graph = torch.cuda.CUDAGraph()
    with _lib.context_scope(lambda key, make: ctx):
        with torch.cuda.stream(side):
            work()   # the warm-up: the context holds its scratch
            side.synchronize()
            with torch.cuda.graph(graph, stream=side):
                out = work()
    return graph, out


@pytest.mark.parametrize('kind', ['scatter', 'readout_grad', 'mass'])
def test_graph_replays_after_other_calls_moved_the_scratch(dev, kind):
    import pmwd_amd as pa
    from pmwd_amd import _lib
    conf, few, val = _state(dev, (20, 12, 35), 1, 1)
    _, many, mval = _state(dev, (20, 12, 35), 6, 2)
    ctx = _lib.Context(conf.mesh_shape, conf.cell_size, dev)
    mesh = torch.randn(conf.mesh_shape + (3,), device=dev,
                       generator=torch.Generator(device=dev).manual_seed(3))

    def work():
        if kind == 'mass':
            return pa.scatter(few, conf)
        if kind == 'scatter':
            return pa.scatter(few, conf, val=val)
        m = mesh.clone().requires_grad_(True)
        with torch.enable_grad():
            out = pa.gather(few, conf, m, val=torch.zeros_like(val))
        return torch.autograd.grad(out, m, val)[0]

    want = work().clone()
    graph, got = _captured(dev, ctx, work)
    for rnd in range(3):
        with _lib.context_scope(lambda key, make: ctx):
            big = pa.scatter(many if rnd else few, conf, val=mval if rnd else val)
            if rnd == 2 and kind != 'mass':
                ctx.trim()
        # what the allocator gets back must not be what the graph writes
        watch = [torch.full((k,), 7.0, device=dev) for k in (60000, 250000, 800000)]
        got.fill_(float('nan'))
        graph.replay()
        torch.cuda.synchronize()
        if kind == 'mass':
            assert torch.equal(got, want)
        else:
            np.testing.assert_allclose(got.cpu().numpy(), want.cpu().numpy(), rtol=1e-5, atol=1e-5)
        assert all(bool((w == 7.0).all()) for w in watch)
        ref = pa.scatter(many if rnd else few, conf, val=mval if rnd else val)
        np.testing.assert_allclose(big.cpu().numpy(), ref.cpu().numpy(), rtol=1e-5, atol=1e-5)
    del graph
    ctx.close()


def test_trim_gives_the_value_scratch_back(dev):
    import pmwd_amd as pa
    from pmwd_amd import _lib
    conf, ptcl, val = _state(dev, (20, 12, 35), 1, 4)
    ctx = _lib.Context(conf.mesh_shape, conf.cell_size, dev)
    with _lib.context_scope(lambda key, make: ctx):
        held = ctx.nbytes
        a = pa.scatter(ptcl, conf, val=val)
        assert ctx.nbytes >= held + 20 * len(ptcl)
        grown = ctx.nbytes
        b = pa.scatter(ptcl, conf, val=val)
        assert ctx.nbytes == grown
        ctx.trim()
        assert ctx.nbytes == held
        c = pa.scatter(ptcl, conf, val=val)
    for x in (b, c):
        np.testing.assert_allclose(x.cpu().numpy(), a.cpu().numpy(), rtol=1e-5, atol=1e-5)
    ctx.close()


def test_threads_on_one_context(dev):
    """Threads that scatter values on one context and stream at once, beside
    one that takes densities there, each get their own numbers."""
    import threading
    import pmwd_amd as pa
    from pmwd_amd import _lib
    cases = [_state(dev, (20, 12, 35), k, 10 + k) for k in (1, 2, 3)]
    conf = cases[0][0]
    _lib.context(conf.mesh_shape, conf.cell_size, dev)   # the one that all share
    works = [lambda p=p, v=v: pa.scatter(p, conf, val=v) for _, p, v in cases]
    works.append(lambda: pa.scatter(cases[0][1], conf))
    want = [w().clone() for w in works]
    wrong = []

    def loop(work, ref):
        try:
            torch.cuda.set_device(dev)
            for _ in range(40):
                got = work()
                torch.cuda.synchronize()
                if not torch.allclose(got, ref, rtol=1e-5, atol=1e-5):
                    wrong.append(float((got - ref).abs().max()))
        except Exception as e:   # reported by the assertion below
            wrong.append(repr(e))

    threads = [threading.Thread(target=loop, args=a) for a in zip(works, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:5]
    assert len(_lib._ctx_cache) == 1
