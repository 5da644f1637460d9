"""Runner workspaces (split-K partials, staged operands) are shared by no two
streams, threads or graphs: one runner used from several at once."""
import threading

import pytest
import torch

from pto_einsum import EinsumBuilder, StageGraph, builder, einsum

pytestmark = pytest.mark.gpu

# Two K splits of a vector kernel, a K split of the matrix-core kernels, a
# staged operand.
CASES = [("bht,bthd->bhd", (4, 16, 2048), (4, 2048, 16, 128)), ("ts,sp->tp", (256, 8192), (8192, 128)),
         ("ikj,jlk->il", (70, 12, 16), (16, 50, 12))]


def _operands(case, n):
    eq, s0, s1 = case
    g = torch.Generator().manual_seed(len(eq))
    return [(torch.randn(s0, generator=g).cuda(), torch.randn(s1, generator=g).cuda()) for _ in range(n)]


@pytest.mark.parametrize("case", CASES)
def test_two_streams(case):
    b = EinsumBuilder(case[0], [case[1], case[2]], torch.float32)
    run, ops = b.build(), _operands(case, 2)
    want = [run(*o) for o in ops]
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream() for _ in ops], [[], []]
    for _ in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i].append(run(*ops[i]))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(x, want[i]) for x in got[i])
    at = {k[1]: w.data_ptr() for k, w in b._workspaces.items()}
    assert {s.cuda_stream for s in streams} <= set(at)
    assert len(set(at.values())) == len(at) == 3      # and the first calls' stream
    b.cleanup()


def test_kept_workspaces_are_bounded():
    case = CASES[1]
    b = EinsumBuilder(case[0], [case[1], case[2]], torch.float32)
    run, (o,) = b.build(), _operands(case, 1)
    want, got = run(*o), []
    torch.cuda.synchronize()
    for s in [torch.cuda.Stream() for _ in range(builder._KEPT_WORKSPACES + 4)] * 2:
        with torch.cuda.stream(s):
            got.append(run(*o))
    torch.cuda.synchronize()
    assert len(b._workspaces) == builder._KEPT_WORKSPACES
    assert all(torch.equal(x, want) for x in got)
    b.cleanup()


def test_two_threads_on_one_stream():
    case = CASES[1]
    ops = _operands(case, 2)
    want = [einsum(case[0], *o) for o in ops]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        for _ in range(100):
            if not torch.equal(einsum(case[0], *ops[i]), want[i]):
                bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_two_graphs_replayed_at_once():
    """Graphs of the same equation, replayed on two streams next to eager
    calls on a third."""
    def stage(ops):
        return lambda: [einsum(c[0], *o) for c, o in zip(CASES, ops)]

    sets = [[_operands(c, 2)[i] for c in CASES] for i in range(2)]
    want = [[t.clone() for t in stage(s)()] for s in sets]
    graphs = [StageGraph(stage(s)) for s in sets]
    streams = [torch.cuda.Stream() for _ in sets]
    for rep in range(4):
        for g in graphs:
            for t in g.outputs:
                t.fill_(float("nan"))
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                g.replay()
        eager = stage(sets[rep % 2])()
        torch.cuda.synchronize()
        for g, w in zip(graphs, want):
            assert all(torch.equal(x, y) for x, y in zip(g.outputs, w))
        assert all(torch.equal(x, y) for x, y in zip(eager, want[rep % 2]))
