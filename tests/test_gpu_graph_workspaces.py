"""Who owns a split-K workspace: a compiled graph its own, an eager weight-only Linear its stream's,
a capture that owns none no workspace at all."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

import borch_amd  # noqa: E402
from borch_amd import int8 as I  # noqa: E402
from borch_amd.nn import intrinsic  # noqa: E402

D = 2048


@pytest.fixture
def dev():
    return torch.device("cuda", torch.cuda.current_device())


class _Spy:
    """The library with the workspace pointers of its weight-only and GEMM calls noted."""

    def __init__(self, lib):
        self._lib, self.seen = lib, []

    def __getattr__(self, name):
        f = getattr(self._lib, name)
        at = {"bq_linear_w8a32_ws": 10, "bq_linear_i8": 12, "bq_gemm_i8": 12}.get(name)
        if at is None:
            return f

        def call(*a):
            self.seen.append(a[at])
            return f(*a)
        return call


@pytest.fixture
def spy(monkeypatch):
    s = _Spy(I.lib())
    monkeypatch.setattr(I, "lib", lambda: s)
    return s


def _chain(seed, weight_only):
    torch.manual_seed(seed)
    m = torch.nn.Sequential(*[intrinsic.LinearReLU(borch_amd.nn.Linear(D, D)) for _ in range(4)]).cuda()
    borch_amd.nn.quantize_for_int8(m, weight_only=weight_only)
    return m


@pytest.mark.parametrize("weight_only", [True, False])
def test_compiled_graphs_own_theirs(weight_only, spy, monkeypatch):
    """Two graphs captured on one stream record different workspaces, neither of them the stream's,
    and run at once on two streams beside eager calls on the captured one, as one after the other."""
    one = torch.cuda.Stream()
    c, x = [], [torch.randn(16, D, device="cuda") for _ in range(2)]
    new = torch.cuda.Stream
    with monkeypatch.context() as m:  # as when torch's pool hands the same stream out again
        m.setattr(torch.cuda, "Stream", lambda *a, **k: new(*a, **k) if a or "stream_id" in k else one)
        for i in range(2):
            spy.seen.clear()
            c.append(borch_amd.compiled(_chain(i, weight_only), graph=True, tune=False))
            c[i](x[i])
            ptrs = set(spy.seen)
            c[i].ptrs = ptrs
            assert len(ptrs) == 1 and None not in ptrs
    with torch.cuda.stream(one):
        spy.seen.clear()
        eager = c[0].model(x[0])
        ptrs = [c[0].ptrs, c[1].ptrs, set(spy.seen)]
    assert len(set.union(*ptrs)) == 3
    torch.cuda.synchronize()
    want = [c[i](x[i]).clone() for i in range(2)]
    torch.cuda.synchronize()
    assert torch.equal(want[0], eager)
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = []
    for _ in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got.append((i, c[i](x[i]).clone()))
        with torch.cuda.stream(one), torch.no_grad():
            got.append((0, c[0].model(x[0])))
    torch.cuda.synchronize()
    assert all(torch.equal(y, want[i]) for i, y in got)


def test_a_capture_of_its_own_records_no_shared_workspace(spy):
    """torch.cuda.graph around weight-only Linears, after a warm-up on the captured stream."""
    m, x = _chain(3, True), torch.randn(16, D, device="cuda")
    s = torch.cuda.Stream()
    with torch.no_grad():
        with torch.cuda.stream(s):
            want = m(x)
        assert None not in spy.seen
        s.synchronize()
        spy.seen.clear()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            y = m(x)
    assert set(spy.seen) == {None}
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)


def test_eager_weight_only_calls_share_with_no_graph(spy, dev):
    """The weight-only Linear's eager workspace is not the one a W8A8 capture records."""
    with torch.no_grad():
        _chain(4, True)(torch.randn(16, D, device="cuda"))
    assert I.split_workspace(dev).data_ptr() not in spy.seen and None not in spy.seen


def test_the_owner_is_this_threads():
    """graph_workspaces holds for its own thread and block only."""
    import threading
    table, other = {}, []
    with I.graph_workspaces(table):
        t = threading.Thread(target=lambda: other.append(I._OWNED.table))
        t.start()
        t.join()
        with I.graph_workspaces({}):
            assert I._OWNED.table is not table
        assert I._OWNED.table is table
    assert other == [None] and I._OWNED.table is None
