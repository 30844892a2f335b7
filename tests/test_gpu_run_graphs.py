"""NVE and NVT device runs whose step counts give graphs of one to four steps,
and of two counts, and terms reduced for the last step only: the same state and
the same terms as one-step calls without graphs.  FP64, whose sums all have a
fixed order, so the two differ by nothing."""
import numpy as np
import pytest

from mspms2_amd import configs
from mspms2_amd.engine import LONG_TERMS_BYTES, SHORT_TERMS_BYTES, Engine
from tests.util import system_of

pytestmark = pytest.mark.gpu

NSTEPS = (1, 2, 3, 5, 6, 8, 9, 66)


@pytest.mark.parametrize("kind", ["nve", "nvt"])
def test_runs_equal_single_steps(kind):
    import torch
    s = system_of(configs.water_box(n_side=3, L=9.4, rc=4.5, kappa=0.6, kmax=4, ksqmax=16, seed=8))
    v0 = np.random.default_rng(2).standard_normal((3, s.natom)) * np.sqrt(s.treq / s.masses())
    dev = torch.device("cuda:0")
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev).contiguous()  # noqa: E731
    eng = Engine.replicas([s], precision="fp64")
    eng.set_list_skin(0.0)  # no list, and so no order of sums, from an earlier run
    x0, fl0, fs0 = eng.packed_positions(), eng.frclong()[0], eng.frcshort()[0]

    def run(parts, graph):
        if kind == "nvt":
            eng.nvt_set(4.0 * s.natom, 2.0 * s.natom, s.treq, 3 * s.natom - 3)
        bufs = [t(x0), t(v0), t(fl0), t(fs0)]
        lt = torch.zeros(LONG_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
        st = torch.zeros(SHORT_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
        uk = torch.zeros(1, dtype=torch.float64, device=dev)
        torch.cuda.synchronize()
        call = eng.nvt_run_device if kind == "nvt" else eng.vver_run_device
        for n in parts:
            call(*bufs, 0.25 * s.delt, 2, n, lt, st, uk, graph=graph)
        eng.sync()
        return [b.cpu() for b in (*bufs, lt, st, uk)]

    for n in NSTEPS:
        print(f"{kind} {n} steps", flush=True)
        want = run([1] * n, False)
        for graph in (True, False):
            for g, w in zip(run([n], graph), want):
                assert torch.equal(g.view(torch.int64), w.view(torch.int64))
    eng.close()


def _waits(stream, calls):
    """Whether calls() waits for work that lies ahead of it on the stream (some
    400 ms of matrix products)."""
    import torch
    with torch.cuda.stream(stream):
        big = torch.zeros(8192, 8192, device="cuda:0")
        out = torch.mm(big, big)
        torch.cuda.synchronize()
        for _ in range(60):
            torch.mm(big, big, out=out)
        done = torch.cuda.Event()
        done.record()
    calls()
    waited = done.query()
    torch.cuda.synchronize()
    return waited


@pytest.mark.parametrize("kind", ["nve", "nvt"])
def test_changing_lengths_capture_once(kind):
    """Runs of changing lengths on the same buffers: once every length has been
    seen, a call waits for nothing (a capture waits for the stream it is to be
    replayed on), and the states are those of one-step calls."""
    import torch
    s = system_of(configs.water_box(n_side=3, L=9.4, rc=4.5, kappa=0.6, kmax=4, ksqmax=16, seed=8))
    v0 = np.random.default_rng(2).standard_normal((3, s.natom)) * np.sqrt(s.treq / s.masses())
    dev = torch.device("cuda:0")
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev).contiguous()  # noqa: E731
    eng = Engine.replicas([s], precision="fp64")
    eng.set_list_skin(0.0)
    start = [t(a) for a in (eng.packed_positions(), v0, eng.frclong()[0], eng.frcshort()[0])]
    bufs = [torch.empty_like(a) for a in start]
    lt = torch.zeros(LONG_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    st = torch.zeros(SHORT_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    uk = torch.zeros(1, dtype=torch.float64, device=dev)
    stream = torch.cuda.Stream()
    call = eng.nvt_run_device if kind == "nvt" else eng.vver_run_device
    lengths = (10, 9, 8, 3, 17)

    def reset():
        if kind == "nvt":
            eng.nvt_set(4.0 * s.natom, 2.0 * s.natom, s.treq, 3 * s.natom - 3)
        with torch.cuda.stream(stream):
            for b, a in zip(bufs, start):
                b.copy_(a)
        torch.cuda.synchronize()

    def run(parts, graph):
        for n in parts:
            call(*bufs, 0.25 * s.delt, 2, n, lt, st, uk, graph=graph, stream=stream.cuda_stream)

    print(f"case {kind} {lengths}", flush=True)
    reset()
    run([1] * sum(lengths), False)
    torch.cuda.synchronize()
    want = [b.cpu() for b in (*bufs, lt, st, uk)]
    reset()
    run(lengths, True)
    torch.cuda.synchronize()
    for g, w in zip((*bufs, lt, st, uk), want):
        assert torch.equal(g.cpu().view(torch.int64), w.view(torch.int64))
    assert not _waits(stream, lambda: run(lengths, True)), "a run waited for the work ahead of it"
    eng.close()


def test_new_thermostats_keep_the_graph():
    """mspms_nvt_set between the runs of one system: no new capture (the call
    does not wait for work on the runs' stream), and the run starts from the new
    state."""
    import torch
    s = system_of(configs.lj_fcc(ncell=4, jitter=0.04, seed=5))
    v0 = np.random.default_rng(2).standard_normal((3, s.natom)) * np.sqrt(s.treq / s.masses())
    dev = torch.device("cuda:0")
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev).contiguous()  # noqa: E731
    eng = Engine.replicas([s], precision="fp64")
    start = [t(eng.packed_positions()), t(v0), t(eng.frclong()[0]), torch.zeros_like(t(v0))]
    lt = torch.zeros(LONG_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    st = torch.zeros(SHORT_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    uk, stream = torch.zeros(1, dtype=torch.float64, device=dev), torch.cuda.Stream()
    bufs = [b.clone() for b in start]

    def one(q):
        eng.nvt_set(q, q, s.treq, 3 * s.natom - 3)
        eng.nvt_run_device(*bufs, s.delt, 1, 4, lt, st, uk, stream=stream.cuda_stream)

    def fresh(q):
        for b, a in zip(bufs, start):
            b.copy_(a)
        torch.cuda.synchronize()
        one(q)
        torch.cuda.synchronize()
        return eng.nvt_get()

    print("case nvt_set between runs", flush=True)
    first, other = fresh(100.0), fresh(7.0)
    assert first != other and fresh(100.0) == first
    assert not _waits(stream, lambda: one(50.0)), "nvt_set or the run after it waited"
    eng.close()


def _node_types(graph):
    """hipGraphNodeType of every node of a captured graph."""
    import ctypes
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip, g, n = ctypes.CDLL(path), ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t()
    assert hip.hipGraphGetNodes(g, None, ctypes.byref(n)) == 0
    nodes, kind, out = (ctypes.c_void_p * n.value)(), ctypes.c_int(), []
    assert hip.hipGraphGetNodes(g, nodes, ctypes.byref(n)) == 0
    for node in nodes:
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        out.append(kind.value)
    return out


@pytest.mark.parametrize("kind", ["nve", "nvt"])
def test_runs_in_a_callers_capture(kind):
    """A run without graphs of its own, captured by the caller: kernels only (a
    memset node can give wrong values from the second replay on), and every
    replay, with eager work between them, leaves what the eager run leaves."""
    import torch
    s = system_of(configs.water_box(n_side=3, L=9.4, rc=4.5, kappa=0.6, kmax=4, ksqmax=16, seed=8))
    v0 = np.random.default_rng(2).standard_normal((3, s.natom)) * np.sqrt(s.treq / s.masses())
    dev = torch.device("cuda:0")
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev).contiguous()  # noqa: E731
    eng = Engine.replicas([s], precision="fp64")
    eng.set_list_skin(0.0)
    start = [t(a) for a in (eng.packed_positions(), v0, eng.frclong()[0], eng.frcshort()[0])]
    bufs = [b.clone() for b in start]
    lt = torch.zeros(LONG_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    st = torch.zeros(SHORT_TERMS_BYTES // 8, dtype=torch.float64, device=dev)
    uk = torch.zeros(1, dtype=torch.float64, device=dev)

    def reset():
        if kind == "nvt":
            eng.nvt_set(4.0 * s.natom, 2.0 * s.natom, s.treq, 3 * s.natom - 3)
        for b, a in zip(bufs, start):
            b.copy_(a)
        for b in (lt, st, uk):
            b.zero_()
        torch.cuda.synchronize()

    def run():
        call = eng.nvt_run_device if kind == "nvt" else eng.vver_run_device
        call(*bufs, 0.25 * s.delt, 2, 3, lt, st, uk, graph=False,
             stream=torch.cuda.current_stream().cuda_stream)

    print(f"case capture {kind}", flush=True)
    reset()
    run()
    torch.cuda.synchronize()
    want = [b.cpu() for b in (*bufs, lt, st, uk)]
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        run()
    kinds = _node_types(g)
    assert set(kinds) <= {0, 5}, kinds     # kernels, and the empty nodes of joins
    g.instantiate()
    for _ in range(4):
        reset()
        g.replay()
        torch.cuda.synchronize()
        for b, w in zip((*bufs, lt, st, uk), want):
            assert torch.equal(b.cpu().view(torch.int64), w.view(torch.int64))
    eng.close()
