"""Whose memory a run's results are in: an executable's own for as long as it
lives, whatever its launches are run, recorded or timed by; a compiled call's
its caller's.  On the CPU, the library's launches played by a model of their
pointers (th_launch_repoint, th_launches_run and th_launches_lend)."""
import contextlib
import ctypes
from types import SimpleNamespace

import pytest
import torch

from tempest_hip import runtime
from tempest_hip.runtime import Compiled, Executable, Group, Program, Value
from tempest_hip.target import Direct

N = 4


class Library:
    """y = 2 x + 1 and s = sum(x) for launch 1, whose values are x, y and s."""

    def __init__(self):
        self.at = {}                # value number -> address
        self.stream = 0             # the library's
        self.log = []

    def floats(self, address, n):
        return torch.frombuffer((ctypes.c_float * n).from_address(address), dtype=torch.float32)

    def run(self):
        x = self.floats(self.at[0], N)
        self.floats(self.at[1], N).copy_(2 * x + 1)
        self.floats(self.at[2], 1).copy_(x.sum())

    def call(self, name, *a):
        self.log.append(name)
        if name == "th_get_stream":
            a[0]._obj.value = self.stream
        elif name == "th_download":
            ctypes.memmove(a[0], a[1], a[2])
        elif name == "th_launches_run":
            self.run()
        elif name == "th_launches_lend":
            _, n, holders, values, offsets, refs, lent, home = a
            assert n == 1 and all(holders[i] == 1 for i in range(refs))
            for base in (lent, home):
                for i in range(refs):
                    self.at[values[i]] = base + offsets[i]
                if base == lent:
                    self.run()
        else:
            raise AssertionError(name)


class Launch:
    handle = ctypes.c_void_p(1)

    def __init__(self, lib):
        self.lib = lib

    def __call__(self):
        self.lib.run()

    def repoint(self, value, ptr):
        self.lib.at[value] = ptr

    def workspace(self):
        return 0


class Target:
    device = 0

    def allocate(self, dtype, n):
        return torch.zeros(n, dtype=dtype)

    def pointable(self, x, at):
        return True

    def capture(self, steps, keep=None, graph=None):
        return Direct(steps)

    def replay(self, graph):
        for s in graph.steps:
            s()


@pytest.fixture
def compiled(monkeypatch):
    lib, current = Library(), SimpleNamespace(cuda_stream=0)
    monkeypatch.setattr(runtime, "call", lib.call)
    monkeypatch.setattr(runtime, "Arena", lambda sizes: SimpleNamespace(addresses=[], bytes=0))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: current)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: empty(*a, **{x: k[x] for x in k if x != "pin_memory"}))

    def build(addresses):
        lib.at = dict(enumerate(addresses[v] for v in ("x", "y", "s")))
        return Launch(lib)

    f32 = torch.float32
    program = Program("affine", {"x": Value("x", f32, (N,), "input"), "y": Value("y", f32, (N,), "result"),
                                 "s": Value("s", f32, (), "result")},
                      [Group("affine", ("x", "y", "s"), ("x",), ("y", "s"), build)], ["x"], ["y", "s"])
    comp = Compiled(program, Target(), [torch.arange(float(N))])
    return SimpleNamespace(comp=comp, lib=lib, current=current, x=lambda k: torch.arange(float(N)) + k)


def want(x):
    return 2 * x + 1


def test_launches_stay_at_the_executables_results(compiled):
    """Between calls every launch points at the allocation the executable was
    built with, which it keeps: what a recording made before a call, or after
    it, writes to."""
    ex = compiled.comp.executable
    home, at = ex._results, dict(compiled.lib.at)
    kept = [compiled.comp(compiled.x(k)) for k in range(3)]
    assert "th_launches_lend" in compiled.lib.log
    assert ex._results is home and (compiled.lib.at[1], compiled.lib.at[2]) == (at[1], at[2])
    for k, (y, s) in enumerate(kept):
        assert torch.equal(y, want(compiled.x(k))) and s == compiled.x(k).sum()
        assert not home.data_ptr() <= y.data_ptr() < home.data_ptr() + home.numel()


@pytest.mark.parametrize("run", ["launch", "recorded", "execute", "replay"])
def test_a_run_leaves_returned_arrays_alone(compiled, run):
    """A launch run by hand, what capture recorded, execute and replay write
    to the executable's results, never into what a call returned."""
    y, s = compiled.comp(compiled.x(1))
    ex = compiled.comp.executable
    x = compiled.x(5)
    ex.point(x)
    {"launch": lambda: ex.launches[0](), "recorded": lambda: ex.target.replay(ex.graph), "execute": ex.execute,
     "replay": ex.replay}[run]()
    assert torch.equal(y, want(compiled.x(1))) and s == compiled.x(1).sum()
    assert torch.equal(ex.outputs()[0], want(x)) and ex.outputs()[1] == x.sum()


def test_another_kind_of_recording_is_what_a_call_replays(compiled):
    """What a target records that is not the launches themselves runs as it
    replays it, into the executable's results."""
    comp, lib = compiled.comp, compiled.lib
    replayed = []
    comp.executable._graph = object()
    comp.executable.target.replay = lambda graph: replayed.append(graph) or lib.run()
    y, s = comp(compiled.x(3))
    assert len(replayed) == 1 and "th_launches_lend" not in lib.log
    assert torch.equal(y, want(compiled.x(3))) and s == compiled.x(3).sum()
    assert torch.equal(comp.executable._results.view(torch.float32)[:N], y) and y.data_ptr() != comp.executable._results.data_ptr()


def test_outputs_show_the_last_call_and_follow_later_ones(compiled):
    """outputs(ex) are the buffers themselves: the last call's results right
    after it, whatever its caller has done to what it was given, and those of
    every later run."""
    y, _ = compiled.comp(compiled.x(1))
    ex = compiled.comp.executable
    shown = ex.outputs()
    assert torch.equal(shown[0], want(compiled.x(1)))
    again, _ = compiled.comp(compiled.x(2))
    assert torch.equal(shown[0], want(compiled.x(2))) and torch.equal(again, want(compiled.x(2)))
    shown[0].zero_()
    assert torch.equal(again, want(compiled.x(2))) and torch.equal(y, want(compiled.x(1)))


@pytest.mark.parametrize("ask", ["outputs", "returned"])
def test_the_last_calls_results_after_the_caller_wrote_over_its_own(compiled, ask):
    x = compiled.x(1)
    y, _ = compiled.comp(x)
    y.mul_(100.0)
    got = compiled.comp.returned()[0] if ask == "returned" else compiled.comp.executable.outputs()[0]
    assert torch.equal(got, want(x)) and torch.equal(y, 100.0 * want(x))


def test_another_current_stream_allocates_nothing(compiled, monkeypatch):
    """Under another current stream than the library's a call runs into the
    executable's results and copies them; a run of the executable's own
    allocates nothing, before and after a call."""
    first, _ = compiled.comp(compiled.x(1))
    ex, home = compiled.comp.executable, compiled.comp.executable._results
    compiled.current.cuda_stream = 7
    made = []
    like = torch.empty_like
    monkeypatch.setattr(torch, "empty_like", lambda *a, **k: made.append(1) or like(*a, **k))
    x = compiled.x(2)
    ex.point(x).execute()
    ex.replay()
    assert not made and ex._results is home and torch.equal(ex.outputs()[0], want(x))
    third, s = compiled.comp(compiled.x(3))
    assert not made and torch.equal(third, want(compiled.x(3))) and s == compiled.x(3).sum()
    assert torch.equal(first, want(compiled.x(1)))
