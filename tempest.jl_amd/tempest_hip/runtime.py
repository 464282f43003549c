"""The executable: slots, binding and pointing, execute!/capture!/replay!.

Mirrors src/Compiler/runtime/runtime.jl and runtime/compile.jl for programs
whose plan is given (the front end that traces and plans them is Julia's and
stays there; ``programs.py`` states each plan it would form):

- ``storage``     the slot pool of plan/storage.jl:236-319 for one stream:
                  values take, in kernel order, the smallest free slot that
                  fits, else the largest free slot grown, else a new one.
- ``prepare``     runtime.jl:194-200, 337-539: slots in one arena
                  (th_arena_create), own buffers for results, one launch per
                  group built on the values' addresses.
- ``bind`` / ``point``  runtime.jl:719-830: copy inputs into own buffers, or
                  take the caller's arrays as storage by reference and
                  repoint the launches that read them where they moved.
- ``execute``, ``capture``, ``replay``  runtime.jl:1158-1214.
- ``compile`` / ``Compiled``  compile.jl:48-62, 310-349: signature check,
                  point, replay, and results returned as copies (numbers
                  read to the host).
"""
from __future__ import annotations

import ctypes
import math
from dataclasses import dataclass, field
from typing import Callable, Sequence

import torch

from ._lib import call
from .launch import Launch
from .target import Direct, Graph, HIPTarget, Move

_ELEMENT = {torch.float32: 4, torch.bfloat16: 2, torch.float16: 2, torch.float64: 8, torch.int32: 4,
            torch.int64: 8, torch.uint8: 1}


@dataclass
class Value:
    """A value of a plan: its element type, its Julia dimensions (column-major,
    first fastest) and its role: an ``input``, a ``result`` (own buffer,
    returned) or ``stored`` (kept between kernels, in a slot)."""

    name: str
    dtype: torch.dtype
    dims: tuple
    role: str

    @property
    def count(self) -> int:
        n = 1
        for d in self.dims:
            n *= int(d)
        return n

    @property
    def nbytes(self) -> int:
        return self.count * _ELEMENT[self.dtype]

    @property
    def scalar(self) -> bool:
        return self.dims == ()


@dataclass
class Group:
    """A kernel of the plan: the claim that runs it builds one launch from the
    addresses of the values it names, in its launch's value order."""

    name: str
    values: tuple[str, ...]
    reads: tuple[str, ...]
    writes: tuple[str, ...]
    build: Callable[[dict[str, int]], Launch]


@dataclass
class Program:
    name: str
    values: dict[str, Value]
    groups: list[Group]
    inputs: list[str]
    outputs: list[str]


@dataclass
class Storage:
    """plan/storage.jl:37-46: lifetimes (first and last kernel), slots, sizes."""

    lifetimes: dict[str, tuple[int, int]]
    slots: dict[str, int]
    sizes: list[int]


def storage(program: Program) -> Storage:
    """Slots for the stored values, one stream (plan/storage.jl:64-80, 236-319)."""
    first: dict[str, int] = {}
    last: dict[str, int] = {}
    for k, g in enumerate(program.groups):
        for v in g.writes:
            first.setdefault(v, k)
            last[v] = max(last.get(v, k), k)
        for v in g.reads:
            first.setdefault(v, k)
            last[v] = max(last.get(v, k), k)
    stored = [v for v in program.values.values() if v.role == "stored"]
    sizes: list[int] = []
    until: list[int] = []  # per slot: the last kernel using what it holds
    slots: dict[str, int] = {}
    for v in sorted(stored, key=lambda v: (first.get(v.name, 0), v.name)):
        k = first.get(v.name, 0)
        free = [s for s in range(len(sizes)) if until[s] < k]
        fits = [s for s in free if sizes[s] >= v.nbytes]
        if fits:
            s = min(fits, key=lambda s: (sizes[s], s))
        elif free:
            s = max(free, key=lambda s: (sizes[s], -s))
        else:
            sizes.append(0)
            until.append(-1)
            s = len(sizes) - 1
        sizes[s] = max(sizes[s], v.nbytes)
        until[s] = last.get(v.name, k)
        slots[v.name] = s
    return Storage({v: (first[v], last[v]) for v in first}, slots, sizes)


class Arena:
    """The slots in one device slab (th_arena_create)."""

    def __init__(self, sizes: Sequence[int], align: int = 256):
        arr = (ctypes.c_uint64 * max(1, len(sizes)))(*sizes)
        self._h = ctypes.c_void_p()
        call("th_arena_create", arr, len(sizes), align, ctypes.byref(self._h))
        self.addresses = []
        for i in range(len(sizes)):
            p = ctypes.c_void_p()
            call("th_arena_slot", self._h, i, ctypes.byref(p))
            self.addresses.append(p.value)
        b = ctypes.c_uint64()
        call("th_arena_bytes", self._h, ctypes.byref(b))
        self.bytes = b.value

    def destroy(self) -> None:
        if self._h is not None:
            call("th_arena_destroy", self._h)
            self._h = None

    def __del__(self):
        try:
            self.destroy()
        except Exception:
            pass


class Pool:
    """A reserved range of device addresses that hands out blocks (th_pool_*):
    the slots of executables allocated one at a time, as ``planned`` allocates
    each (src/Compiler/runtime/runtime.jl:415), all inside one range."""

    def __init__(self, reserve: int = 64 << 30):
        self._h = ctypes.c_void_p()
        self._closed = False
        call("th_pool_create", ctypes.c_uint64(reserve), ctypes.byref(self._h))

    def alloc(self, nbytes: int, align: int = 256) -> int:
        p = ctypes.c_void_p()
        call("th_pool_alloc", self._h, ctypes.c_uint64(nbytes), ctypes.c_uint64(align), ctypes.byref(p))
        return p.value

    def free(self, ptr: int) -> None:
        call("th_pool_free", self._h, ctypes.c_void_p(ptr))

    def info(self) -> tuple[int, int, int]:
        """(base address, reserved bytes, mapped bytes)."""
        b, r, m = ctypes.c_void_p(), ctypes.c_uint64(), ctypes.c_uint64()
        call("th_pool_info", self._h, ctypes.byref(b), ctypes.byref(r), ctypes.byref(m))
        return b.value, r.value, m.value

    def destroy(self) -> None:
        """Give the range back; blocks still taken keep it until the last of
        them is freed (th_pool_destroy), so the handle stays for their frees."""
        if not self._closed:
            self._closed = True
            call("th_pool_destroy", self._h)

    def __del__(self):
        try:
            self.destroy()
        except Exception:
            pass


class PoolSlots:
    """The slots of one executable taken from a Pool one by one, freed with it."""

    def __init__(self, pool: Pool, sizes: Sequence[int], align: int = 256):
        self.pool = pool
        self.addresses = [pool.alloc(n, align) for n in sizes]
        self.bytes = sum(sizes)

    def destroy(self) -> None:
        for a in self.addresses:
            self.pool.free(a)
        self.addresses = []

    def __del__(self):
        try:
            self.destroy()
        except Exception:
            pass


def _shown(name: str, doc: str) -> property:
    """An attribute that tells its reader where the executable's results lie, or
    that runs into them: reading it ends what only a program that sees nothing
    but its calls' results may have (Executable.lend)."""
    def read(self):
        self._settle()
        return getattr(self, name)
    return property(read, doc=doc)


class Executable:
    """A prepared program: its storage, launches and (once captured) graph.
    Its slots lie in one arena slab, or, given a Pool, are taken from the
    pool's reserved range one by one."""

    results = _shown("_results", "The results' one allocation, for as long as the executable.")
    addresses = _shown("_addresses", "Where each value lies.")
    launches = _shown("_launches", "A launch a group, in order.")
    graph = _shown("_graph", "What capture recorded, or None.")

    def __init__(self, program: Program, target: HIPTarget, inputs: Sequence[torch.Tensor], point: bool = True,
                 pool: Pool | None = None):
        self.program = program
        self.target = target
        self.storage = storage(program)
        self.arena = Arena(self.storage.sizes) if pool is None else PoolSlots(pool, self.storage.sizes)
        self.own: dict[str, torch.Tensor] = {}
        self.bound: dict[str, torch.Tensor] = {}
        self._addresses: dict[str, int] = {}
        # The results share one allocation, each at a 256-byte boundary, so a
        # call returns them with one copy and reads its numbers at once.
        self.result_at: dict[str, tuple[int, int]] = {}
        at = 0
        for name, v in program.values.items():
            if v.role == "result":
                nbytes = max(1, v.count) * _ELEMENT[v.dtype]
                self.result_at[name] = (at, nbytes)
                at += (nbytes + 255) // 256 * 256
        self._results = target.allocate(torch.uint8, max(at, 256))
        self._seen = False  # whether anyone has been told where the results lie
        # What the last run wrote instead, the stream it ran on, the memory's version then.
        self._last: tuple[torch.Tensor, torch.cuda.Stream, int] | None = None
        for name, v in program.values.items():
            if v.role == "stored":
                self._addresses[name] = self.arena.addresses[self.storage.slots[name]]
            elif v.role == "result":
                self._addresses[name] = self._results.data_ptr() + self.result_at[name][0]
        self._check(inputs)
        for name, x in zip(program.inputs, inputs):
            self._take(name, x, point)
        self._launches = [g.build(dict(self._addresses)) for g in program.groups]
        self._place_workspaces(pool)
        # Every place a launch holds a result's address, as th_launches_lend takes them.
        refs = [(l.handle.value, i, self.result_at[v][0]) for g, l in zip(program.groups, self._launches)
                for i, v in enumerate(g.values) if v in self.result_at]
        n = max(1, len(refs))
        self._result_refs = ((ctypes.c_void_p * n)(*(r[0] for r in refs)), (ctypes.c_int32 * n)(*(r[1] for r in refs)),
                             (ctypes.c_uint64 * n)(*(r[2] for r in refs)), len(refs))
        self._handles = (ctypes.c_void_p * max(1, len(self._launches)))(*(l.handle.value for l in self._launches))
        self._graph: Graph | Direct | None = None
        self._moved: set[int] = set()

    def _place_workspaces(self, pool: Pool | None) -> None:
        """Give each launch's workspace (attention's dS', split sums, ...) a
        slot beside the program's: the slots and workspaces are laid out
        again in one arena (or taken from the pool), the launches repointed
        to it.  The first arena, built before the workspaces were known,
        goes."""
        self.workspaces = [l.workspace() for l in self._launches]
        if not any(self.workspaces):
            return
        sizes = list(self.storage.sizes) + [w for w in self.workspaces if w]
        arena = Arena(sizes) if pool is None else PoolSlots(pool, sizes)
        for name, v in self.program.values.items():
            if v.role == "stored":
                self._addresses[name] = arena.addresses[self.storage.slots[name]]
        for g, l in zip(self.program.groups, self._launches):
            for i, v in enumerate(g.values):
                if v in self.program.values and self.program.values[v].role == "stored":
                    l.repoint(i, self._addresses[v])
        j = len(self.storage.sizes)
        for l, w in zip(self._launches, self.workspaces):
            if w:
                l.set_workspace(arena.addresses[j])
                j += 1
        self.arena.destroy()
        self.arena = arena

    # -- binding -------------------------------------------------------------

    def _check(self, inputs: Sequence[torch.Tensor]) -> None:
        if len(inputs) != len(self.program.inputs):
            raise ValueError(f"{self.program.name} takes {len(self.program.inputs)} arrays, got {len(inputs)}")
        for name, x in zip(self.program.inputs, inputs):
            v = self.program.values[name]
            if not isinstance(x, torch.Tensor) or x.dtype != v.dtype or x.numel() != v.count:
                raise ValueError(f"{self.program.name}: argument {name} must be {v.count} elements of {v.dtype}, "
                                 f"got {getattr(x, 'dtype', type(x))} x {getattr(x, 'numel', lambda: '?')()}")

    def _take(self, name: str, x: torch.Tensor, point: bool) -> None:
        v = self.program.values[name]
        if point and self.target.pointable(x, x.data_ptr()):
            self.bound[name] = x
            self._addresses[name] = x.data_ptr()
            self.own.pop(name, None)
        else:
            buf = self.own.get(name)
            if buf is None:
                buf = self.target.allocate(v.dtype, v.count)
                self.own[name] = buf
            self.target.upload_into(buf, x.reshape(-1))
            self.bound.pop(name, None)
            self._addresses[name] = buf.data_ptr()

    def bind(self, *inputs: torch.Tensor) -> "Executable":
        """bind!(ex, inputs...) (runtime.jl:719): copy into own buffers."""
        return self._rebind(inputs, point=False)

    def point(self, *inputs: torch.Tensor) -> "Executable":
        """point!(ex, inputs...) (runtime.jl:818): the caller's arrays become storage."""
        return self._rebind(inputs, point=True)

    def _rebind(self, inputs, point: bool) -> "Executable":
        self._check(inputs)
        for name, x in zip(self.program.inputs, inputs):
            before = self._addresses[name]
            self._take(name, x, point)
            after = self._addresses[name]
            if after != before:
                for k, (g, l) in enumerate(zip(self.program.groups, self._launches)):
                    for i, v in enumerate(g.values):
                        if v == name:
                            l.repoint(i, after)
                            self._moved.add(k)
        return self

    # -- running --------------------------------------------------------------

    def _alive(self) -> None:
        for l in self._launches:
            l.handle  # raises for a destroyed launch

    def lend(self) -> torch.Tensor | None:
        """One run whose results go to memory of its own, laid out as
        ``result_at``, which its caller keeps; every launch, and so every
        recording, timing or run of it, stays at the executable's results.
        None, and nothing run, where those are what the caller has to have
        (someone knows where they lie), where torch would not order the memory
        with the launches (another current stream than the library's), or
        where the recording is not the launches themselves (a graph's every
        node with a result would be retargeted)."""
        if self._seen or not (self._graph is None or isinstance(self._graph, Direct)):
            return None
        handle = ctypes.c_void_p()
        call("th_get_stream", ctypes.byref(handle))
        stream = torch.cuda.current_stream(self.target.device)
        if (handle.value or 0) != stream.cuda_stream:
            return None
        self._alive()
        self._last = None
        memory = torch.empty_like(self._results)
        call("th_launches_lend", self._handles, len(self._launches), *self._result_refs, memory.data_ptr(),
             self._results.data_ptr())
        self._moved.clear()
        self._last = memory, stream, 0 if memory.is_inference() else memory._version
        return memory

    def _settle(self) -> None:
        """From here on every run's results are where the executable says, the
        last one's too: copied there on the stream that it ran on, or, where
        their holder has written over them, computed again."""
        self._seen = True
        if self._last is None:
            return
        (memory, stream, version), self._last = self._last, None
        with torch.cuda.stream(stream):
            if memory.is_inference() or memory._version == version:
                self._results.copy_(memory)
            else:
                self.execute()

    def execute(self) -> "Executable":
        """execute!(ex) (runtime.jl:1158): each launch in order."""
        self._last = None
        self._alive()
        call("th_launches_run", self._handles, len(self._launches))
        self._moved.clear()  # the launches themselves carry the new addresses
        return self

    def capture(self, graph: bool | None = None) -> "Executable":
        """capture!(ex) (runtime.jl:1185): one graph of every launch, or the
        launches themselves where the target measures direct launches faster
        for this many kernels (HIPTarget.graph_pays); ``graph`` forces it."""
        if self._graph is not None:
            self._graph = self.target.recapture(self._graph, self._launches, as_graph=graph)
        else:
            self._graph = self.target.capture(self._launches, graph=graph)
        self._moved.clear()
        return self

    @property
    def graphed(self) -> bool:
        """Whether what capture recorded replays as a graph."""
        return isinstance(self._graph, Graph)

    def replay(self) -> "Executable":
        """replay!(ex) (runtime.jl:1208): retarget what moved, then one graph launch."""
        if self._graph is None:
            raise RuntimeError("replay before capture")
        self._last = None
        if isinstance(self._graph, Graph):
            for k in sorted(self._moved):
                self.target.retarget(self._graph, k,
                                     [Move(n, 0, self._addresses[n], 0) for n in self.program.groups[k].values],
                                     lambda: None)
        self._moved.clear()
        self.target.replay(self._graph)
        return self

    def outputs(self) -> list[torch.Tensor]:
        """outputs(ex): the result buffers themselves (the next run overwrites them)."""
        out = []
        results = self.results
        for name in self.program.outputs:
            v = self.program.values[name]
            off, nbytes = self.result_at[name]
            t = results[off:off + nbytes].view(v.dtype)
            out.append(t[0] if v.scalar else t.view(*reversed(v.dims)) if len(v.dims) > 1 else t)
        return out

    def work(self) -> tuple[float, float]:
        """Algorithmic bytes and flops of one run, summed over launches."""
        b = f = 0.0
        for l in self._launches:
            w = l.work()
            b += w.bytes
            f += w.flops
        return b, f

    def explain(self) -> str:
        """explain (runtime.jl:1216-1238): each kernel and what runs it."""
        ws = sum(1 for w in self.workspaces if w)
        lines = [f"{self.program.name}: {len(self._launches)} launches, arena {self.arena.bytes} bytes "
                 f"in {len(self.storage.sizes)} slots" + (f" and {ws} workspaces" if ws else "")]
        for g, l in zip(self.program.groups, self._launches):
            lines.append(f"  {g.name}: reads {', '.join(g.reads)}; writes {', '.join(g.writes)}; {l.describe()}")
        if self._graph is not None:
            lines.append("  replays as " + ("one graph" if self.graphed else "its launches, one by one (cheaper "
                                            "than a graph for this many kernels on this device)"))
        return "\n".join(lines)


def prepare(program: Program, target: HIPTarget, *inputs: torch.Tensor, point: bool = True,
            pool: Pool | None = None) -> Executable:
    return Executable(program, target, inputs, point=point, pool=pool)


class Compiled:
    """compile(f, args...) for a planned program (compile.jl:48-62, 310-349)."""

    def __init__(self, program: Program, target: HIPTarget, inputs: Sequence[torch.Tensor], capture: bool = True):
        self.executable = ex = prepare(program, target, *inputs)
        self.signature = [(x.dtype, tuple(x.shape)) for x in inputs]
        if capture:
            ex.capture()
        # Where each result lies in the executable's result allocation, and
        # the span holding the numbers (read to the host in one copy).
        self._layout = []
        for name in program.outputs:
            v = program.values[name]
            off, nbytes = ex.result_at[name]
            shape = tuple(reversed(v.dims)) if len(v.dims) > 1 else (max(1, v.count),)
            strides = tuple(math.prod(shape[i + 1:]) for i in range(len(shape)))
            self._layout.append((v.dtype, v.scalar, shape, strides, off // _ELEMENT[v.dtype]))
        spans = [ex.result_at[n] for n in program.outputs if program.values[n].scalar]
        self._numbers = (min(a for a, _ in spans), max(a + n for a, n in spans)) if spans else None
        if spans:
            lo, hi = self._numbers
            self._host = torch.empty((hi - lo + 255) // 256 * 256, dtype=torch.uint8, pin_memory=True)
            self._host_numbers = [self._host.view(dt)[at - lo // _ELEMENT[dt]] if scalar else None
                                  for dt, scalar, _, _, at in self._layout]

    def __call__(self, *args: torch.Tensor):
        sig = [(getattr(x, "dtype", None), tuple(getattr(x, "shape", ()))) for x in args]
        if sig != self.signature:
            raise ValueError(f"call does not match the compiled signature {self.signature}: {sig}")
        ex = self.executable
        ex.point(*args)
        # The results go to an allocation that this call's caller keeps: a copy
        # into one would read and write them once more (1 GiB: 418 us of a
        # 1049 us call).
        lent = ex.lend()
        if lent is not None:
            return self._returned(lent, lent=True)
        ex.replay() if ex._graph is not None else ex.execute()
        return self.returned()

    def returned(self):
        """Arrays copied, numbers read to the host (compile.jl:334-349): one
        copy of the result allocation, whose views are the arrays returned,
        then one read of the span holding the numbers."""
        ex = self.executable
        if ex._last is not None:
            ex._settle()
        return self._returned(ex._results.clone(), lent=False)

    def _returned(self, fresh: torch.Tensor, lent: bool):
        # The arrays first: the device is still at work on the numbers.
        typed = {}
        out = []
        for dtype, scalar, shape, strides, at in self._layout:
            if scalar:
                out.append(None)
                continue
            if dtype not in typed:
                typed[dtype] = fresh.view(dtype)
            out.append(typed[dtype].as_strided(shape, strides, at))
        if self._numbers is not None:
            lo, hi = self._numbers
            if lent:  # on the library's stream, which is torch's current one
                call("th_download", self._host.data_ptr(), fresh.data_ptr() + lo, hi - lo)
            else:
                self._host[:hi - lo].copy_(fresh[lo:hi])
            for i, number in enumerate(self._host_numbers):
                if number is not None:
                    out[i] = number.item()
        return tuple(out)


def compile(program: Program, target: HIPTarget, *inputs: torch.Tensor, capture: bool = True) -> Compiled:
    return Compiled(program, target, inputs, capture=capture)
