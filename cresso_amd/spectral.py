"""Host orchestration of the spectral/hash route.

The library keeps no state of its own: plans live here, keyed by
(device, shape, freqs, hash_bins, hash_tables), together with their device
workspace (carrier tables, cached coordinate-hash bins, scratch).

A step of several spectral tensors (`step_many`) first batches the tensors
that share a plan (and dtypes, hard channel and hash state): one batched C
call steps a batch, every launch covering all its tensors, with the plan's
tables held once and per-step scratch (about 4 bytes per element plus its
blocks' partial sums) once per tensor.  A batch holds at most BATCH_BYTES of
such scratch; larger groups are cut into that many chunks.  The units of work
(batches and single tensors) are spread over up to LANES side streams (default priority),
so that one unit's small finish kernels and partly filled sweeps overlap
with another's work.  Every lane has its own workspace per unit kind: units
that share a workspace run one after another on that lane's stream, so its
per-step scratch is never used concurrently.  The side streams wait for the
caller's stream before the first launch and the caller's stream waits for
all of them after the last, so the step is ordered like any other work on
the caller's stream; the group's scalar tensors step on the caller's stream
meanwhile.  A single spectral tensor runs on the caller's stream
directly.

Device memory held: per (plan, lane) a workspace of the plan's tables (about
(2 + 4) bytes per element at two tables of <= 256 bins) and its scratch;
the optimizer's load_state_dict keeps those whose plan the loaded state still
uses (`retain`) and frees the others; `reset()` frees them all.
"""

from __future__ import annotations

import ctypes
import weakref
from typing import Dict, List, Sequence, Tuple

import torch

from . import _native

# (param dtype, grad dtype) pairs of the library's spectral step; the force is
# the grad converted to the work dtype, as in cresso_v5.py:907-912: fp32 for
# fp32/bf16/fp16 params, fp64 for fp64 params, whose state is fp64 too and
# whose plans carry the fp64 work dtype (cresso_v5.py:119-124).
_DTYPE_PAIRS = {(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                (torch.float32, torch.bfloat16), (torch.float32, torch.float16), (torch.float64, torch.float64)}

_VEC_KEYS = ("q_cos", "q_sin", "p_cos", "p_sin", "metric_cos", "metric_sin", "metric_p_cos", "metric_p_sin",
             "calcium_cos", "calcium_sin", "mode_confidence")


def assign_lanes(keys: Sequence[tuple], lanes: int) -> List[int]:
    """Lane of each tensor of a multi-tensor step, given its plan key.

    The m tensors of one key take min(lanes, m) distinct lanes, round robin
    from a start lane that moves on with every new key (so single tensors of
    different shapes spread over the lanes).  Each (key, lane) pair is one
    workspace, used by its tensors one after another on that lane's stream.
    """
    count: Dict[tuple, int] = {}
    for k in keys:
        count[k] = count.get(k, 0) + 1
    seen: Dict[tuple, int] = {}
    base: Dict[tuple, int] = {}
    out = []
    for k in keys:
        if k not in base:
            base[k] = len(base) % lanes
        j = seen.get(k, 0)
        seen[k] = j + 1
        out.append((base[k] + j % min(lanes, count[k])) % lanes)
    return out


def _make_plan(lib, shape, freqs: Tuple[int, ...], rank: int, bins: int, tables: int, work: int) -> ctypes.c_void_p:
    shp = (ctypes.c_int64 * 8)(*shape)
    fr = (ctypes.c_int64 * max(1, len(freqs)))(*freqs)
    plan = lib.cresso_spectral_plan_create_ex(shp, len(shape), fr, rank, bins, tables, work)
    if not plan:
        _native.check(-1, "spectral route plan")
    return ctypes.c_void_p(plan)


class _Workspace:
    """A plan with its device workspace: for one tensor (count=None) or for
    batches of up to `count` tensors."""

    def __init__(self, lib, shape, freqs_host: Tuple[int, ...], rank: int, bins: int, tables: int, group: dict,
                 device: torch.device, count=None, work: int = _native.F32):
        self.lib = lib
        self.count = count
        self.plan = _make_plan(lib, shape, freqs_host, rank, bins, tables, work)
        hyper = _native.hyper_from_group(group)
        stream = ctypes.c_void_p(_native.stream_handle(device))
        if count is None:
            nbytes = int(lib.cresso_spectral_workspace_bytes(self.plan))
            self.buf = torch.empty(nbytes, dtype=torch.uint8, device=device)
            rc = lib.cresso_spectral_workspace_init(self.plan, ctypes.c_void_p(self.buf.data_ptr()),
                                                    ctypes.c_size_t(nbytes), ctypes.byref(hyper), stream)
        else:
            nbytes = int(lib.cresso_spectral_batched_workspace_bytes(self.plan, count))
            self.buf = torch.empty(nbytes, dtype=torch.uint8, device=device)
            rc = lib.cresso_spectral_batched_workspace_init(self.plan, count, ctypes.c_void_p(self.buf.data_ptr()),
                                                            ctypes.c_size_t(nbytes), ctypes.byref(hyper), stream)
        _native.check(rc, "spectral workspace init")

    def __del__(self):
        plan = getattr(self, "plan", None)
        if plan is not None and plan.value:
            try:
                self.lib.cresso_spectral_plan_destroy(plan)
            except Exception:
                pass


def lane_scratch_bytes(numel: int) -> int:
    """Least per-tensor scratch of a batched step: the tangent field (4 bytes
    per element), a few KB and small per-row and per-column sums.  (The blocks'
    partial sums and histograms come on top: SpectralEngine._lane_bytes.)"""
    return 4 * numel + (1 << 16)


class SpectralEngine:
    READY = True
    LANES = 4                 # side streams of a multi-tensor step
    BATCH = True              # batch same-plan tensors into one launch per kernel
    BATCH_BYTES = 512 << 20   # per-tensor scratch held by one batch (C4: 3 % faster than 256 MiB, as fast as 1 GiB)

    lane_bytes: Dict[tuple, int] = {}   # plan key -> per-tensor scratch of its batches (a dict of each engine's own)

    def __init__(self):
        self.lib = _native.load()
        self.lane_bytes = {}
        self.ws: Dict[tuple, _Workspace] = {}   # (plan key, unit kind, lane) -> workspace
        self.version = 0                        # changes with every workspace made or dropped
        self.side: Dict[torch.device, List[torch.cuda.Stream]] = {}
        self.forks: Dict[torch.device, _Fork] = {}
        self.freq_cache: Dict[int, Tuple[int, ...]] = {}

    def reset(self) -> None:
        """Forget cached frequency lists and free every workspace."""
        self.freq_cache.clear()
        self.ws.clear()
        self.version += 1

    def retain(self, keys) -> None:
        """Forget cached frequency lists; free the workspaces whose plan key is
        not in `keys` (a workspace depends on its plan key only)."""
        self.freq_cache.clear()
        for wkey in [k for k in self.ws if k[0] not in keys]:
            del self.ws[wkey]
        self.version += 1

    def plan_key(self, param: torch.Tensor, st: dict, group: dict) -> tuple:
        """The plan key of a spectral tensor: (device, shape, freqs, hash_bins, hash_tables, work dtype)."""
        work = _native.F64 if param.dtype == torch.float64 else _native.F32
        return (param.device, tuple(int(d) for d in param.shape), self._freqs(st), int(group["hash_bins"]),
                int(group["hash_tables"]), work)

    def _freqs(self, st: dict) -> Tuple[int, ...]:
        fr = st["freqs"]
        key = id(fr)
        got = self.freq_cache.get(key)
        if got is None or got[0] is not fr:
            host = tuple(int(v) for v in fr.detach().to("cpu", torch.long).reshape(-1).tolist())
            got = (fr, host)
            self.freq_cache[key] = got
        return got[1]

    def _workspace(self, key: tuple, lane: int, rank: int, group: dict, count=None) -> _Workspace:
        wkey = (key, count is not None, lane)
        ws = self.ws.get(wkey)
        if ws is None or (count is not None and ws.count < count):
            device, shape, freqs, bins, tables, work = key
            ws = None
            self.ws.pop(wkey, None)
            ws = _Workspace(self.lib, shape, freqs, rank, bins, tables, group, device, count, work)
            self.ws[wkey] = ws
            self.version += 1
        return ws

    def _lane_bytes(self, key: tuple, rank: int, numel: int) -> int:
        """Per-tensor scratch of a batched step, for sizing batches: the
        library's stride between tensors of a batched workspace."""
        got = self.lane_bytes.get(key)
        if got is None:
            if not isinstance(key, tuple):   # (no plan to ask)
                return lane_scratch_bytes(numel)
            _, shape, freqs, bins, tables, work = key
            plan = _make_plan(self.lib, shape, freqs, rank, bins, tables, work)
            try:
                one, two = (int(self.lib.cresso_spectral_batched_workspace_bytes(plan, n)) for n in (1, 2))
            finally:
                self.lib.cresso_spectral_plan_destroy(plan)
            got = self.lane_bytes[key] = two - one
        return got

    def _prepare(self, param: torch.Tensor, grad: torch.Tensor, st: dict, group: dict):
        """Validate one tensor's state and build its descriptor; -> (key, rank, desc)."""
        if (param.dtype, grad.dtype) not in _DTYPE_PAIRS:
            raise RuntimeError(f"CRESSO5 spectral route on MI355X supports fp64/fp32/bf16/fp16 params with grads of "
                               f"the same dtype, and fp32 params with bf16/fp16 grads (got {param.dtype} / {grad.dtype})")
        sdt = torch.float64 if param.dtype == torch.float64 else torch.float32
        for k in ("force_rms", "drive_energy", "surprise", "action", "omega") + _VEC_KEYS:
            if st[k].dtype != sdt:
                raise RuntimeError(f"CRESSO5 spectral state {k} has dtype {st[k].dtype}, expected {sdt}")
        rank = int(st["omega"].numel())
        bins, tables = int(group["hash_bins"]), int(group["hash_tables"])
        key = self.plan_key(param, st, group)
        shape = key[1]
        cut = int(group["thin_matrix_hard_cutoff"])
        thin = param.ndim == 2 and cut > 0 and min(shape) <= cut
        hard = param.numel() >= int(group["hard_channel_min_size"]) and not thin
        d = _native.SpectralDesc()
        d.param = param.data_ptr()
        d.grad = grad.data_ptr()
        d.param_dtype = _native.DTYPE_CODE[param.dtype]
        d.grad_dtype = _native.DTYPE_CODE[grad.dtype]
        d.numel = param.numel()
        d.force_rms = st["force_rms"].data_ptr()
        d.drive_energy = st["drive_energy"].data_ptr()
        d.surprise = st["surprise"].data_ptr()
        d.action = st["action"].data_ptr()
        d.omega = st["omega"].data_ptr()
        for k in _VEC_KEYS:
            setattr(d, k, st[k].data_ptr())
        if hard and bins > 0 and "hash_energy" in st:
            for k in ("hash_energy", "hash_impulse", "hash_refractory"):
                if tuple(st[k].shape) != (tables, bins) or st[k].dtype != sdt:
                    raise RuntimeError(f"CRESSO5 spectral state {k} has shape {tuple(st[k].shape)}, expected "
                                       f"({tables}, {bins}) {sdt} (hash_bins/hash_tables changed after init?)")
            d.hash_energy = st["hash_energy"].data_ptr()
            d.hash_impulse = st["hash_impulse"].data_ptr()
            d.hash_refractory = st["hash_refractory"].data_ptr()
        d.step = int(st["step"]) + 1
        d.hard = 1 if hard else 0
        return key, rank, d

    def _streams(self, device: torch.device, n: int) -> List[torch.cuda.Stream]:
        have = self.side.setdefault(device, [])
        while len(have) < n:
            have.append(torch.cuda.Stream(device=device))   # default priority
        return have[:n]

    def _units(self, prepared: list, sts: list) -> list:
        """Cut a step's tensors into units: (unit key, plan key, rank, [desc], [state]).
        Tensors batch when they share the plan, dtypes, hard channel and hash
        state; fp64 tensors step one at a time (fp64 plans are not batched)."""
        groups: Dict[tuple, list] = {}
        for i, (key, rank, d) in enumerate(prepared):
            bkey = (key, d.param_dtype, d.grad_dtype, d.hard, bool(d.hash_energy))
            alone = not self.BATCH or d.param_dtype == _native.F64
            groups.setdefault((bkey, i) if alone else bkey, []).append(i)
        units = []
        for bkey, idx in groups.items():
            key, rank, _ = prepared[idx[0]]
            if len(idx) == 1:
                units.append(((key, False), key, rank, [prepared[idx[0]][2]], [sts[idx[0]]]))
                continue
            per = self._lane_bytes(key, rank, prepared[idx[0]][2].numel)
            chunks = -(-len(idx) * per // self.BATCH_BYTES)
            m = -(-len(idx) // chunks)
            for c in range(0, len(idx), m):
                sel = idx[c:c + m]
                units.append(((key, True, m), key, rank, [prepared[i][2] for i in sel], [sts[i] for i in sel]))
        return units

    def step_many(self, items: Sequence[Tuple[torch.Tensor, torch.Tensor, dict]], group: dict, between=None) -> None:
        """Every spectral tensor of a param group: (param, grad, state) each.
        between: work for the caller's stream that may run beside the side
        streams (called once)."""
        plan = self._plan(items, group)
        for _, _, sts, _, _ in plan:
            for st in sts:
                st["step"] += 1
        Launch(self, [(ws, (_native.SpectralDesc * len(descs))(*descs), lane, device)
                      for ws, descs, _, lane, device in plan]).run(_native.hyper_from_group(group), between)

    def _plan(self, items, group: dict) -> list:
        """The step's units: (workspace, [desc], [state], lane or None, device).
        lane None: the caller's stream (a single tensor).  Workspaces created
        here are initialised on the caller's stream, before the lanes fork."""
        if len(items) == 1:
            p, g, st = items[0]
            key, rank, d = self._prepare(p, g, st, group)
            return [(self._workspace(key, 0, rank, group), [d], [st], None, p.device)]
        by_dev: Dict[torch.device, list] = {}
        for it in items:
            by_dev.setdefault(it[0].device, []).append(it)
        plan = []
        for device, its in by_dev.items():
            prepared = [self._prepare(p, g, st, group) for p, g, st in its]
            units = self._units(prepared, [st for _, _, st in its])
            nl = min(self.LANES, len(units))
            lanes = assign_lanes([u[0][:2] for u in units], nl)
            for (ukey, key, rank, descs, sts), lane in zip(units, lanes):
                count = ukey[2] if ukey[1] else None
                plan.append((self._workspace(key, lane, rank, group, count), descs, sts, lane, device))
        return plan

    def _fork(self, device: torch.device, lanes: int) -> "_Fork":
        fork = self.forks.get(device)
        if fork is None or len(fork.streams) < lanes:   # (streams are made as they are needed)
            fork = self.forks[device] = _Fork(self.lib, self._streams(device, lanes), device)
        return fork


class _Fork:
    """A device's side streams and the library's events that fork them from
    and join them to the caller's stream."""

    def __init__(self, lib, streams: List[torch.cuda.Stream], device: torch.device):
        self.lib = lib
        self.streams = streams
        self.handles = (ctypes.c_void_p * len(streams))(*[int(s.cuda_stream) for s in streams])
        with torch.cuda.device(device):
            self.fork = lib.cresso_fork_create(len(streams))
        if not self.fork:
            _native.check(-1, "side streams")

    def __del__(self):
        if getattr(self, "fork", None):
            try:
                self.lib.cresso_fork_destroy(self.fork)
            except Exception:
                pass


class Launch:
    """The launches of a step: units (workspace, descriptor array, lane or
    None, device).  Per device one call steps the units; several units run on
    the side streams, which fork from the caller's stream before the first
    launch and join it after the last (a lone tensor: the caller's stream)."""

    def __init__(self, engine: SpectralEngine, units: list):
        self.engine = engine
        self.keep = units                 # workspaces and descriptor arrays
        self.devices = []
        for device in dict.fromkeys(u[3] for u in units):
            mine = [u for u in units if u[3] == device]
            arr = (_native.SpectralUnit * len(mine))()
            for a, (ws, descs, lane, _) in zip(arr, mine):
                a.plan, a.workspace, a.workspace_bytes = ws.plan.value, ws.buf.data_ptr(), ws.buf.numel()
                a.descs, a.count, a.batched = ctypes.addressof(descs), len(descs), 0 if ws.count is None else 1
                a.lane = 0 if lane is None else lane
            lanes = 0 if mine[0][2] is None else 1 + max(u[2] for u in mine)
            self.devices.append((device, arr, len(mine), lanes))

    def run(self, hyper, between=None) -> None:
        """between: run after the launches, on the caller's stream, beside the
        side streams."""
        lib, forked = self.engine.lib, []
        try:
            for device, arr, n, lanes in self.devices:
                caller = ctypes.c_void_p(_native.stream_handle(device))
                if lanes == 0:
                    handles, count = ctypes.pointer(caller), 1
                else:
                    fork = self.engine._fork(device, lanes)
                    handles, count = fork.handles, lanes
                    forked.append((fork, caller, lanes))   # (a begin that fails may have forked some)
                    _native.check(lib.cresso_fork_begin(fork.fork, caller, handles, lanes), "side streams")
                _native.check(lib.cresso_spectral_step_units(arr, n, ctypes.byref(hyper), handles, count),
                              "spectral route step")
            if between is not None:
                between()
        except BaseException:
            self._join(forked)   # (the first error is the one to raise)
            raise
        failed = self._join(forked)
        if failed is not None:
            raise failed

    def _join(self, forked: list):
        """Every forked stream joins its caller's, whatever happens; -> the first error."""
        failed = None
        for fork, caller, lanes in forked:
            try:
                _native.check(self.engine.lib.cresso_fork_end(fork.fork, caller, fork.handles, lanes), "side streams")
            except RuntimeError as err:
                failed = failed or err
        return failed


class SteadyStep:
    """The steady state of a group's spectral tensors: the units of a step that
    has run, with their workspaces, and the C++ guard that checks every
    parameter, grad and state tensor again on each step and writes their
    descriptors.  fill() returns False when anything differs; the general path
    then takes the step.  The workspaces stay the engine's: one that it drops
    is freed, and the steady step is at an end (ready())."""

    def __init__(self, engine: SpectralEngine, items, group: dict, hb):
        plan = engine._plan(items, group)
        if any(ws.count is None and len(descs) != 1 for ws, descs, _, _, _ in plan):
            raise ValueError("a unit without a batched workspace holds one tensor")
        by_state = {id(st): (p, st) for p, _, st in items}
        order = [by_state[id(st)] for _, _, sts, _, _ in plan for st in sts]
        descs = [d for _, ds, _, _, _ in plan for d in ds]
        self.engine = engine
        self.version = engine.version
        self.guard = hb.SpectralGuard([p for p, _ in order], [st["freqs"] for _, st in order],
                                      [(d.param_dtype, d.grad_dtype) for d in descs], [d.hard for d in descs],
                                      [1 if d.hash_energy else 0 for d in descs], int(group["hash_bins"]),
                                      int(group["hash_tables"]))
        self.descs = (_native.SpectralDesc * len(descs))()
        units, at, size = [], 0, ctypes.sizeof(_native.SpectralDesc)
        for ws, ds, _, lane, device in plan:
            units.append((ws, (_native.SpectralDesc * len(ds)).from_buffer(self.descs, at * size), lane, device))
            at += len(ds)
        self.launch = Launch(engine, units)
        self.launch.keep = [u[1] for u in units]
        self.workspaces = [weakref.ref(u[0]) for u in units]

    def ready(self) -> bool:
        if self.version != self.engine.version:
            return False
        for ws in self.workspaces:
            if ws() is None:
                return False
        return True

    def fill(self, state: dict) -> bool:
        return self.ready() and self.guard.fill(state, ctypes.addressof(self.descs))

    def run(self, state: dict, hyper, between=None) -> None:
        """The step (after fill() returned True)."""
        self.guard.bump(state)
        self.launch.run(hyper, between)
