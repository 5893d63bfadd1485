"""CPU tests of the drop-in contract: constructor validation, routing, state
layout and size, checkpoint dtype repair, failure semantics, C-ABI exports."""

import ctypes
import re
from pathlib import Path

import numpy as np
import pytest
import torch

import cresso_amd
from cresso_amd import CRESSO5, count_optimizer_state_elements, theoretical_state_elements
from cresso_amd import _native
from oracle import cresso_oracle as O

ROOT = Path(__file__).resolve().parents[1]


def test_modes_match_oracle_restatement():
    from cresso_amd.modes import hash_unit, mode_list, omega_tensor, freqs_tensor
    for args in [(8, 2, 5), (16, 2, 7), (16, 4, 7), (16, 3, 7), (8, 1, 5), (4, 2, 0), (40, 2, 2), (30, 1, 5), (0, 2, 5)]:
        assert mode_list(*args) == O.frequency_pack(*args)
        fr = freqs_tensor(*args, device="cpu")
        assert torch.equal(fr, O.make_freqs(*args))
        assert torch.equal(omega_tensor(fr), O.omega_from_freqs(fr))
    # omega is the correctly rounded fp32 square root (numpy's is IEEE): the
    # fp64 route widens this value, so one ulp would show at fp64 precision.
    fr = freqs_tensor(32, 2, 6, device="cpu").numpy().astype(np.float64)
    exact = np.sqrt(1.0 + (fr * fr).sum(axis=1)).astype(np.float32)
    assert np.array_equal(omega_tensor(torch.from_numpy(fr)).numpy(), exact)
    for n in range(20):
        for s in (0, 17, 101, 151, 170):
            assert hash_unit(n, s) == O.hash_unit(n, s)


@pytest.mark.parametrize("kw,msg", [
    (dict(lr=-1.0), "lr must be >= 0.0"),
    (dict(dt=1.5), "dt must be <= 1.0"),
    (dict(eps=float("nan")), "eps must be a finite scalar"),
    (dict(rank=-1), "rank must be non-negative"),
    (dict(hash_tables=0), "hash_tables must be >= 1"),
    (dict(min_spectral_size=0), "min_spectral_size must be >= 1"),
    (dict(thin_matrix_route="dense"), "thin_matrix_route must be one of"),
    (dict(cuda_ops="sometimes"), "cuda_ops must be one of"),
    (dict(min_gain=2.0, max_gain=1.0), "min_gain must be <= max_gain"),
    (dict(drive_clip=0.01), "drive_clip must be >= 0.1"),
    (dict(thin_matrix_min_aspect=0.5), "thin_matrix_min_aspect must be >= 1.0"),
    (dict(warmup_steps=-2), "warmup_steps must be non-negative"),
])
def test_constructor_validation_messages(kw, msg):
    p = torch.nn.Parameter(torch.zeros(4))
    with pytest.raises(ValueError, match=re.escape(msg)):
        CRESSO5([p], **kw)


def test_defaults_and_cuda_ops_normalization():
    p = torch.nn.Parameter(torch.zeros(4))
    g = CRESSO5([p]).param_groups[0]
    assert g["lr"] == 2e-3 and g["rank"] == 8 and g["hash_bins"] == 128 and g["cuda_ops"] == "auto"
    assert CRESSO5([p], cuda_ops=False).param_groups[0]["cuda_ops"] == "off"
    assert CRESSO5([p], cuda_ops=True).param_groups[0]["cuda_ops"] == "auto"
    assert cresso_amd.CRESSO is CRESSO5


@pytest.mark.parametrize("shape,route", [
    ((128, 16), "scalar"), ((4096, 16), "scalar"), ((16, 4096), "scalar"), ((4096, 4096), "spectral"),
    ((2048,), "spectral"), ((1000,), "scalar"), ((40, 30), "spectral"), ((200, 6), "scalar"), ((), "scalar"),
    ((512, 256, 3, 3), "spectral"), ((100, 20), "scalar"), ((64, 65), "spectral"),
])
def test_routing_matches_oracle(shape, route):
    p = torch.nn.Parameter(torch.zeros(shape))
    opt = CRESSO5([p])
    assert opt._route(p, opt.param_groups[0]) == route
    assert O.OracleCRESSO5([p]).route(p) == route


def test_thin_spectral_override_and_state_counts():
    for route, expect in (("scalar", 8), ("spectral", theoretical_state_elements((128, 16), rank=4, thin_matrix_route="spectral"))):
        p = torch.nn.Parameter(torch.zeros(128, 16))
        opt = CRESSO5([p], rank=4, thin_matrix_route=route)
        g = opt.param_groups[0]
        st = opt._init_spectral(p, g) if opt._route(p, g) == "spectral" else opt._init_scalar(p)
        assert count_optimizer_state_elements(opt) == expect
        assert ("q_cos" in st) == (route == "spectral")


def test_theoretical_state_elements_matches_oracle():
    for shape in [(128, 16), (4096, 4096), (2048,), (512, 256, 3, 3), (200, 6), (12, 10)]:
        for kw in [dict(), dict(thin_matrix_route="spectral"), dict(hash_bins=64, hash_tables=3),
                   dict(micro_field_max_size=256), dict(hard_channel_min_size=10**9)]:
            assert theoretical_state_elements(shape, 8, **kw) == O.theoretical_state_elements(shape, 8, **kw)


def test_spectral_state_layout_matches_oracle():
    p = torch.nn.Parameter(torch.zeros(64, 48))
    opt = CRESSO5([p], hash_bins=64, hash_tables=2)
    st = opt._init_spectral(p, opt.param_groups[0])
    orc = O.OracleCRESSO5([p.detach()], hash_bins=64, hash_tables=2)
    ost = {}
    orc._init_spectral(p.detach(), ost, torch.float32)
    assert list(st.keys()) == list(ost.keys())
    for k, v in ost.items():
        if torch.is_tensor(v):
            assert st[k].dtype == v.dtype and torch.equal(st[k], v), k
    assert count_optimizer_state_elements(opt) == theoretical_state_elements((64, 48), 8, hash_bins=64)


def test_load_state_dict_keeps_int_freqs_and_fp32_state_for_bf16_params():
    p = torch.nn.Parameter(torch.zeros(64, 48, dtype=torch.bfloat16))
    opt = CRESSO5([p], hash_bins=64)
    st = opt._init_spectral(p, opt.param_groups[0])
    st["q_cos"].fill_(0.123456789)
    st["step"] = 7
    sd = opt.state_dict()
    p2 = torch.nn.Parameter(torch.zeros(64, 48, dtype=torch.bfloat16))
    opt2 = CRESSO5([p2], hash_bins=64)
    opt2.load_state_dict(sd)
    st2 = opt2.state[p2]
    assert st2["freqs"].dtype == torch.long and torch.equal(st2["freqs"], st["freqs"])
    assert st2["q_cos"].dtype == torch.float32 and torch.equal(st2["q_cos"], st["q_cos"])
    assert st2["step"] == 7


def test_required_rejects_cpu_params():
    p = torch.nn.Parameter(torch.ones(4, 4))
    p.grad = torch.ones_like(p)
    opt = CRESSO5([p], cuda_ops="required", min_spectral_size=1)
    with pytest.raises(RuntimeError, match="cuda_ops='required'.*CUDA parameter"):
        opt.step()


def test_auto_and_off_do_not_silently_fall_back_to_cpu():
    for mode in ("auto", "off"):
        p = torch.nn.Parameter(torch.ones(4, 4))
        p.grad = torch.ones_like(p)
        with pytest.raises(RuntimeError):
            CRESSO5([p], cuda_ops=mode).step()


def test_sparse_grad_rejected():
    p = torch.nn.Parameter(torch.ones(4, 4))
    p.grad = torch.ones(4, 4).to_sparse()
    with pytest.raises(RuntimeError, match="does not support sparse gradients"):
        CRESSO5([p]).step()


def test_params_without_grad_are_skipped():
    p = torch.nn.Parameter(torch.ones(4, 4))
    opt = CRESSO5([p], cuda_ops="required")
    opt.step()
    assert len(opt.state) == 0


def test_library_loads_and_exports_every_declared_symbol():
    lib_path = ROOT / "cresso_amd" / "libcresso_hip.so"
    if not lib_path.exists():
        pytest.skip("library not built (python -m cresso_amd.build)")
    header = (ROOT / "include" / "cresso_hip.h").read_text()
    declared = set(re.findall(r"^\s*(?:[\w\*]+\s+)+\**(cresso_\w+)\s*\(", header, flags=re.M))
    assert {"cresso_hip_abi_version", "cresso_hip_last_error", "cresso_scalar_plan_step"} <= declared
    lib = ctypes.CDLL(str(lib_path))
    for name in sorted(declared):
        assert hasattr(lib, name), name
    lib = _native.load()
    assert lib.cresso_hip_abi_version() == _native.ABI_VERSION


def test_library_load_touches_its_thread_local_message(monkeypatch):
    # untouched, it leaves every library's thread-local accesses on the slow way (torch's host calls 10 to 25 % slower)
    if not _native.library_path().exists():
        pytest.skip("library not built")
    called = []

    class Library(ctypes.CDLL):
        def __getattribute__(self, name):
            f = super().__getattribute__(name)
            if name == "cresso_hip_last_error" and "_declared" in self.__dict__:
                called.append(name)
            return f

    declare = _native._declare

    def declared(lib):
        declare(lib)
        lib.__dict__["_declared"] = True

    monkeypatch.setattr(_native, "_LIB", None)
    monkeypatch.setattr(_native, "_ERR", None)
    monkeypatch.setattr(_native, "_declare", declared)
    monkeypatch.setattr(_native.ctypes, "CDLL", Library)
    _native.load()
    assert called


def test_plan_creation_rejects_bad_descriptors_without_gpu():
    lib_path = ROOT / "cresso_amd" / "libcresso_hip.so"
    if not lib_path.exists():
        pytest.skip("library not built")
    lib = _native.load()
    d = (_native.ScalarDesc * 1)()
    d[0].ndim = 2
    d[0].shape[0], d[0].shape[1] = 4, 4
    d[0].numel = 15  # inconsistent with the shape
    h = _native.Hyper()
    h.drive_clip = 4.0
    assert not lib.cresso_scalar_plan_create(d, 1, ctypes.byref(h))
    assert b"numel" in lib.cresso_hip_last_error()


def test_unit_drive_update_rejects_dtype_before_any_launch():
    # an unsupported param dtype is refused by the host checks, so the call
    # returns before touching the (here fake) device pointers or any GPU
    lib_path = ROOT / "cresso_amd" / "libcresso_hip.so"
    if not lib_path.exists():
        pytest.skip("library not built")
    lib = _native.load()
    fake = ctypes.c_void_p(1 << 20)
    h = _native.Hyper()
    h.drive_clip = 4.0
    rc = lib.cresso_drive_update(fake, _native.DTYPE_CODE[torch.float64], fake, fake, fake, None, None, fake, fake,
                                 16, 1, 1, ctypes.byref(h), fake, 1 << 20, None)
    assert rc == _native.CRESSO_E_UNSUPPORTED
    assert b"not supported" in lib.cresso_hip_last_error()


def test_hash_c_oracle_matches_numpy_oracle():
    so = ROOT / "oracle" / "_build" / "libcresso_hash_oracle.so"
    if not so.exists():
        pytest.skip("oracle C restatement not built (make -C oracle)")
    import numpy as np
    lib = ctypes.CDLL(str(so))
    lib.cresso_oracle_hash_bins.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_void_p]
    lib.cresso_oracle_hash_counts.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_void_p]
    for n, bins, salt in [(5000, 64, 0), (5000, 37, 3), (100003, 256, 1), (777, 7, 9)]:
        out = np.empty(n, dtype=np.int32)
        lib.cresso_oracle_hash_bins(n, bins, salt, out.ctypes.data)
        np.testing.assert_array_equal(out, O.hash_index_np(n, bins, salt).astype(np.int32))
        cnt = np.empty(bins, dtype=np.int64)
        lib.cresso_oracle_hash_counts(n, bins, salt, cnt.ctypes.data)
        np.testing.assert_array_equal(cnt, np.bincount(out, minlength=bins))


def test_hash_bigint_brute_force_on_small_n():
    # Textbook restatement with Python big ints: wrap to signed 64 bits after
    # every step, arithmetic shift on the signed value, floor-mod.
    def wrap(v):
        v &= (1 << 64) - 1
        return v - (1 << 64) if v >> 63 else v

    for salt in (0, 1, 5):
        s = salt + 1
        for bins in (64, 37):
            got = O.hash_index_np(300, bins, salt)
            for i in range(300):
                h = wrap(i * (1103515245 + 97 * s) + (12345 + 0x9E3779B1 * s))
                h = wrap(h ^ (h >> 16))
                h = wrap(h * (2246822519 + 1315423911 * s))
                h = wrap(h ^ (h >> 13))
                h = wrap(h * (3266489917 + 374761393 * s))
                h = wrap(h ^ (h >> 16))
                assert got[i] == h % bins


def test_host_batch_guard_cpu_behaviour():
    # the C++ steady-state helper is built with the library; on CPU tensors it
    # refuses the fast path, and bump() advances every state["step"]
    import ctypes

    hb = _native.host_batch()
    assert hb is not None, "cresso_amd/_hostbatch extension not built"
    ps = [torch.nn.Parameter(torch.zeros(4, 4)) for _ in range(3)]
    for p in ps:
        p.grad = torch.zeros(4, 4)
    guard = hb.BatchGuard(ps)
    buf = (ctypes.c_void_p * 3)()
    assert guard.gather(ps, ctypes.addressof(buf)) is False      # CPU grads: no fast path
    assert guard.gather(ps[:2], ctypes.addressof(buf)) is False  # different group
    states = [{"step": 0}, {"step": 7}, {"step": 2}]
    guard.bump(states)
    assert [s["step"] for s in states] == [1, 8, 3]
    ps[0].grad = None
    with pytest.raises(ValueError):
        hb.BatchGuard(ps)


def test_host_batch_guard_holds_references_and_refuses_replaced_params():
    # The guard keeps each planned parameter alive (so no new object can take
    # its address) and refuses the fast path once a parameter object is replaced.
    import ctypes
    import gc
    import weakref

    hb = _native.host_batch()
    assert hb is not None, "cresso_amd/_hostbatch extension not built"
    ps = [torch.nn.Parameter(torch.zeros(4, 4)) for _ in range(3)]
    for p in ps:
        p.grad = torch.zeros(4, 4)
    guard = hb.BatchGuard(ps)
    ref = weakref.ref(ps[1])
    old = ps[1]
    ps[1] = torch.nn.Parameter(torch.zeros(4, 4))
    ps[1].grad = torch.zeros(4, 4)
    del old
    gc.collect()
    assert ref() is not None          # still referenced by the guard
    buf = (ctypes.c_void_p * 3)()
    assert guard.gather(ps, ctypes.addressof(buf)) is False
    del guard
    gc.collect()
    assert ref() is None              # released with the guard


def test_host_batch_guard_compares_layouts_and_states():
    # what a scalar plan holds the addresses of: each change, seen; undone, accepted again
    hb = _native.host_batch()
    assert hb is not None, "cresso_amd/_hostbatch extension not built"
    ps = [torch.nn.Parameter(torch.zeros(4, 4)) for _ in range(3)]
    keys = [("q", "impulse")] * 2 + [("field",)]
    state = {}
    for p, ks in zip(ps, keys):
        p.grad = torch.zeros(4, 4)
        state[p] = dict(step=5, other="kept", **{k: torch.zeros(4, 4) if k == "field" else torch.zeros(()) for k in ks})
    pair = torch.zeros(2)
    state[ps[1]].update(q=pair[0], impulse=pair[1])   # views of one buffer
    states = [state[p] for p in ps]
    guard = hb.BatchGuard(ps, states, keys)
    assert guard.holds(ps, state) and guard.holds(ps, state)

    def seen(change, undo):
        change()
        assert not guard.holds(ps, state)
        undo()
        assert guard.holds(ps, state)

    data = ps[0].data
    for other in (data.t(), data.view(2, 8), data.clone()):
        seen(lambda: setattr(ps[0], "data", other), lambda: setattr(ps[0], "data", data))
    q = states[0]["q"]
    seen(lambda: states[0].update(q=q.clone()), lambda: states[0].update(q=q))
    kept = q.data
    seen(lambda: setattr(q, "data", torch.ones(())), lambda: setattr(q, "data", kept))
    view = states[1]["q"]
    seen(lambda: setattr(view, "data", pair[1]), lambda: setattr(view, "data", pair[0]))
    field = states[2]["field"].data
    seen(lambda: setattr(states[2]["field"], "data", field.t()), lambda: setattr(states[2]["field"], "data", field))
    seen(lambda: setattr(states[2]["field"], "data", field[:2]), lambda: setattr(states[2]["field"], "data", field))
    seen(lambda: states[1].update(step=4), lambda: states[1].update(step=5))
    seen(lambda: state.update({ps[2]: dict(states[2])}), lambda: state.update({ps[2]: states[2]}))
    guard.bump(states)
    assert [s["step"] for s in states] == [6, 6, 6] and guard.holds(ps, state)
    states[0]["step"] = 5
    assert not guard.holds(ps, state)
    guard.bump(states)   # (a count that was changed is not taken for the plan's after the next step either)
    assert not guard.holds(ps, state)
    states[0]["step"] = 7
    assert guard.holds(ps, state)
    states[0]["other"] = 1   # (no entry of the plan's)
    assert guard.holds(ps, state)
    del states[0]["q"]
    assert not guard.holds(ps, state)
    with pytest.raises(ValueError):
        hb.BatchGuard(ps, states, [("q", "missing")] * 3)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16, torch.float16])
def test_scalar_descriptors_are_the_same_from_cpp_and_python(dtype, monkeypatch):
    import ctypes

    from cresso_amd.optimizer import _MICRO_KEYS, _SCALAR_KEYS, _ScalarBatch

    opt = CRESSO5([torch.nn.Parameter(torch.zeros(1))], micro_field_max_size=20)
    ps = [torch.nn.Parameter(torch.zeros(s, dtype=dtype)) for s in ((), (7,), (3, 5), (40, 2, 3), (1,) * 8)]
    micro = [False, True, True, False, False]
    keys = [_MICRO_KEYS if m else _SCALAR_KEYS for m in micro]
    sts = [opt._init_micro(p) if m else opt._init_scalar(p) for p, m in zip(ps, micro)]
    for i, st in enumerate(sts):
        st["step"] = i
    gs = [torch.zeros_like(p) for p in ps]
    out = (_native.ScalarDesc * 5)()
    assert _native.host_batch().scalar_descs(ps, gs, sts, keys, [3 if m else 0 for m in micro], ctypes.addressof(out))
    fast = bytes(_ScalarBatch.descriptors_of(ps, gs, sts, keys))
    monkeypatch.setattr(_native, "host_batch", lambda: None)
    assert fast == bytes(_ScalarBatch.descriptors_of(ps, gs, sts, keys))
    monkeypatch.undo()
    sts[1]["micro_impulse"] = sts[1]["micro_impulse"].view(7, 1)
    with pytest.raises(RuntimeError, match="micro_impulse"):
        _ScalarBatch.descriptors_of(ps, gs, sts, keys)
    sts[0]["q"] = torch.zeros(2)
    with pytest.raises(RuntimeError, match="state 'q'"):
        _ScalarBatch.descriptors_of(ps, gs, sts, keys)


def test_spectral_lane_assignment():
    # the multi-tensor spectral step: m tensors of one shape use min(4, m)
    # distinct lanes (one workspace each), shapes spread over the lanes
    from cresso_amd.spectral import assign_lanes

    keys = ["a"] * 6 + ["b"] + ["c"] * 2 + ["d"]
    lanes = assign_lanes(keys, 4)
    assert len(lanes) == len(keys) and all(0 <= x < 4 for x in lanes)
    by = {}
    for k, x in zip(keys, lanes):
        by.setdefault(k, []).append(x)
    assert len(set(by["a"])) == 4 and len(set(by["c"])) == 2
    assert by["a"][:4] == [0, 1, 2, 3] and by["a"][4:] == [0, 1]   # round robin
    assert by["b"] == [1] and by["c"] == [2, 3] and by["d"] == [3]  # start lane moves with each new key
    assert assign_lanes(["x", "y"], 1) == [0, 0]
    assert assign_lanes([], 4) == []


def test_spectral_batch_units_and_chunks():
    # the multi-tensor spectral step's units: same plan, dtypes, hard channel
    # and hash state batch together; a batch holds at most BATCH_BYTES of
    # per-tensor scratch, larger groups are cut into near-equal chunks
    from cresso_amd import _native
    from cresso_amd.spectral import SpectralEngine, lane_scratch_bytes

    eng = SpectralEngine.__new__(SpectralEngine)   # no library needed for the grouping
    eng.BATCH, eng.BATCH_BYTES = True, 3 * lane_scratch_bytes(100)

    def desc(numel, hard=1, hash_on=True, pdt=_native.F32):
        d = _native.SpectralDesc()
        d.numel, d.hard, d.param_dtype, d.grad_dtype = numel, hard, pdt, pdt
        d.hash_energy = 4096 if hash_on else None
        return d

    prepared = [("a", 8, desc(100)) for _ in range(7)] + [("b", 8, desc(50))] + [("a", 8, desc(100, hard=0))] \
        + [("a", 8, desc(100, pdt=_native.BF16))] + [("c", 8, desc(10)), ("c", 8, desc(10, hash_on=False))]
    sts = [{"i": i} for i in range(len(prepared))]
    units = eng._units(prepared, sts)
    got = [(u[0], [s["i"] for s in u[4]]) for u in units]
    # seven "a" tensors at three per batch: chunks of 3, 3, 1 (ceil(7 / ceil(7/3)) = 3)
    assert got[:3] == [(("a", True, 3), [0, 1, 2]), (("a", True, 3), [3, 4, 5]), (("a", True, 3), [6])]
    assert [g[1] for g in got[3:]] == [[7], [8], [9], [10], [11]]
    assert all(not u[0][1] for u in units[3:])
    eng.BATCH = False
    assert [len(u[4]) for u in eng._units(prepared, sts)] == [1] * len(prepared)


def test_steady_step_holds_no_dropped_workspace():
    # SpectralEngine.reset() frees every workspace; a steady step that was made
    # before must neither keep one alive nor run with it (stand-ins for the
    # workspaces: nothing is launched)
    import gc
    import types
    import weakref

    from cresso_amd.spectral import SpectralEngine, SteadyStep

    if not (ROOT / "cresso_amd" / "libcresso_hip.so").exists():
        pytest.skip("library not built")

    class Workspace:
        def __init__(self):
            self.plan, self.buf, self.count = types.SimpleNamespace(value=8), torch.zeros(16), None

    ps = [torch.nn.Parameter(torch.zeros(64, 48)), torch.nn.Parameter(torch.zeros(32, 40))]
    opt = CRESSO5(ps, cuda_ops="required", rank=8, hash_bins=64, hash_tables=2)
    group = opt.param_groups[0]
    eng = SpectralEngine()
    items = []
    for lane, p in enumerate(ps):
        p.grad = torch.zeros_like(p)
        st = opt._init_spectral(p, group)
        items.append((p, p.grad, st))
        eng.ws[(eng.plan_key(p, st, group), False, lane)] = Workspace()
    step = SteadyStep(eng, items, group, _native.host_batch())
    refs = [weakref.ref(w) for w in eng.ws.values()]
    assert step.ready()
    eng.reset()
    gc.collect()
    assert not step.ready() and not step.fill(opt.state)
    assert all(r() is None for r in refs)


def _plan(shape, rank, bins, tables):
    """(panel rows, panel rows of the general sweeps, workspace bytes) of an fp32 plan (no GPU needed)."""
    import ctypes

    from cresso_amd.modes import freqs_tensor

    lib = _native.load()
    fr = freqs_tensor(rank, len(shape), 5, "cpu").reshape(-1).tolist()
    plan = lib.cresso_spectral_plan_create_ex((ctypes.c_int64 * 8)(*shape), len(shape), (ctypes.c_int64 * len(fr))(*fr),
                                              rank, bins, tables, _native.F32)
    assert plan
    plan = ctypes.c_void_p(plan)
    got = (int(lib.cresso_spectral_plan_panel_rows(plan, 0)), int(lib.cresso_spectral_plan_panel_rows(plan, 1)),
           int(lib.cresso_spectral_workspace_bytes(plan)))
    lib.cresso_spectral_plan_destroy(plan)
    return got


PANELS = [
    # shape, rank, bins, tables, matrix-core (or only) sweeps' rows, general sweeps' rows
    # ranks above 16: 32 rows from 512 blocks on
    ((512, 512), 24, 64, 2, 16, 16), ((1024, 2048), 24, 64, 2, 16, 16), ((3072, 768), 24, 64, 2, 32, 32),
    ((2048, 2048), 24, 256, 4, 32, 32), ((2500, 1100), 20, 64, 2, 32, 32), ((8192, 4096), 32, 64, 2, 32, 32),
    # matrix-core plans: 16, 32 and 64 rows; the general sweeps as tall where
    # the rows tile by 32, else multiples of 8 with at most 1024 blocks
    ((512, 512), 8, 64, 2, 16, 16), ((10, 500), 8, 64, 2, 10, 10), ((1536, 2048), 8, 64, 2, 32, 32),
    ((2500, 1100), 8, 64, 2, 32, 16), ((2048, 2048), 8, 64, 2, 64, 64), ((6000, 1000), 8, 64, 2, 64, 24),
    ((9000, 700), 8, 64, 2, 64, 32), ((2500, 1100), 16, 256, 4, 64, 16), ((50257, 768), 8, 64, 2, 64, 64),
    # one or three tables, two-byte bins, too few columns: the general sweeps only
    ((2048, 2048), 8, 64, 3, 16, 16), ((2048, 2048), 8, 512, 2, 16, 16), ((30000, 60), 8, 64, 2, 32, 32), ((6000, 1000), 8, 64, 3, 24, 24),
]


@pytest.mark.parametrize("shape,rank,bins,tables,rows,general", PANELS, ids=[f"{c[0]}_r{c[1]}_t{c[3]}" for c in PANELS])
def test_spectral_plan_panels(shape, rank, bins, tables, rows, general):
    if not (ROOT / "cresso_amd" / "libcresso_hip.so").exists():
        pytest.skip("library not built")
    assert _plan(shape, rank, bins, tables)[:2] == (rows, general)


@pytest.mark.parametrize("shape,rank,bins,tables", [((704, 5824), 4, 128, 3), ((960, 5632), 4, 512, 1)])
def test_plans_near_the_noalloc_limit_fit_it_with_taller_panels(shape, rank, bins, tables):
    # rows that tile by 32: fewer blocks' partial sums where the workspace would
    # not fit the no-alloc entry's 32 MiB otherwise; ordinary panels well below it
    if not (ROOT / "cresso_amd" / "libcresso_hip.so").exists():
        pytest.skip("library not built")
    rows, general, nbytes = _plan(shape, rank, bins, tables)
    assert nbytes <= 32 << 20 and rows == general == 64
    half = (shape[0] // 2,) + shape[1:]
    assert _plan(half, rank, bins, tables)[0] == 16


def test_ragged_plan_near_the_noalloc_limit_fits_it_with_one_panel_height():
    # the general sweeps then take the matrix-core sweeps' panels
    if not (ROOT / "cresso_amd" / "libcresso_hip.so").exists():
        pytest.skip("library not built")
    rows, general, nbytes = _plan((997, 3775), 16, 128, 4)
    assert nbytes <= 32 << 20 and rows == general == 64
    assert _plan((797, 3775), 16, 128, 4)[:2] == (64, 16)


def test_spectral_batches_stay_within_their_scratch():
    # (640,4096) at four tables of 256 bins: 16-row panels, whose histogram
    # partials take half as much as the tangent field again
    if not (ROOT / "cresso_amd" / "libcresso_hip.so").exists():
        pytest.skip("library not built")
    import ctypes

    from cresso_amd.spectral import SpectralEngine

    shape = (640, 4096)
    ps = [torch.nn.Parameter(torch.zeros(shape)) for _ in range(8)]
    opt = CRESSO5(ps, cuda_ops="required", rank=16, max_frequency=7, hash_bins=256, hash_tables=4)
    group, eng = opt.param_groups[0], SpectralEngine()
    eng.BATCH_BYTES = 40 << 20
    sts = [opt._init_spectral(p, group) for p in ps]
    prepared = [eng._prepare(p, p.data, st, group) for p, st in zip(ps, sts)]
    units = eng._units(prepared, sts)
    fr = sts[0]["freqs"].reshape(-1).tolist()
    plan = eng.lib.cresso_spectral_plan_create_ex((ctypes.c_int64 * 8)(*shape), 2, (ctypes.c_int64 * len(fr))(*fr), 16,
                                                  256, 4, _native.F32)
    plan = ctypes.c_void_p(plan)
    size = [int(eng.lib.cresso_spectral_batched_workspace_bytes(plan, k)) for k in (1, 2)]
    eng.lib.cresso_spectral_plan_destroy(plan)
    assert sum(len(u[4]) for u in units) == 8 and len(units) > 1
    assert max(len(u[4]) for u in units) * (size[1] - size[0]) <= eng.BATCH_BYTES


@pytest.mark.parametrize("fails", ["begin", "step", "between", "end", "step and end"])
def test_spectral_launch_joins_its_streams_after_an_error(fails, monkeypatch):
    # whatever fails in a step on side streams, every stream that was forked
    # joins the caller's again, and the first error is the one raised (a
    # recording stand-in for the library: nothing is launched)
    import ctypes
    import types

    from cresso_amd import spectral

    calls, handles = [], (ctypes.c_void_p * 2)(16, 32)

    def op(name):
        def call(first, *args):
            dev = int(first) if not hasattr(first, "_length_") else len(calls)
            calls.append((name, dev if name != "step" else -1))
            return -1 if name in fails.split(" and ") else 0
        return call

    lib = types.SimpleNamespace(cresso_fork_begin=op("begin"), cresso_fork_end=op("end"),
                                cresso_spectral_step_units=op("step"))
    forks = {"a": types.SimpleNamespace(fork=1, handles=handles), "b": types.SimpleNamespace(fork=2, handles=handles)}
    engine = types.SimpleNamespace(lib=lib, _fork=lambda device, lanes: forks[device])
    launch = spectral.Launch.__new__(spectral.Launch)
    launch.engine, launch.keep = engine, []
    launch.devices = [(d, (_native.SpectralUnit * 1)(), 1, 2) for d in ("a", "b")]
    monkeypatch.setattr(_native, "stream_handle", lambda device: 64)

    def check(rc, what):
        if rc:
            raise RuntimeError(f"{what} {calls[-1][0]}")

    monkeypatch.setattr(_native, "check", check)

    def between():
        calls.append(("between", -1))
        if fails == "between":
            raise RuntimeError("between")

    with pytest.raises(RuntimeError, match=fails.split(" and ")[0]):
        launch.run(_native.Hyper(), between)
    begun = [d for name, d in calls if name == "begin"]
    assert begun and [d for name, d in calls if name == "end"] == begun


def test_load_state_dict_keeps_same_plan_workspaces():
    """A spectral workspace depends only on its plan key (shape, freqs,
    hash_bins, hash_tables, work dtype): load_state_dict keeps those the
    loaded state still uses and frees the rest (no GPU needed: the workspaces
    here are stand-in objects in the engine's table)."""
    lib_path = ROOT / "cresso_amd" / "libcresso_hip.so"
    if not lib_path.exists():
        pytest.skip("library not built")
    from cresso_amd.spectral import SpectralEngine

    p = torch.nn.Parameter(torch.zeros(64, 48))
    q = torch.nn.Parameter(torch.zeros(32, 40))
    opt = CRESSO5([p, q], cuda_ops="required", rank=8, hash_bins=64, hash_tables=2)
    group = opt.param_groups[0]
    for t in (p, q):
        opt.state[t] = opt._init_spectral(t, group)
    eng = SpectralEngine()
    opt._spectral_engine = eng
    kp = eng.plan_key(p, opt.state[p], group)
    kq = eng.plan_key(q, opt.state[q], group)
    stale = (kp[0], (7, 7)) + kp[2:]
    keep_p, keep_q, drop = object(), object(), object()
    eng.ws = {(kp, False, 0): keep_p, (kq, True, 2): keep_q, (stale, False, 1): drop}
    sd = opt.state_dict()
    opt.load_state_dict(sd)
    assert eng.ws == {(kp, False, 0): keep_p, (kq, True, 2): keep_q}
    # a loaded state with other freqs for p no longer uses p's plan
    sd2 = opt.state_dict()
    sd2["state"][0]["freqs"] = sd2["state"][0]["freqs"].flip(0).clone()
    opt.load_state_dict(sd2)
    assert set(eng.ws) == {(kq, True, 2)}


def test_spectral_plan_rank_limits_without_gpu():
    # plan creation is host work: ranks up to 32 plan on the fp32 and fp64
    # work dtypes (ranks above 16 take the general sweeps); a refusal carries
    # the library's message instead of a fallback
    lib_path = ROOT / "cresso_amd" / "libcresso_hip.so"
    if not lib_path.exists():
        pytest.skip("library not built")
    from cresso_amd.modes import mode_list

    lib = _native.load()
    shape = (1024, 512)

    def create(rank, work):
        freqs = [f for m in mode_list(rank, 2, 7) for f in m]
        return lib.cresso_spectral_plan_create_ex((ctypes.c_int64 * 8)(*shape), 2,
                                                  (ctypes.c_int64 * len(freqs))(*freqs), rank, 64, 2, work)

    for rank in (17, 24, 32):
        plan = create(rank, _native.F32)
        assert plan, lib.cresso_hip_last_error()
        assert lib.cresso_spectral_workspace_bytes(ctypes.c_void_p(plan)) > 0
        lib.cresso_spectral_plan_destroy(ctypes.c_void_p(plan))
    plan = create(24, _native.F64)
    assert plan, lib.cresso_hip_last_error()
    lib.cresso_spectral_plan_destroy(ctypes.c_void_p(plan))
    assert not create(33, _native.F32)
    assert b"rank 33" in lib.cresso_hip_last_error()
