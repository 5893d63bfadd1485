"""Steps of mixed groups after the second, which the C++ guards take when
nothing has changed: the same results as an optimizer whose every step goes
the general way, over changes that must send a step back there."""

import pytest
import torch

from gpu_util import announce, needs_gpu

pytestmark = [pytest.mark.gpu, needs_gpu]

SHAPES = [(256, 300), (64, 65), (64, 65), (4096, 16), (1500,), (10,), (24, 6, 3, 3)]


def _pair(shapes, **kw):
    import cresso_amd

    gen = torch.Generator().manual_seed(51)
    p0 = [0.02 * torch.randn(s, generator=gen) for s in shapes]
    out = []
    for _ in range(2):
        ps = [torch.nn.Parameter(p.cuda()) for p in p0]
        out.append((ps, cresso_amd.CRESSO5(ps, cuda_ops="required", rank=8, hash_bins=64, hash_tables=2, **kw)))
    return gen, out


def _steps(gen, pair, n, change=None):
    for k in range(n):
        grads = [1e-3 * torch.randn(p.shape, generator=gen) for p in pair[0][0]]
        for i, (ps, opt) in enumerate(pair):
            for p, g in zip(ps, grads):
                p.grad = g.cuda()
            if change is not None:
                change(k, ps, opt)
            if i == 1:
                opt._steady.clear()   # the general way
            opt.step()
    torch.cuda.synchronize()
    (pa, oa), (pb, ob) = pair
    for a, b in zip(pa, pb):
        assert torch.equal(a, b)
        for key, v in oa.state[a].items():
            w = ob.state[b][key]
            assert torch.equal(v, w) if torch.is_tensor(v) else v == w, key


@pytest.mark.parametrize("shapes", [SHAPES, SHAPES[:1], SHAPES[1:3]], ids=["mixed", "one", "batch"])
def test_steady_steps_are_the_general_steps(shapes):
    announce(f"steady steps {len(shapes)}")
    gen, pair = _pair(shapes)
    _steps(gen, pair, 6)
    assert pair[0][1]._steady[0][2] is not None   # the steady step was made


def test_steady_steps_follow_changes():
    """A skipped grad, other layouts and dtypes of grads, new parameter storage, replaced state tensors, another
    step count, group options and learning rate."""
    announce("steady steps with changes")
    gen, pair = _pair(SHAPES)

    def change(k, ps, opt):
        if k == 3:
            ps[1].grad = None
        if k == 5:
            ps[0].grad = ps[0].grad.t().contiguous().t()
        if k == 7:
            ps[2].data = ps[2].data.clone()
        if k == 9:
            st = opt.state[ps[0]]
            st["q_cos"] = st["q_cos"].clone() * 0.5
            st["step"] = 3
        if k == 10:
            opt.param_groups[0]["lr"] = 1e-3
        if k == 12:
            opt.param_groups[0]["weight_decay"] = 0.01
        if k == 14:
            opt.load_state_dict(opt.state_dict())
        if k == 16:
            with torch.no_grad():
                ps[5].zero_()

    _steps(gen, pair, 19, change)


def test_steady_step_refuses_what_the_general_step_refuses():
    gen, pair = _pair(SHAPES)
    _steps(gen, pair, 4)
    ps, opt = pair[0]
    for p in ps:
        p.grad = torch.zeros_like(p)
    ps[1].grad = torch.zeros_like(ps[1]).to_sparse()
    with pytest.raises(RuntimeError, match="sparse"):
        opt.step()
    ps[1].grad = torch.zeros_like(ps[1])
    opt.state[ps[0]]["hash_energy"] = opt.state[ps[0]]["hash_energy"].t().contiguous()
    with pytest.raises(RuntimeError, match="shape"):
        opt.step()


MICRO = dict(micro_field_max_size=64)
SCALARS = [(4096, 16), (900,), (16, 64), (10,), (6, 8)]   # the last two: micro fields with MICRO
GROUPS = {"mixed": SCALARS + [(64, 65)], "scalar": SCALARS}
KEPT = []   # replaced storage stays alive: a step that still used it would write to live memory


def _layout(ps, opt):
    ps[0].data = ps[0].data.t()   # same storage, other element order


def _reshape(ps, opt):
    ps[2].data = ps[2].data.view(64, 16)


def _state_entry(ps, opt):
    st = opt.state[ps[0]]
    KEPT.append(st["q"])
    st["q"] = 0.5 * st["q"]


def _state_storage(ps, opt):
    st = opt.state[ps[1]]
    KEPT.append(st["impulse"].data)
    st["impulse"].data = 0.5 * st["impulse"].data


def _state_dict(ps, opt):
    KEPT.append(opt.state[ps[1]])
    opt.state[ps[1]] = {k: 0.5 * v if torch.is_tensor(v) else v for k, v in opt.state[ps[1]].items()}


def _micro_field(ps, opt):
    st = opt.state[ps[4]]
    KEPT.append(st["micro_energy"])
    st["micro_energy"] = 0.5 * st["micro_energy"]


def _step_count(ps, opt):
    opt.state[ps[0]]["step"] = 1
    opt.state[ps[4]]["step"] = 0


CHANGES = [_layout, _reshape, _state_entry, _state_storage, _state_dict, _micro_field, _step_count]


@pytest.mark.parametrize("group", sorted(GROUPS))
@pytest.mark.parametrize("change", CHANGES, ids=[c.__name__[1:] for c in CHANGES])
def test_planned_scalar_tensors_follow_changes(group, change):
    """A change to a scalar or micro tensor's layout, shape, state or step count after steady steps, against an
    optimizer that plans every step anew: the same bits."""
    announce(f"{group} group, {change.__name__[1:]} changed")
    gen, pair = _pair(GROUPS[group], **MICRO)

    def at(k, ps, opt):
        if k == 4:
            change(ps, opt)
            for p in ps:
                p.grad = 1e-3 * torch.arange(p.numel(), device="cuda", dtype=torch.float32).view(p.shape)
        if opt is pair[1][1]:
            opt._batches.clear()

    _steps(gen, pair, 7, at)
    KEPT.clear()


@pytest.mark.parametrize("group", sorted(GROUPS))
def test_planned_scalar_tensors_follow_changes_without_the_helper(group, monkeypatch):
    """All of these changes, one after the other, where the C++ helper is not built."""
    from cresso_amd import _native

    announce(f"{group} group, no helper")
    monkeypatch.setattr(_native, "host_batch", lambda: None)
    gen, pair = _pair(GROUPS[group], **MICRO)
    changes = {2 + 2 * i: c for i, c in enumerate(CHANGES)}

    def at(k, ps, opt):
        if k in changes:
            changes[k](ps, opt)
            for p in ps:
                p.grad = 1e-3 * torch.arange(p.numel(), device="cuda", dtype=torch.float32).view(p.shape)
        if opt is pair[1][1]:
            opt._batches.clear()

    _steps(gen, pair, 2 * len(changes) + 3, at)
    KEPT.clear()


def _no_q(ps, opt):
    del opt.state[ps[0]]["q"]


def _wide_q(ps, opt):
    opt.state[ps[0]]["q"] = opt.state[ps[0]]["q"].double()


def _host_impulse(ps, opt):
    opt.state[ps[0]]["impulse"] = opt.state[ps[0]]["impulse"].cpu()


def _long_action(ps, opt):
    opt.state[ps[1]]["action"] = torch.zeros(2, device="cuda")


def _flat_field(ps, opt):
    opt.state[ps[4]]["micro_energy"] = opt.state[ps[4]]["micro_energy"].view(-1)


REFUSED = [_no_q, _wide_q, _host_impulse, _long_action, _flat_field]


@pytest.mark.parametrize("group", sorted(GROUPS))
@pytest.mark.parametrize("change", REFUSED, ids=[c.__name__[1:] for c in REFUSED])
def test_planned_scalar_tensors_refuse_bad_states(group, change):
    """A scalar or micro state that no plan can be made of is refused on a steady step too."""
    gen, pair = _pair(GROUPS[group], **MICRO)
    _steps(gen, pair, 4)
    ps, opt = pair[0]
    for p in ps:
        p.grad = torch.zeros_like(p)
    before = [p.detach().clone() for p in ps]
    change(ps, opt)
    with pytest.raises(RuntimeError, match="state"):
        opt.step()
    torch.cuda.synchronize()
    for i in (0, 1, 4):
        assert torch.equal(ps[i], before[i])
