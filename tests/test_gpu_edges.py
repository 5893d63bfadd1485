"""The matrix-core sweeps on tensors whose rows and columns are no multiple of
a panel (16, 32 or 64 rows) or a slab (256 columns), and with weight decay
(the force stored by the first sweep): the sizes where the last panel moves up
and the last wave moves left, in every table count and dtype form, against the
CPU oracle and, batched, against single steps bit for bit."""

import pytest
import torch

from gpu_util import BF16_PARAM_TOL, F32_TOL, announce, compare, needs_gpu, run_pair

pytestmark = [pytest.mark.gpu, needs_gpu]

KW = dict(lr=2e-3, rank=8, max_frequency=5, hash_bins=64, hash_tables=2, min_spectral_size=1, thin_matrix_max_width=0)
R16 = dict(KW, rank=16, max_frequency=7, hash_bins=256, hash_tables=4)

CASES = [
    # one row or column past a full panel or slab; one wave of columns; the smallest panel
    ("rows17_cols65", (17, 65), KW),
    ("rows16_cols64", (16, 64), KW),
    ("rows33_cols255", (33, 255), KW),
    ("rows129_cols257", (129, 257), KW),
    ("rows300_cols513", (300, 513), dict(KW, rank=4, max_frequency=3)),
    # panels of 64 rows (more than 16384 rows times slabs) and of 32, ragged both ways
    ("panel64", (8200, 520), KW),
    ("panel32", (2500, 1100), KW),
    # one row or column short of the path (the general sweeps)
    ("rows15_cols64", (15, 64), KW),
    ("rows64_cols63", (64, 63), KW),
    ("r16_t4", (100, 333), R16),
    ("conv4d", (48, 20, 3, 3), KW),
    ("grid3d", (19, 23, 29), dict(KW, rank=16)),
    ("decay", (256, 512), dict(KW, weight_decay=0.02)),
    ("decay_ragged_maximize", (211, 301), dict(KW, weight_decay=0.02, maximize=True)),
    ("ragged_maximize", (211, 301), dict(KW, maximize=True)),
    ("decay_r16_t4", (130, 700), dict(R16, weight_decay=0.02)),
]


@pytest.mark.parametrize("name,shape,kw", CASES, ids=[c[0] for c in CASES])
def test_edges_match_oracle(name, shape, kw):
    announce(f"edges {name} {shape}")
    compare(*run_pair([shape], torch.float32, kw, steps=3, seed=31, grad_std=1e-3, param_std=0.02))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("decay", [0.0, 0.01], ids=["plain", "decay"])
def test_edges_half_dtypes_first_step(dtype, decay):
    # one step: with weight decay the force then depends on identical params on both sides
    announce(f"edges {dtype} weight decay {decay}")
    kw = dict(KW, weight_decay=decay)
    res = run_pair([(77, 331), (64, 1026)], dtype, kw, steps=1, seed=32, grad_std=0.05, param_std=0.05)
    compare(*res, param_tol=BF16_PARAM_TOL, state_tol=F32_TOL)


@pytest.mark.parametrize("shape,kw", [((77, 331), KW), ((513, 300), dict(KW, weight_decay=0.02)), ((40, 130), R16)],
                         ids=["ragged", "decay", "r16_t4"])
def test_edges_batched_steps_are_bit_identical(shape, kw):
    """Four same-shape tensors in one batch against each alone."""
    import cresso_amd

    announce(f"edges batched {shape}")
    gen = torch.Generator().manual_seed(33)
    p0 = [0.02 * torch.randn(shape, generator=gen) for _ in range(4)]
    grads = [[1e-3 * torch.randn(shape, generator=gen) for _ in p0] for _ in range(3)]
    together = [torch.nn.Parameter(p.cuda()) for p in p0]
    alone = [torch.nn.Parameter(p.cuda()) for p in p0]
    opts = [cresso_amd.CRESSO5(together, cuda_ops="required", **kw)]
    opts += [cresso_amd.CRESSO5([p], cuda_ops="required", **kw) for p in alone]
    for gs in grads:
        for ps in (together, alone):
            for p, g in zip(ps, gs):
                p.grad = g.cuda()
        for opt in opts:
            opt.step()
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(together, alone)):
        assert torch.equal(a, b), i
        sa, sb = opts[0].state[a], opts[1 + i].state[b]
        for k, v in sb.items():
            assert torch.equal(sa[k], v) if torch.is_tensor(v) else sa[k] == v, (i, k)


PANELS = [
    # name, shape, options, panel rows, whether the general sweeps run
    ("full32", (1536, 2048), KW, 32, False),
    ("ragged32_decay", (2500, 1100), dict(KW, weight_decay=0.02, maximize=True), 32, False),
    ("ragged64_decay", (8200, 520), dict(KW, weight_decay=0.02), 64, False),
    ("ragged64_r16_t4", (2500, 1100), R16, 64, False),
    ("general_ragged", (6000, 1000), dict(KW, local_sharpness=0.3), 24, True),
    ("general_full32", (1536, 2048), dict(KW, instant_metric_power=0.7), 32, True),
    ("rank24_32", (3072, 768), dict(KW, rank=24, max_frequency=6), 32, True),
    ("rank24_32_ragged_t4", (2500, 1100), dict(R16, rank=24), 32, True),
]


@pytest.mark.parametrize("name,shape,kw,rows,general", PANELS, ids=[c[0] for c in PANELS])
def test_panel_heights_match_oracle(name, shape, kw, rows, general):
    """Every panel height that a plan can choose, full and ragged, with the height asserted.  (The oracle adds its
    bins in fp64: in fp32, one after the other, up to 67 thousand elements a bin err by sqrt(67e3) 2^-24 = 1.5e-5.)"""
    announce(f"panels {name} {shape}")
    res = run_pair([shape], torch.float32, kw, steps=2, seed=34, grad_std=1e-3, param_std=0.02, hash_accum="fp64")
    compare(*res)
    engine = res[1]._spectral_engine
    (ws,) = engine.ws.values()
    assert engine.lib.cresso_spectral_plan_panel_rows(ws.plan, 1 if general else 0) == rows
