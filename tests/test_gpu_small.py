"""The register kernels of small tensors (scalar and micro-field routes) at the
edges of their range: one element, one past a thread's share, the largest
tensors of eight and sixteen elements a thread and the first past them, axes
whose factors just fit in LDS, every rank, against the CPU oracle."""

import pytest
import torch

from gpu_util import BF16_PARAM_TOL, F32_TOL, announce, compare, needs_gpu, run_pair

pytestmark = [pytest.mark.gpu, needs_gpu]

KW = dict(lr=2e-3, rank=4, hash_bins=64, hash_tables=2, min_spectral_size=1 << 30)
OPTIONS = dict(KW, weight_decay=0.02, maximize=True, local_sharpness=0.3, instant_metric_power=0.7, warmup_steps=0)
SHAPES = [(), (1,), (1, 1), (1, 7), (1023,), (1025,), (64, 16), (33, 31), (8, 1024), (8193,), (16384,), (4, 4096),
          (16385,), (5, 3276), (1, 4095), (1, 4096), (2, 8192), (16, 2000), (16, 2048), (2048, 16),
          (32768,), (32769,), (40, 700), (7, 40, 100), (3, 5, 7), (2, 4, 1000), (16, 8, 3, 3), (2, 3, 2, 5, 3)]


@pytest.mark.parametrize("kw", [KW, OPTIONS, dict(KW, instant_metric_coupling=0.0)], ids=["plain", "options", "no_axes"])
def test_small_scalar_tensors_match_oracle(kw):
    announce(f"small scalar tensors {sorted(set(kw) - set(KW))}")
    compare(*run_pair(SHAPES, torch.float32, kw, steps=3, seed=41))


@pytest.mark.parametrize("kw", [KW, dict(KW, weight_decay=0.02, maximize=True, instant_metric_power=0.7, energy_power=1.0)],
                         ids=["plain", "options"])
def test_small_micro_tensors_match_oracle(kw):
    announce("small micro tensors")
    shapes = [s for s in SHAPES if s != ()]
    compare(*run_pair(shapes, torch.float32, dict(kw, micro_field_max_size=20000), steps=3, seed=42))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("micro", [0, 20000], ids=["scalar", "micro"])
def test_small_half_dtypes_first_step(dtype, micro):
    announce(f"small {dtype} micro {micro}")
    res = run_pair([(1,), (1025,), (33, 31), (4, 4096), (3, 5, 7)], dtype, dict(KW, micro_field_max_size=micro), steps=1,
                   seed=43, grad_std=0.05, param_std=0.05)
    compare(*res, param_tol=BF16_PARAM_TOL, state_tol=F32_TOL)


@pytest.mark.parametrize("kw", [KW, OPTIONS, dict(KW, instant_metric_coupling=0.0)], ids=["plain", "options", "no_axes"])
@pytest.mark.parametrize("extra", [[], [(2048, 16)]], ids=["wide", "middle"])
def test_middle_tensors_beside_wide_ones_match_oracle(kw, extra):
    """Tensors of 16 to 32 Ki elements in a plan that has larger ones: in the wide form's launches, or, beside a
    resident tensor of their size, in the middle kernel's."""
    announce(f"middle tensors, {len(extra)} resident, {sorted(set(kw) - set(KW))}")
    shapes = [(16385,), (40, 700), (7, 40, 100), (32768,), (33, 734), (2, 3, 5000), (300, 257), (65537,)] + extra
    compare(*run_pair(shapes, torch.float32, kw, steps=3, seed=45))


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_small_tensor_with_a_bad_gradient_has_no_number_left(bad):
    """One NaN or infinite gradient element: the reservoirs and every updated value become NaN, as in the reference."""
    import cresso_amd

    p = torch.nn.Parameter(0.02 * torch.randn(40, 50, device="cuda"))
    p.grad = 1e-3 * torch.randn_like(p)
    p.grad[3, 7] = bad
    opt = cresso_amd.CRESSO5([p], cuda_ops="required", **KW)
    opt.step()
    torch.cuda.synchronize()
    assert not torch.isfinite(opt.state[p]["force_rms"])
    assert not torch.isfinite(p).any()


@pytest.mark.parametrize("shape", [(4096, 16), (16, 4096), (2048, 16), (768, 8)])
def test_scalar_step_beside_another_streams_work_is_bit_identical(shape):
    """The one-workgroup kernels beside spectral steps on another stream, whose blocks hold some of a workgroup's waves
    up for microseconds, against the same steps on an idle GPU: no wave may read a state value that another has
    already written back."""
    import cresso_amd

    announce(f"scalar {shape} beside a side stream")
    kw = dict(rank=8, hash_bins=64, hash_tables=2, cuda_ops="required")
    gen = torch.Generator().manual_seed(44)
    p0 = [0.02 * torch.randn(shape, generator=gen) for _ in range(4)]
    grads = [[(1e-3 * torch.randn(shape, generator=gen)).cuda() for _ in p0] for _ in range(4)]
    quiet = [torch.nn.Parameter(p.cuda()) for p in p0]
    busy = [torch.nn.Parameter(p.cuda()) for p in p0]
    opts = [cresso_amd.CRESSO5(quiet, **kw), cresso_amd.CRESSO5(busy, **kw)]
    other = torch.nn.Parameter(0.02 * torch.randn(256, 512, device="cuda"))
    other.grad = 1e-3 * torch.randn_like(other)
    load = cresso_amd.CRESSO5([other], **kw)
    side = torch.cuda.Stream()
    for k in range(60):
        for ps in (quiet, busy):
            for p, g in zip(ps, grads[k % 4]):
                p.grad = g
        opts[0].step()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            for _ in range(3):
                load.step()
        opts[1].step()
        torch.cuda.synchronize()
        for a, b in zip(quiet, busy):
            assert torch.equal(a, b), k
