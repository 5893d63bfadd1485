"""Optimizer steps that users of CRESSO5 run, as timing cases.

One pass is one `CRESSO5.step()` over the parameters of one program, with the
gradients in place, from a state in mid-training (as after a resume).  The
parameters and gradients are views of one flat buffer each, and so is every
kind of state (one row per tensor), as programs keep them that checkpoint or
exchange them in one piece; a pass returns these buffers whole.

Families (what a case's "set" stands for):
  lora    low-rank adapters of a transformer's projections: per layer an
          (r, in) and an (out, r) matrix for each of q, k, v, o and, where
          "hidden" is set, gate, up, down.  Thin matrices: the scalar route.
  mlp     a small perceptron: weight matrices and biases, mixed routes;
          with "micro" the opt-in dense micro-field route takes its tensors.
  matrix  one weight matrix or embedding table: the spectral route.
  volume  one 3-D parameter (a learned grid).
  conv    a residual convolution network: 4-D weights, norms, the head.
  block   transformer layers trained in full (q, k, v, o, gate, up, down and
          two norm weights each), with the embedding where "vocab" is set.
"""

import math

import torch

import cresso_amd

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
DEVICE = "cuda"
LR = 2e-3
STEP = 200          # steps taken before the pass
PAD = 256           # elements: every tensor of a flat buffer starts at a multiple
THIN_WIDTH, THIN_ASPECT, MIN_SPECTRAL = 64, 4.0, 1024   # the optimizer's routing defaults

# keywords of CRESSO5 other than its defaults, per case
OPTIONS = dict(rank=8, max_frequency=5, hash_bins=128, hash_tables=2, weight_decay=0.0, micro=0)


def _case(name, set, dtype="fp32", grad=None, **kw):
    case = {"set": set, "dtype": dtype, "grad": grad or dtype, **OPTIONS, **kw}
    return dict(case, name=name) if name else case


def listed():
    return [
        # adapters of a two-layer encoder: the smallest step, 16 tensors of 6 Ki elements
        _case("lora_small", "lora", layers=2, width=768, hidden=0, r=8, rank=4, hash_bins=64),
        # 105 layers' attention adapters, 840 thin matrices: bench.py's C3
        _case("lora_840", "lora", layers=105, width=4096, hidden=0, r=16, rank=4, hash_bins=64),
        # adapters of every projection of a 22-layer transformer in bf16: widths 2048 and 5632
        _case("lora_mlp_bf16", "lora", dtype="bf16", layers=22, width=2048, hidden=5632, r=16),
        # a digit classifier with default options: spectral, thin and 1-D tensors in one group
        _case("mlp_small", "mlp", inputs=784, width=256, layers=3, classes=10),
        # a small coordinate network on the micro-field route
        _case("micro_net", "mlp", inputs=32, width=64, layers=9, classes=3, micro=4096),
        # one attention-sized matrix: C1's shape and options
        _case("matrix_2048", "matrix", rows=2048, cols=2048, hash_bins=64),
        # one large fp32 matrix: C2, bench.py's default workload
        _case("matrix_4096", "matrix", rows=4096, cols=4096, hash_bins=64),
        # one very large bf16 matrix at rank 16 with four tables: C5's main tensor
        _case("matrix_8192_bf16", "matrix", dtype="bf16", rows=8192, cols=8192, rank=16, max_frequency=7, hash_bins=256,
              hash_tables=4),
        # an embedding table whose vocabulary is not a round number
        _case("embedding_odd", "matrix", rows=50257, cols=768),
        # an 18-layer residual network with parameter-free shortcuts: 4-D weights of 3x3 and 7x7, norms, the head
        _case("conv_net", "conv", width=64, classes=1000),
        # full fine-tuning of two bf16 transformer layers with weight decay
        _case("block_bf16_decay", "block", dtype="bf16", layers=2, width=2048, hidden=5632, vocab=0, weight_decay=0.01),
        # the whole 1.2 B-parameter transformer: bench.py's C4
        _case("model_1b", "block", layers=22, width=2048, hidden=5632, vocab=32000, hash_bins=64),
    ]


def draw(rng):
    def log(lo, hi, step=1):
        return max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step)

    def size(lo, hi):   # half of them round, as most programs' are
        return log(lo, hi, 64 if rng.random() < 0.5 else 1)

    dtype = rng.choice(("fp32", "fp32", "bf16", "bf16", "fp16"))
    kw = dict(rank=rng.choice((4, 8, 8, 16)), hash_bins=rng.choice((64, 128, 256)),
              weight_decay=rng.choice((0.0, 0.0, 0.01, 0.1)))
    kind = rng.choice(("lora", "mlp", "matrix", "matrix", "volume", "conv", "block"))
    if kind == "lora":
        kw.update(layers=log(1, 48), width=size(256, 8192), hidden=rng.choice((0, size(1024, 16384))),
                  r=rng.choice((4, 8, 16, 32, 33, 64)))
    elif kind == "mlp":
        kw.update(inputs=size(24, 1024), width=size(64, 1024), layers=rng.randint(2, 8), classes=log(2, 100),
                  micro=rng.choice((0, 4096)))
    elif kind == "matrix":
        kw.update(rows=size(128, 16384), cols=size(128, 6144), hash_tables=rng.choice((2, 2, 4)))
        if dtype != "fp32" and rng.random() < 0.3:   # master weights in fp32, gradients in 16 bits
            return _case(None, "matrix", "fp32", dtype, **kw)
    elif kind == "volume":
        kw.update(d0=size(16, 128), d1=size(32, 512), d2=size(32, 512))
    elif kind == "conv":
        kw.update(width=rng.choice((16, 24, 32, 48, 64, 96)), classes=log(10, 1000), rank=rng.choice((4, 8)))
    else:
        kw.update(layers=rng.randint(1, 4), width=size(256, 2048), hidden=size(512, 5632), vocab=rng.choice((0, log(1000, 32000))))
    return _case(None, kind, dtype, **kw)


def _shapes(c):
    kind = c["set"]
    if kind == "lora":
        w, h, r = c["width"], c["hidden"], c["r"]
        io = [(w, w)] * 4 + ([(w, h), (w, h), (h, w)] if h else [])
        return [s for _ in range(c["layers"]) for i, o in io for s in ((r, i), (o, r))]
    if kind == "mlp":
        dims = [c["inputs"]] + [c["width"]] * (c["layers"] - 1) + [c["classes"]]
        return [s for i, o in zip(dims, dims[1:]) for s in ((o, i), (o,))]
    if kind == "matrix":
        return [(c["rows"], c["cols"])]
    if kind == "volume":
        return [(c["d0"], c["d1"], c["d2"])]
    if kind == "conv":
        w = c["width"]
        out = [(w, 3, 7, 7), (w,), (w,)]
        prev = w
        for stage in range(4):
            k = w << stage
            for block in range(2):
                out += [(k, prev, 3, 3), (k,), (k,), (k, k, 3, 3), (k,), (k,)]
                prev = k
        return out + [(c["classes"], prev), (c["classes"],)]
    w, h = c["width"], c["hidden"]
    out = [(c["vocab"], w)] if c["vocab"] else []
    return out + ([(w, w)] * 4 + [(h, w)] * 2 + [(w, h)] + [(w,)] * 2) * c["layers"]


def _route(shape, c):
    n = math.prod(shape)
    if n <= c["micro"]:
        return "micro"
    thin = len(shape) == 2 and min(shape) <= THIN_WIDTH and max(shape) / min(shape) >= THIN_ASPECT
    return "scalar" if n < MIN_SPECTRAL or thin else "spectral"


def _places(shapes):
    """Offsets of the tensors of a flat buffer, and its length."""
    at, places = 0, []
    for s in shapes:
        places.append(at)
        at += -(-math.prod(s) // PAD) * PAD
    return places, at


def _views(flat, shapes):
    return [flat[a:a + math.prod(s)].view(s) for a, s in zip(_places(shapes)[0], shapes)]


SCALARS = ("force_rms", "drive_energy", "surprise", "action")
OSCILLATOR = ("q", "impulse", "metric_q", "metric_impulse")
MODES = ("q_cos", "q_sin", "p_cos", "p_sin", "metric_cos", "metric_sin", "metric_p_cos", "metric_p_sin", "calcium_cos",
         "calcium_sin", "mode_confidence")
HASH = ("hash_energy", "hash_impulse", "hash_refractory")
MICRO = ("micro_energy", "micro_impulse", "micro_refractory")


def _inputs(c, seed):
    """(shapes, routes, flat params, flat grads, state buffers, per-tensor views of them)."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    shapes = _shapes(c)
    routes = [_route(s, c) for s in shapes]
    total = _places(shapes)[1]

    def randn(*size):
        return torch.randn(size, generator=gen, device=DEVICE)

    def rand(lo, hi, *size):
        return lo + (hi - lo) * torch.rand(size, generator=gen, device=DEVICE)

    param = (0.02 * randn(total)).to(DTYPES[c["dtype"]])
    # per-tensor scale log-uniform in [1e-4, 1e-2]; one element in a hundred is a spike
    sigma = (10.0 ** (-4.0 + 2.0 * torch.rand(len(shapes), generator=host, dtype=torch.float64))).tolist()
    grad = randn(total)
    for v, s in zip(_views(grad, shapes), sigma):
        v.mul_(s)
    spikes = torch.rand(total, generator=gen, device=DEVICE) < 0.01
    grad = torch.where(spikes, 20.0 * grad, grad).to(DTYPES[c["grad"]])
    del spikes

    count = {r: routes.count(r) for r in ("scalar", "spectral", "micro")}
    rank, tables, bins = c["rank"], c["hash_tables"], c["hash_bins"]
    rms = torch.tensor(sigma, dtype=torch.float32, device=DEVICE)
    state = {"force_rms": rms * rand(1.5, 2.5, len(shapes)), "drive_energy": rand(0.5, 1.5, len(shapes)),
             "surprise": rand(0.6, 1.4, len(shapes)), "action": 0.1 * randn(len(shapes))}
    if count["scalar"]:
        for k, m, s in zip(OSCILLATOR, (0.0, 0.0, 0.5, 0.0), (0.2, 0.1, 0.1, 0.05)):
            state[k] = m + s * randn(count["scalar"])
    if count["spectral"]:
        for k, s in zip(MODES, (0.3, 0.3, 0.1, 0.1, 0.2, 0.2, 0.1, 0.1, 0.0, 0.0, 0.3)):
            state[k] = s * randn(count["spectral"], rank) if s else rand(0.0, 0.5, count["spectral"], rank)
        state["hash_energy"] = rand(0.5, 1.5, count["spectral"], tables, bins)
        state["hash_impulse"] = 0.1 * randn(count["spectral"], tables, bins)
        state["hash_refractory"] = rand(0.0, 0.3, count["spectral"], tables, bins)
    if count["micro"]:
        n = _places([s for s, r in zip(shapes, routes) if r == "micro"])[1]
        state.update(micro_energy=rand(0.5, 1.5, n), micro_impulse=0.3 * randn(n), micro_refractory=rand(0.0, 1.0, n))
    return shapes, routes, param, grad, state, _state_views(shapes, routes, state)


def _state_views(shapes, routes, state):
    """One dict of state tensors (views of the buffers) per tensor."""
    seen = {"scalar": 0, "spectral": 0, "micro": 0}
    micro = [s for s, r in zip(shapes, routes) if r == "micro"]
    fields = {k: _views(state[k], micro) for k in MICRO if k in state}
    out = []
    for i, route in enumerate(routes):
        st = {k: state[k][i] for k in SCALARS}
        j = seen[route]
        seen[route] += 1
        if route == "scalar":
            st.update({k: state[k][j] for k in OSCILLATOR})
        elif route == "spectral":
            st.update({k: state[k][j] for k in MODES + HASH})
        else:
            st.update({k: fields[k][j] for k in MICRO})
        out.append(st)
    return out


def prepare(case, seed):
    shapes, routes, param, grad, state, views = _inputs(case, seed)
    params = [torch.nn.Parameter(v) for v in _views(param, shapes)]
    for p, g in zip(params, _views(grad, shapes)):
        if g.dtype != p.dtype:   # 16-bit gradients of fp32 weights
            p.grad_dtype = g.dtype
        p.grad = g
    opt = cresso_amd.CRESSO5(params, lr=LR, rank=case["rank"], max_frequency=case["max_frequency"],
                             hash_bins=case["hash_bins"], hash_tables=case["hash_tables"],
                             weight_decay=case["weight_decay"], micro_field_max_size=case["micro"], cuda_ops="required")
    for p, route, st in zip(params, routes, views):
        if route == "spectral":
            freqs = torch.tensor(_frequencies(case["rank"], p.ndim, case["max_frequency"]), device=DEVICE)
            st = dict(st, freqs=freqs, omega=torch.sqrt(1.0 + freqs.float().square().sum(1)))
        opt.state[p] = dict(st, step=STEP)
    return {"opt": opt, "first": params[0], "out": {"param": param, "state": state}}


def run(state):
    state["opt"].step()
    return {"step": state["opt"].state[state["first"]]["step"], **state["out"]}


def work(case):
    item = torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
    gitem = torch.empty((), dtype=DTYPES[case["grad"]]).element_size()
    total = nbytes = flops = 0
    for s in _shapes(case):
        n, route = math.prod(s), _route(s, case)
        total += n
        nbytes += (2 * item + gitem) * n
        if route == "spectral":
            # element math; two projections and two reconstructions on the modes' distinct column carriers
            flops += n * (100 + 4 * 2 * 2 * case["rank"])
            nbytes += 8 * (11 * case["rank"] + 3 * case["hash_bins"] * case["hash_tables"])
        else:
            flops += n * 80
            nbytes += 24 * n if route == "micro" else 64
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    # Measured against exact(): 32-bit values and state within 1.5e-7, the action (one sum of cancelling terms) within
    # 5e-6.  16-bit weights: an update that lands beside a rounding boundary moves a value by one unit in the last
    # place, a few values in a million.
    return {"rel": 2e-5, "max": 2e-4} if case["dtype"] == "fp32" else {"rel": 1e-4, "max": 2e-2}


# --------------------------------------------------------------------------
# the same step in 64 bits
# --------------------------------------------------------------------------
H = dict(energy_power=1.2, dt=0.15, impulse_friction=0.18, contact_gain=0.16, restoring=0.62, cubic=0.006, metric_dt=0.09,
         metric_friction=0.22, metric_coupling=0.36, instant=0.55, root=0.16, echo=0.06, transport=0.18, hash_decay=0.92,
         impulse_decay=0.78, hash_coupling=0.42, hash_mix=0.22, direct=0.18, residual=0.06, micro_decay=0.94,
         micro_impulse=0.82, micro_mix=0.35, reservoir=0.95, refractory=0.90, refractory_gain=0.55, conf_decay=0.92,
         conf_gain=0.50, surprise_gain=0.18, surprise_decay=0.95, prediction=0.16, novelty=0.04, warmup=10, brake=0.18,
         target=1.0, min_gain=0.04, max_gain=6.0, clip=4.0, spike=0.25, eps=1e-8)
EPS = H["eps"]


def _frequencies(rank, ndim, fmax):
    """The modes' integer frequencies: axes, diagonals, pairs, then a fixed sequence."""
    modes = [(0,) * ndim]
    wanted = [tuple(f if i == a else 0 for i in range(ndim)) for f in range(1, fmax + 1) for a in range(ndim)]
    for f in range(1, fmax + 1):
        wanted.append((f,) * ndim)
        if ndim > 1:
            wanted.append(tuple(f if i % 2 == 0 else max(1, fmax + 1 - f) for i in range(ndim)))
    if ndim > 1:
        for f1 in range(1, fmax + 1):
            for f2 in range(1, fmax + 1):
                for a in range(ndim):
                    v = [0] * ndim
                    v[a], v[(a + 1) % ndim] = f1, f2
                    wanted.append(tuple(v))
    for v in wanted:
        if v not in modes:
            modes.append(v)
    primes = (2, 3, 5, 7, 11, 13, 17, 19)
    tries, k = 0, 1
    while len(modes) < rank:
        v = [(k * primes[a] + a * a + 3 * a + 1) % (fmax + 1) for a in range(ndim)]
        active = sum(x != 0 for x in v)
        if active == 0:
            v[k % ndim] = 1 + k % fmax
        elif active == 1 and ndim > 1:
            v[(k + 1) % ndim] = 1 + (k // 2) % fmax
        if tuple(v) not in modes or tries >= max(64, 10 * rank * ndim):
            modes.append(tuple(v))
        tries, k = tries + 1, k + 1
    return modes[:rank]


def _unit(n, salt):
    v = (n + 1) * 0x9E3779B1 + (salt + 11) * 0x85EBCA77
    v ^= v >> 16
    v = v * 0x7FEB352D & 0xFFFFFFFF
    v ^= v >> 15
    v = v * 0x846CA68B & 0xFFFFFFFF
    return float((v ^ v >> 16) & 0xFFFFFF) / (1 << 24)


def _axis(u, a, ndim):
    return u.view([-1 if i == a else 1 for i in range(ndim)])


def _carriers(shape, freqs):
    """The normalized (cos, sin) field of every mode."""
    nd, out = len(shape), []
    axes = [(torch.arange(d, dtype=torch.float64, device=DEVICE) + 0.5) / d for d in shape]

    def normal(x):
        x = (x + torch.zeros(shape, dtype=torch.float64, device=DEVICE)).sub_(x.mean())
        return x.div_(torch.sqrt(x.square().mean() + 1e-12).clamp_min(1e-6))

    for r, f in enumerate(freqs):
        if not any(f):
            out.append((torch.ones(shape, dtype=torch.float64, device=DEVICE), torch.zeros(shape, dtype=torch.float64, device=DEVICE)))
            continue
        if r % 4 == 1:
            on = [(math.pi * f[a] * axes[a], a) for a in range(nd) if f[a]]
            out.append(tuple(normal(math.prod(_axis(fn(ph), a, nd) for ph, a in on)) for fn in (torch.cos, torch.sin)))
            continue
        phase = 0.0
        for a, u in enumerate(axes):
            part = math.pi * f[a] * u
            if r % 4:
                part = part + math.pi * (0.25 + 1.75 * _unit(r, 17 + a)) * max(1, f[a]) * (u - 0.5).square()
            phase = phase + _axis(part, a, nd)
        window = 1.0
        if r % 4 == 3:
            for a, u in enumerate(axes):
                mid, wide = 0.15 + 0.70 * _unit(r, 101 + a), 0.18 + 0.20 * _unit(r, 151 + a)
                window = window * _axis(torch.exp(-0.5 * ((u - mid) / wide).square()), a, nd)
        out.append((normal(window * torch.cos(phase)), normal(window * torch.sin(phase))))
    return out


def _bins(n, bins, table):
    s = table + 1
    i = torch.arange(n, dtype=torch.int64, device=DEVICE)
    i = i * (1103515245 + 97 * s) + (12345 + 0x9E3779B1 * s)
    i = (i ^ (i >> 16)) * (2246822519 + 1315423911 * s)
    i = (i ^ (i >> 13)) * (3266489917 + 374761393 * s)
    return torch.remainder(i ^ (i >> 16), bins)


def _bin_mean(x, index, bins):
    spread = 1024   # rows of sums, so that few additions meet
    at = index + bins * (torch.arange(index.numel(), device=DEVICE) % spread)
    total = torch.zeros(spread * bins, dtype=torch.float64, device=DEVICE).index_add_(0, at, x.reshape(-1))
    return total.view(spread, bins).sum(0) / torch.bincount(index, minlength=bins).clamp_min(1)


def _rms(x):
    return torch.sqrt(x.square().mean() + EPS)


def _ema(old, new, decay):
    return old.mul_(decay).add_(new, alpha=1.0 - decay)


def _to_rms(x, target):
    return x * (target / _rms(x).clamp_min(EPS))


def _instant(rel, coupling):
    """Per-axis marginal density metric."""
    nd, logm = rel.ndim, 0.0
    if rel.numel() <= 1:
        return torch.ones_like(rel)
    dens = rel.clamp_min(EPS).clamp(max=1e6)
    for a in range(nd):
        m = dens.mean(dim=[i for i in range(nd) if i != a], keepdim=True) if nd > 1 else dens
        logm = logm + torch.log((m / m.mean().clamp_min(EPS)).clamp_min(EPS))
    return torch.exp(coupling / nd * logm).clamp(0.08, 12.0)


def _update(st, drive, p):
    _ema(st["drive_energy"], drive.square().mean(), H["reservoir"])
    gain = (H["target"] / torch.sqrt(st["drive_energy"] + EPS)).clamp(H["min_gain"], H["max_gain"])
    p.sub_(LR * (drive * gain))


def _shape_drive(st, t, pred, err, p, echo=None, hashed=None, spectral=False):
    """Shaped drive of the scalar and spectral routes, and the update."""
    clip, sur = H["clip"], st["surprise"]
    frms, prms = _rms(t), _rms(pred)
    align = ((t * pred).mean() / (frms * prms + EPS)).clamp(-1.0, 1.0)
    gate = torch.where(prms > math.sqrt(EPS), ((align + 1.0) * 0.5).clamp(0.0, 1.0), torch.zeros_like(align))
    mix = H["prediction"] * (1.0 - math.exp(-(STEP + 1) / H["warmup"])) * gate / (1.0 + sur)
    bound = torch.tanh(t / clip) * clip
    rational = t / (1.0 + t.abs() / clip)
    root = t.sign() * torch.sqrt(t.abs().clamp(max=clip * clip) + EPS)
    root = _to_rms(root, _rms(rational))
    spike, rmix = H["spike"] / (1.0 + sur), H["root"] / (1.0 + 0.5 * sur)
    shaped = (1.0 - rmix) * ((1.0 - spike) * rational + spike * bound) + rmix * root
    novel = torch.tanh(err / (clip * (1.0 + sur))) * clip
    dmix = H["direct"] / (1.0 + 0.35 * sur)
    srms = _rms(shaped)
    core = (1.0 - dmix) * shaped + dmix * _to_rms(t, srms)
    drive = (1.0 - mix) * core + mix * pred + H["novelty"] * novel + H["residual"] / (1.0 + sur) * _to_rms(err, _rms(core))
    if spectral:
        drive = drive + H["echo"] * _to_rms(echo, srms) + H["hash_mix"] * _to_rms(hashed, srms)
    _update(st, drive, p)


def _begin(st, f):
    _ema(st["force_rms"], _rms(f), H["reservoir"])
    scale = st["force_rms"].clamp_min(EPS)
    return scale, (f.abs() / scale + EPS).clamp(max=1e4)


def _bank_power(port, st, p, w):
    """Energy-driven action and its friction, for one bank."""
    st["action"].mul_(0.985).add_((port * p).mean() - 0.5 * (p.square().mean() + w.square().mean()), alpha=H["dt"])
    return H["impulse_friction"] + H["contact_gain"] * torch.tanh(st["action"].abs())


def _scalar(st, f, p):
    scale, rel = _begin(st, f)
    dens = torch.log1p((f.abs() / scale + EPS).pow(H["energy_power"])).mean()
    mq, mp, dt = st["metric_q"], st["metric_impulse"], H["metric_dt"]
    port = dens - mq.tanh()
    mp.mul_(1.0 - dt * H["metric_friction"]).add_(port - mq, alpha=dt)
    mq.add_(mp, alpha=dt).clamp_(-3.0, 3.0)
    metric = torch.exp(H["metric_coupling"] * mq).clamp(0.06, 16.0)
    t = (f / (scale * metric * _instant(rel, H["instant"]) + EPS)).clamp(-1e4, 1e4)
    q, imp = st["q"], st["impulse"]
    err = t - q
    sur = _ema(st["surprise"], _rms(err), H["surprise_decay"])
    port = err.mean()
    push = (1.0 + H["surprise_gain"] * sur / (1.0 + sur)) / (1.0 + H["brake"] * sur) * port
    st["action"].mul_(0.985).add_(port * imp - 0.5 * (imp.square() + q.square()), alpha=H["dt"])
    friction = H["impulse_friction"] + H["contact_gain"] * torch.tanh(st["action"].abs())
    imp.mul_((1.0 - H["dt"] * friction).clamp_min(0.0)).add_(push - H["restoring"] * q - H["cubic"] * q.pow(3), alpha=H["dt"])
    q.add_(imp, alpha=H["dt"]).clamp_(-8.0, 8.0)
    pred = q.expand_as(t)
    _shape_drive(st, t, pred, t - pred, p)


def _micro(st, f, p):
    scale, rel = _begin(st, f)
    e, imp, ref = st["micro_energy"], st["micro_impulse"], st["micro_refractory"]
    _ema(e, rel.pow(H["energy_power"]), H["micro_decay"])
    metric = (e / e.mean().clamp_min(EPS)).pow(H["hash_coupling"] / H["energy_power"]).clamp(0.08, 12.0)
    t = (f / (scale * metric * _instant(rel, min(0.35, H["instant"])) + EPS)).clamp(-1e4, 1e4)
    _ema(ref, t.abs(), H["refractory"])
    pred = _ema(imp, t / (1.0 + H["refractory_gain"] * ref), H["micro_impulse"])
    err, clip = t - pred, H["clip"]
    sur = _ema(st["surprise"], _rms(err), H["surprise_decay"])
    spike = H["spike"] / (1.0 + sur)
    shaped = (1.0 - spike) * t / (1.0 + t.abs() / clip) + spike * torch.tanh(t / clip) * clip
    target = _rms(shaped)
    dmix, mmix = H["direct"] / (1.0 + 0.35 * sur), H["micro_mix"] / (1.0 + 0.25 * sur)
    drive = ((1.0 - dmix - 0.5 * mmix).clamp(0.0, 1.0) * shaped + dmix * _to_rms(t, target) + mmix * _to_rms(pred, target)
             + H["residual"] / (1.0 + sur) * _to_rms(err, target))
    _update(st, drive, p)


def _spectral(st, f, p, c, carriers, indices, omega):
    bins, tables = c["hash_bins"], c["hash_tables"]
    shrink = 1.0 / math.sqrt(max(1.0, 0.7 * math.log2(c["rank"] + 1.0)))

    def project(x):
        return tuple(torch.stack([(x * b[k]).mean() for b in carriers]) for k in (0, 1))

    def rebuild(cc, sc, gates=None):
        out = torch.zeros_like(f)
        for r, (bc, bs) in enumerate(carriers):
            g = shrink if gates is None else shrink * gates[r]
            out.addcmul_(bc, cc[r] * g).addcmul_(bs, sc[r] * g)
        return out

    scale, rel = _begin(st, f)
    source = rel.pow(H["energy_power"])
    logsum = 0.0
    for k, idx in enumerate(indices):
        e = _ema(st["hash_energy"][k], _bin_mean(source, idx, bins), H["hash_decay"])
        hm = (e / e.mean().clamp_min(EPS)).clamp_min(EPS).pow(H["hash_coupling"] / H["energy_power"])
        logsum = logsum + torch.log(hm.clamp(0.08, 12.0))[idx]
    hash_metric = torch.exp(logsum / tables).clamp(0.08, 12.0).view_as(f)
    dens = torch.log1p(source)
    for name, port in zip(("cos", "sin"), project(dens / dens.mean().clamp_min(EPS) - 1.0)):
        mq, mp = st["metric_" + name], st["metric_p_" + name]
        mp.mul_(1.0 - H["metric_dt"] * H["metric_friction"]).add_(port - omega.square() * mq, alpha=H["metric_dt"])
        mq.add_(mp, alpha=H["metric_dt"]).clamp_(-3.0, 3.0)
    logm = rebuild(st["metric_cos"], st["metric_sin"]).clamp(-3.0, 3.0)
    metric = torch.exp(H["metric_coupling"] * logm).clamp(0.06, 16.0)
    t = (f / (scale * metric * _instant(rel, H["instant"]) * hash_metric + EPS)).clamp(-1e4, 1e4)
    del rel, source, dens, logm, metric, hash_metric, logsum
    qs, conf = (st["q_cos"], st["q_sin"]), st["mode_confidence"]
    err = t - rebuild(*qs, torch.sigmoid(H["conf_gain"] * conf))
    sur = _ema(st["surprise"], _rms(err), H["surprise_decay"])
    source = err + H["transport"] * t
    ports = project(source)
    hashed = 0.0
    for k, idx in enumerate(indices):
        mean = _bin_mean(source, idx, bins)
        ref = _ema(st["hash_refractory"][k], mean.abs(), H["hash_decay"])
        hashed = hashed + _ema(st["hash_impulse"][k], mean / (1.0 + H["refractory_gain"] * ref), H["impulse_decay"])[idx]
    hashed = (hashed / tables).view_as(f)
    support = (ports[0] * qs[0] + ports[1] * qs[1]) / (torch.sqrt(ports[0] ** 2 + ports[1] ** 2 + EPS)
                                                       * torch.sqrt(qs[0] ** 2 + qs[1] ** 2 + EPS) + EPS)
    _ema(conf, support.clamp(-1.0, 1.0), H["conf_decay"]).clamp_(-4.0, 4.0)
    for name, q, port in zip(("cos", "sin"), qs, ports):
        pm, ca = st["p_" + name], st["calcium_" + name]
        _ema(ca, port.abs(), H["refractory"])
        push = (port / (1.0 + H["refractory_gain"] * ca) * (1.0 + H["surprise_gain"] * sur / (1.0 + sur))
                / (1.0 + H["brake"] * sur))
        friction = _bank_power(push, st, pm, omega * q)
        pm.mul_((1.0 - H["dt"] * friction).clamp_min(0.0))
        pm.add_(push - H["restoring"] * omega.square() * q - H["cubic"] * q.pow(3), alpha=H["dt"])
        q.add_(pm, alpha=H["dt"]).clamp_(-8.0, 8.0)
    pred = rebuild(*qs, torch.sigmoid(H["conf_gain"] * conf))
    _shape_drive(st, t, pred, t - pred, p, rebuild(*project(t)), hashed, True)


def exact(case, seed):
    with torch.no_grad():
        shapes, routes, param, grad, state, _ = _inputs(case, seed)
        param, grad = param.double(), grad.double()
        state = {k: v.double() for k, v in state.items()}
        cache = {}
        for s, route, p, g, st in zip(shapes, routes, _views(param, shapes), _views(grad, shapes),
                                      _state_views(shapes, routes, state)):
            f = g + case["weight_decay"] * p
            if route != "spectral":
                (_scalar if route == "scalar" else _micro)(st, f, p)
                continue
            freqs = _frequencies(case["rank"], len(s), case["max_frequency"])
            if s not in cache:
                cache[s] = (_carriers(s, freqs), [_bins(math.prod(s), case["hash_bins"], t) for t in range(case["hash_tables"])])
            omega = torch.sqrt(1.0 + torch.tensor(freqs, dtype=torch.float64, device=DEVICE).square().sum(1))
            _spectral(st, f, p, case, *cache[s], omega)
        return {"step": STEP + 1, "param": param, "state": state}
