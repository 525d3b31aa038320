"""Timed cases of the package: one polar_step, chains of steps (polar_express) and Muon
updates, from the smallest calls, where launches and latency count, to whole LLM weights.

A case is a dict: ``op`` names the entry point, ``batch``, ``m``, ``n`` the matrices
(``batch`` 0: a 2-D input), the rest its options.  ``listed()`` are fixed cases, ``draw``
makes others over the same ranges.
"""

from __future__ import annotations

import math

import torch

import muon_ascend950
import muon_fusion_ascend950_amd as mf

_DEV = "cuda"
_LR, _MOMENTUM, _DECAY = 0.02, 0.95, 0.01


def listed():
    return [
        # One step on the smallest, unaligned weight: three short launches.
        {"name": "step_129x130", "op": "step", "batch": 0, "m": 129, "n": 130},
        # Batched unaligned matrices: masked edge tiles, a long K over few rows.
        {"name": "step_2x150x2050", "op": "step", "batch": 2, "m": 150, "n": 2050},
        # A chain on small matrices of odd width, which no 16-byte access fits.
        {"name": "express_3x129x257", "op": "express", "batch": 3, "m": 129, "n": 257},
        # Batched projections, one step and the normalised five-step chain.
        {"name": "step_8x512x2048", "op": "step", "batch": 8, "m": 512, "n": 2048},
        {"name": "express_8x512x2048", "op": "express", "batch": 8, "m": 512, "n": 2048},
        # A middle-sized ragged weight.
        {"name": "step_1000x3001", "op": "step", "batch": 0, "m": 1000, "n": 3001},
        # An MLP up-projection and its transposed shape (right-Gram form).
        {"name": "step_4096x14336", "op": "step", "batch": 0, "m": 4096, "n": 14336},
        {"name": "step_14336x4096", "op": "step", "batch": 0, "m": 14336, "n": 4096},
        # Attention projections of a layer, orthogonalised in one call (the largest case).
        {"name": "express_4x4096x4096", "op": "express", "batch": 4, "m": 4096, "n": 4096},
        # The update of one parameter with bfloat16 gradients, plain momentum.
        {"name": "muon_1024x4096_bf16grad", "op": "muon", "batch": 0, "m": 1024, "n": 4096,
         "grad": "bfloat16", "nesterov": False},
        # The update of one large MLP weight.
        {"name": "muon_4096x14336", "op": "muon", "batch": 0, "m": 4096, "n": 14336,
         "grad": "float32", "nesterov": True},
        # An optimizer step over the matrices of two transformer layers.
        {"name": "optimizer_2x768", "op": "optimizer", "layers": 2, "d": 768},
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["step", "step", "express", "express", "muon", "optimizer"])
    if op == "optimizer":
        return {"op": op, "layers": rng.randint(1, 4), "d": 64 * rng.randint(4, 16)}
    while True:
        short = spread(64, 4096)
        long_ = spread(short, 14336)
        batch = spread(1, 32)
        # a third of the widths odd, a third whole 64-element blocks, the rest as drawn
        kind = rng.randrange(3)
        if kind == 0:
            long_ |= 1
        elif kind == 1:
            short = max(64, short - short % 64)
            long_ = max(short, long_ - long_ % 64)
        m, n = (long_, short) if rng.random() < 0.3 else (short, long_)
        case = {"op": op, "batch": 0 if batch == 1 else batch, "m": m, "n": n}
        if op == "muon":
            case["grad"] = rng.choice(["float32", "bfloat16"])
            case["nesterov"] = rng.random() < 0.7
        w = work(case)
        if max(1, batch) * m * n <= 1 << 26 and w["flops"] <= 6e12 and w["bytes"] <= 1.2e9:
            return case


def _shapes(case):
    """(batch, m, n) of every matrix or batch of matrices of a case."""
    if case["op"] == "optimizer":
        d = case["d"]
        per_layer = [(1, d, d)] * 4 + [(1, 4 * d, d), (1, d, 4 * d)]
        return per_layer * case["layers"]
    return [(max(1, case["batch"]), case["m"], case["n"])]


def work(case):
    op = case["op"]
    steps = 1 if op == "step" else 5
    nbytes = flops = 0
    for b, m, n in _shapes(case):
        s, l = min(m, n), max(m, n)
        # A = X·Xᵀ (symmetric: half the products), P = b·A + c·A², Y = a·X + P·X
        flops += steps * b * (s * s * l + 2 * s * s * s + 2 * s * s * l)
        if op in ("step", "express"):
            nbytes += b * m * n * 4  # X in, Y out, bf16
        else:
            # parameter and momentum buffer read and written, gradient read
            nbytes += b * m * n * (16 + (2 if case.get("grad") == "bfloat16" else 4))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # One step's rounding to bf16 puts it 1.6e-3 to 1.8e-3 from the formula in 64 bits, so
    # two roundings of it lie within about 2.5e-3.  Five steps amplify the small singular
    # values' rounding: sums in another order moved the result by up to 6.7e-3.
    if case["op"] == "step":
        return {"rel": 4e-3}
    if case["op"] == "express":
        return {"rel": 3e-2}
    # The parameter (standard deviation 0.02) moves by lr * scale * O; O has entries of
    # about 1 / sqrt(long side).  The buffer is float32 arithmetic, far inside this.
    def moved(m, n):
        return _LR * math.sqrt(max(1.0, m / n)) / math.sqrt(max(m, n)) / 0.02

    return {"rel": 3e-2 * max(moved(m, n) for _, m, n in _shapes(case))}


def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(int(seed))


def _x(case, gen):
    """bf16 input of a step: Gaussian, divided by its Frobenius norm (the norm of every
    matrix a chain's first step sees)."""
    shape = (case["m"], case["n"]) if not case["batch"] else (case["batch"], case["m"], case["n"])
    x = torch.randn(shape, generator=gen, device=_DEV, dtype=torch.float32)
    if case["op"] == "step":
        x /= torch.linalg.vector_norm(x, dim=(-2, -1), keepdim=True) * 1.01 + 1e-6
    return x.to(torch.bfloat16)


def _muon_tensors(shape, gen, grad_dtype):
    """Parameter, gradient and momentum buffer of a matrix in training: a weight of
    standard deviation 0.02, a gradient of noise over a few strong directions, a buffer
    that holds an average of such gradients."""
    def gradient(scale):
        m, n = shape[-2:]
        lead = shape[:-2]
        u = torch.randn(lead + (m, 4), generator=gen, device=_DEV) / 2
        v = torch.randn(lead + (4, n), generator=gen, device=_DEV)
        noise = torch.randn(shape, generator=gen, device=_DEV)
        for i in range(4):
            noise += u[..., :, i:i + 1] * v[..., i:i + 1, :]
        return noise * scale

    p = torch.randn(shape, generator=gen, device=_DEV) * 0.02
    return p, gradient(1e-3).to(grad_dtype), gradient(3e-4)


def prepare(case, seed):
    gen = _gen(seed)
    op = case["op"]
    if op in ("step", "express"):
        return {"op": op, "x": _x(case, gen)}
    if op == "muon":
        shape = (case["m"], case["n"]) if not case["batch"] else (case["batch"], case["m"], case["n"])
        p, g, buf = _muon_tensors(shape, gen, getattr(torch, case["grad"]))
        return {"op": op, "p": p, "g": g, "buf": buf, "nesterov": case["nesterov"]}
    params, bufs = [], []
    for _, m, n in _shapes(case):
        p, g, buf = _muon_tensors((m, n), gen, torch.float32)
        p = torch.nn.Parameter(p)
        p.grad = g
        params.append(p)
        bufs.append(buf)
    opt = mf.Muon(params, lr=_LR, momentum=_MOMENTUM, weight_decay=_DECAY)
    for p, buf in zip(params, bufs):
        opt.state[p]["momentum_buffer"] = buf
    return {"op": op, "opt": opt, "params": params, "bufs": bufs}


def run(state):
    op = state["op"]
    if op == "step":
        return muon_ascend950.polar_step(state["x"], *mf.COEFFICIENTS[0])
    if op == "express":
        return mf.polar_express(state["x"])
    if op == "muon":
        mf.muon_update(state["p"], state["g"], state["buf"], lr=_LR, momentum=_MOMENTUM,
                       nesterov=state["nesterov"], weight_decay=_DECAY)
        return state["p"], state["buf"]
    state["opt"].step()
    return [p.detach() for p in state["params"]] + list(state["bufs"])


def _step64(x, a, b, c):
    """One step of one float64 matrix on its shorter side."""
    if x.shape[0] > x.shape[1]:
        return _step64(x.t().contiguous(), a, b, c).t()
    gram = x @ x.t()
    p = b * gram + c * (gram @ gram)
    return a * x + p @ x


def _express64(x):
    x = x / (torch.linalg.vector_norm(x) * 1.01 + 1e-6)
    for a, b, c in mf.COEFFICIENTS:
        x = _step64(x, a, b, c)
    return x


def _batched64(f, x):
    x = x.double()
    if x.ndim == 2:
        return f(x).contiguous()
    return torch.stack([f(m) for m in x])


def _muon64(p, g, buf, nesterov):
    m, n = p.shape[-2:]
    g, buf = g.double(), buf.double()
    buf = buf + (1.0 - _MOMENTUM) * (g - buf)
    g = g + _MOMENTUM * (buf - g) if nesterov else buf
    o = _batched64(_express64, g)
    scale = _LR * math.sqrt(max(1.0, m / n))
    return p.double() * (1.0 - _LR * _DECAY) - scale * o, buf


def exact(case, seed):
    state = prepare(case, seed)
    op = state["op"]
    if op == "step":
        return _batched64(lambda m: _step64(m, *mf.COEFFICIENTS[0]), state["x"])
    if op == "express":
        return _batched64(_express64, state["x"])
    if op == "muon":
        return _muon64(state["p"], state["g"], state["buf"], state["nesterov"])
    pairs = [_muon64(p.detach(), p.grad, buf, True)
             for p, buf in zip(state["params"], state["bufs"])]
    return [p for p, _ in pairs] + [b for _, b in pairs]
