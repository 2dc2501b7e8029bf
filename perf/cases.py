"""What this package is timed on: passes through its public entry points over the sizes,
types and options that its users give it.

A case is a dict of plain values.  Its "path" names the entry point:

    plain    zeropower_via_newtonschulz5 / PolarExpress on one gradient, or on the three
             blocks of a W_QKV gradient: the call the plain arms make for each parameter
    iterate  _horner_iterate in fp32: the convergence study's iteration
    clip     batched_rmfro_clip: the deflation front-end by itself, X0 in fp32 or bf16
    groups   polar_groups of a deflated arm: the polar step of a whole model
    step     Muon.step: momentum, polar factors, update and the AdamW backup

Inputs are Gaussian gradients, and momenta with a few large singular values over a Gaussian
bulk where the path looks for them; every fourth momentum of a batch has none.
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "spectral-deflation_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from defmuon_amd.optim import deflation_batched as defl  # noqa: E402
from defmuon_amd.optim import deflation_cutoff, muon, polar_express  # noqa: E402

DEV = "cuda"
STEPS = 5
ARMS = {"ns5": muon.zeropower_via_newtonschulz5, "polarexpress": polar_express.PolarExpress}
DEFLATED = {"deflated_ns_cut": deflation_cutoff.CutoffDeflatedNSPolar,
            "deflated_pe_cut": deflation_cutoff.CutoffDeflatedPEPolar}
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # a hidden matrix of a toy model: nothing but launches and latency
        {"name": "plain 192x96", "path": "plain", "arm": "ns5", "blocks": 1, "rows": 192,
         "cols": 96, "dtype": "fp32"},
        # the c_fc gradient of GPT-2 small, one call per parameter
        {"name": "plain 768x3072", "path": "plain", "arm": "ns5", "blocks": 1, "rows": 768,
         "cols": 3072, "dtype": "fp32"},
        # GPT-2 large's W_QKV gradient, three blocks in one call
        {"name": "plain qkv 3x1280x1280", "path": "plain", "arm": "polarexpress", "blocks": 3,
         "rows": 1280, "cols": 1280, "dtype": "fp32"},
        # a ragged layer of a model kept in bf16
        {"name": "plain bf16 1000x333", "path": "plain", "arm": "polarexpress", "blocks": 1,
         "rows": 1000, "cols": 333, "dtype": "bf16"},
        # the convergence study on a handful of dumped momenta
        {"name": "iterate fp32 8x1536x768", "path": "iterate", "batch": 8, "n": 1536, "m": 768},
        # the front-end of the accuracy studies: fp32 X0 of one shape group
        {"name": "clip 24x1024x1024", "path": "clip", "batch": 24, "n": 1024, "m": 1024,
         "dtype": "fp32"},
        # a width that is no multiple of anything
        {"name": "clip ragged 6x1001x333", "path": "clip", "batch": 6, "n": 1001, "m": 333,
         "dtype": "bf16"},
        # one deflated matrix: latency of the whole deflated path
        {"name": "groups 1x3072x768", "path": "groups", "arm": "deflated_ns_cut",
         "square": 0, "tall": 1, "m": 768, "ratio": 4},
        # the polar step of GPT-2 small
        {"name": "groups gpt2-small", "path": "groups", "arm": "deflated_ns_cut",
         "square": 48, "tall": 24, "m": 768, "ratio": 4},
        # the polar step of GPT-2 large: the largest work there is
        {"name": "groups gpt2-large", "path": "groups", "arm": "deflated_pe_cut",
         "square": 144, "tall": 72, "m": 1280, "ratio": 4},
        # the optimizer over four GPT-2-small layers and the embeddings, plain arm
        {"name": "step ns5 4 layers", "path": "step", "arm": "ns5", "layers": 4, "d": 768,
         "vocab": 50257},
        # ... and deflated
        {"name": "step deflated 4 layers", "path": "step", "arm": "deflated_ns_cut", "layers": 4,
         "d": 768, "vocab": 50257},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A matrix side: a multiple of 64, of 8, or any number at all."""
    v = _log_int(rng, lo, hi)
    q = rng.choice((64, 64, 8, 1))
    return max(lo, min(hi, v // q * q))


def draw(rng):
    path = rng.choice(("plain", "plain", "plain", "iterate", "clip", "clip", "groups", "groups",
                       "step"))
    if path == "plain":
        a, b = _width(rng, 32, 1280), _width(rng, 32, 5120)
        if rng.random() < 0.5:
            a, b = b, a
        blocks = rng.choice((1, 1, 3))
        return {"path": path, "arm": rng.choice(sorted(ARMS)), "blocks": blocks,
                "rows": a, "cols": b, "dtype": rng.choice(("fp32", "fp32", "bf16"))}
    if path == "iterate":
        m = _width(rng, 32, 1024)
        return {"path": path, "batch": _log_int(rng, 1, 12), "n": m * rng.choice((1, 2, 4)), "m": m}
    if path == "clip":
        m = _width(rng, 64, 1280)
        return {"path": path, "batch": _log_int(rng, 1, 32),
                "n": max(m, int(m * rng.uniform(1, 4.3))), "m": m,
                "dtype": rng.choice(("fp32", "bf16"))}
    if path == "groups":
        return {"path": path, "arm": rng.choice(sorted(DEFLATED)),
                "square": _log_int(rng, 1, 96) - 1, "tall": _log_int(rng, 1, 48),
                "m": _width(rng, 64, 1280), "ratio": rng.choice((2, 3, 4))}
    return {"path": path, "arm": rng.choice(sorted(ARMS) + sorted(DEFLATED)),
            "layers": rng.randint(1, 4), "d": _width(rng, 64, 1024) // 8 * 8,
            "vocab": _log_int(rng, 512, 50257)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _momenta(batch, n, m, gen, all_spiked=False):
    """(batch, n, m) fp32: N(0, 1/n) bulk and, but for every fourth matrix, up to eight
    singular values 50 to 10 times it (as many as a deflation window of m columns holds)."""
    A = torch.randn(batch, n, m, device=DEV, generator=gen).mul_(n ** -0.5)
    window = min(n, m)
    window = max(1, math.ceil(defl.GATE_WINDOW * window))
    spikes = max(0, min(8, window - 1))
    if spikes:
        U = torch.randn(batch, n, spikes, device=DEV, generator=gen).mul_(n ** -0.5)
        V = torch.randn(batch, spikes, m, device=DEV, generator=gen).mul_(m ** -0.5)
        s = 2.0 * torch.logspace(math.log10(50.0), math.log10(10.0), spikes, device=DEV)
        s = s.expand(batch, spikes).clone()
        if not all_spiked:
            s[3::4] = 0
        A.baddbmm_(U * s[:, None, :], V)
    return A


def _group_shapes(case):
    """(batch, n, m) of each group of the step, in the optimizer's order (by shape)."""
    m = case["m"]
    groups = [(case["square"], m, m), (case["tall"], case["ratio"] * m, m)]
    return [g for g in groups if g[0]]


def _model_shapes(case):
    d = case["d"]
    shapes = {"wte.weight": (case["vocab"], d), "wpe.weight": (1024, d)}
    for i in range(case["layers"]):
        shapes[f"h.{i}.ln_1.weight"] = (d,)
        shapes[f"h.{i}.attn.c_attn.weight"] = (3 * d, d)
        shapes[f"h.{i}.attn.c_proj.weight"] = (d, d)
        shapes[f"h.{i}.ln_2.weight"] = (d,)
        shapes[f"h.{i}.mlp.c_fc.weight"] = (4 * d, d)
        shapes[f"h.{i}.mlp.c_proj.weight"] = (d, 4 * d)
    return shapes


def _is_muon(name, shape):
    return len(shape) == 2 and "wte" not in name and "wpe" not in name


def _step_inputs(case, seed):
    """Parameters and gradients of the model, by name."""
    gen = _generator(seed)
    params, grads = {}, {}
    for name, shape in _model_shapes(case).items():
        params[name] = torch.randn(*shape, device=DEV, generator=gen).mul_(0.02)
        if not _is_muon(name, shape):
            grads[name] = torch.randn(*shape, device=DEV, generator=gen).mul_(0.01)
        elif "c_attn" in name:
            grads[name] = _momenta(3, shape[0] // 3, shape[1], gen, True).reshape(shape)
        else:
            grads[name] = _momenta(1, *shape, gen, True)[0]
    return params, grads


LR, WEIGHT_DECAY, MOMENTUM, BETAS, EPS = 0.01, 0.1, 0.95, (0.9, 0.95), 1e-8


def _sketch(batch, m, seed):
    return torch.randn(batch, m, defl.sketch_dims(m)[0], device=DEV, generator=_generator(seed))


def prepare(case, seed):
    path = case["path"]
    gen = _generator(seed)
    if path == "plain":
        shape = (case["rows"], case["cols"])
        if case["blocks"] > 1:
            shape = (case["blocks"],) + shape
        G = torch.randn(*shape, device=DEV, generator=gen).mul_(1e-2).to(DTYPES[case["dtype"]])
        return case, G
    if path == "iterate":
        X = torch.randn(case["batch"], case["n"], case["m"], device=DEV, generator=gen)
        X /= X.flatten(1).norm(dim=1)[:, None, None]
        return case, X
    if path == "clip":
        A = _momenta(case["batch"], case["n"], case["m"], gen)
        return case, A, _sketch(case["batch"], case["m"], seed + 1)
    if path == "groups":
        As = [_momenta(*g, gen) for g in _group_shapes(case)]
        return case, As, DEFLATED[case["arm"]](), [torch.Generator(device=DEV) for _ in As], seed
    deflation_cutoff.install()
    values, grads = _step_inputs(case, seed)
    params = {k: torch.nn.Parameter(v) for k, v in values.items()}
    opt = muon.Muon(list(params.items()), lr=LR, weight_decay=WEIGHT_DECAY, momentum=MOMENTUM,
                    polar_method=case["arm"], adamw_betas=BETAS, adamw_eps=EPS)
    for k, p in params.items():
        p.grad = grads[k]
    return case, params, opt


def run(state):
    case, path = state[0], state[0]["path"]
    if path == "plain":
        return ARMS[case["arm"]](state[1], STEPS)
    if path == "iterate":
        return defl._horner_iterate(state[1], [muon.NS_ABC] * STEPS)
    if path == "clip":
        return defl.batched_rmfro_clip(state[1], Omega=state[2], out_dtype=DTYPES[case["dtype"]])
    if path == "groups":
        _, As, arm, gens, seed = state
        for i, g in enumerate(gens):
            g.manual_seed(seed * 31 + i)
        return arm.polar_groups(As, gens, steps=STEPS)
    _, params, opt = state
    opt.step()
    out = {k: p.detach() for k, p in params.items()}
    for k, p in params.items():
        st = opt.state[p]
        for s in ("momentum_buffer", "moment1", "moment2"):
            if s in st:
                out[k + " " + s] = st[s]
    return out


# ---------------------------------------------------------------------------
# the work of a pass
# ---------------------------------------------------------------------------

def _chain_flops(n, m):
    """One matrix: X^T X and its square by their upper halves, and the product with X."""
    return STEPS * (float(m) * m * n + float(m) ** 3 + 2.0 * m * m * n)


def _front_flops(n, m):
    """The four products of the sketch iteration with A."""
    return 4 * 2.0 * n * m * defl.sketch_dims(m)[0]


def work(case):
    path = case["path"]
    if path == "plain":
        n, m = max(case["rows"], case["cols"]), min(case["rows"], case["cols"])
        size = DTYPES[case["dtype"]].itemsize
        return {"bytes": case["blocks"] * n * m * (size + 2),
                "flops": case["blocks"] * _chain_flops(n, m)}
    if path == "iterate":
        b, n, m = case["batch"], case["n"], case["m"]
        return {"bytes": b * n * m * 8, "flops": b * _chain_flops(n, m)}
    if path == "clip":
        b, n, m = case["batch"], case["n"], case["m"]
        return {"bytes": b * n * m * (4 + DTYPES[case["dtype"]].itemsize),
                "flops": b * _front_flops(n, m)}
    if path == "groups":
        gs = _group_shapes(case)
        return {"bytes": sum(b * n * m * 6 for b, n, m in gs),
                "flops": sum(b * (_chain_flops(n, m) + _front_flops(n, m)) for b, n, m in gs)}
    nbytes = flops = 0
    for name, shape in _model_shapes(case).items():
        size = math.prod(shape)
        if not _is_muon(name, shape):
            nbytes += size * 28
            continue
        nbytes += size * 20
        blocks = 3 if "c_attn" in name else 1
        rows, cols = shape[0] // blocks, shape[1]
        n, m = max(rows, cols), min(rows, cols)
        flops += blocks * _chain_flops(n, m)
        if case["arm"] in DEFLATED:
            flops += blocks * _front_flops(n, m)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the same arithmetic summed in another order differs by: the
    bf16 chains by 0.005 to 0.008 (other tile sizes walk K in another order), the updated
    parameters by 2.3e-4, the fp32 paths by 3.5e-6 (iterate) and 2e-6 (clip) from 64 bits;
    X0 in bf16 by a last place where the fp32 values straddle a rounding boundary."""
    path = case["path"]
    if path == "iterate":
        return {"rel": 1.4e-5, "max": 2e-4}
    if path == "clip" and case["dtype"] == "fp32":
        return {"rel": 8e-6, "max": 1e-4}
    if path == "clip":
        return {"rel": 4e-4, "max": 8e-3}
    if path == "step":
        return {"rel": 1e-3, "max": 1e-2}
    return {"rel": 0.03, "max": 0.4}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _chain64(X, coeffs):
    """X <- aX + X (b G + c G^2), G = X^T X, on a (batch, n, m) fp64 stack."""
    if X.shape[-2] < X.shape[-1]:
        return _chain64(X.mT.contiguous(), coeffs).mT
    for a, b, c in coeffs:
        G = X.mT.contiguous() @ X
        X = a * X + X @ (b * G + c * (G @ G))
    return X


def _coeffs(arm):
    if arm in ("ns5", "deflated_ns_cut"):
        return [muon.NS_ABC] * STEPS
    return polar_express.pe_schedule(STEPS)


def _plain64(G, arm):
    X = G.double()
    norm = X.flatten(-2).norm(dim=-1)[..., None, None]
    X = X / (norm + 1e-7 if arm == "ns5" else norm * 1.01 + 1e-7)
    return _chain64(X, _coeffs(arm))


def _orth64(Y):
    R = torch.linalg.cholesky((Y.mT.contiguous() @ Y).cpu(), upper=True)
    return Y @ torch.linalg.inv(R).to(Y.device)


def _clip64(A, Omega, pad):
    """(X0, k, d) of the deflation front-end on one batch."""
    A, Omega = A.double(), Omega.double()
    At = A.mT.contiguous()
    r, kw = defl.sketch_dims(A.shape[-1])
    Q = _orth64(A @ Omega)
    for _ in range(defl.RSVD_NITER):
        Q = _orth64(A @ _orth64(At @ Q))
    Bt = At @ Q
    lam, W = torch.linalg.eigh((Bt.mT.contiguous() @ Bt).cpu())
    lam, W = lam.flip(-1).to(A.device), W.flip(-1).to(A.device)
    s = lam.clamp_min(0).sqrt()
    kr = (s > defl.DEFLATE_THRESH * s[:, :1]).sum(-1)
    fired = (s[:, kw - 1] < defl.GATE_RATIO * s[:, 0]) & (kr >= 1) & (kr < r)
    k = torch.where(fired, kr.clamp(1, r - 1), torch.zeros_like(kr))
    h = (torch.arange(r, device=A.device)[None] < k[:, None]).double()
    U, V = Q @ W, Bt @ (W / s[:, None, :])
    R = A - (U * (s * h)[:, None, :]) @ V.mT.contiguous()
    d = R.flatten(1).norm(dim=1) + 1e-7
    X0 = R / d[:, None, None] + (U * (h / pad)[:, None, :]) @ V.mT.contiguous()
    return X0, k, d


def _group64(A, gen, arm):
    Omega = torch.randn(A.shape[0], A.shape[2], defl.sketch_dims(A.shape[2])[0], device=DEV,
                        generator=gen)
    X0, k, d = _clip64(A, Omega, DEFLATED[arm].PAD)
    return _chain64(X0, _coeffs(arm)), k, d


def exact(case, seed):
    path = case["path"]
    if path == "step":
        return _step64(case, seed)
    state = prepare(case, seed)
    if path == "plain":
        return _plain64(state[1], case["arm"])
    if path == "iterate":
        return _chain64(state[1].double(), [muon.NS_ABC] * STEPS)
    if path == "clip":
        return _clip64(state[1], state[2], defl.DIVISOR_PAD)
    _, As, _, gens, s = state
    for i, g in enumerate(gens):
        g.manual_seed(s * 31 + i)
    return [_group64(A, g, case["arm"]) for A, g in zip(As, gens)]


def _step64(case, seed):
    """The first step from fresh state."""
    arm = case["arm"]
    params, grads = _step_inputs(case, seed)
    out, polar, groups = {}, {}, {}
    for name, p in params.items():
        g = grads[name].double()
        if not _is_muon(name, p.shape):
            m1, m2 = (1 - BETAS[0]) * g, (1 - BETAS[1]) * g * g
            scale = (1 - BETAS[0]) / (1 - BETAS[1]) ** 0.5
            out[name] = p.double() * (1 - LR * WEIGHT_DECAY) - LR / scale * (
                m1 / (EPS + m2.sqrt()))
            out[name + " moment1"], out[name + " moment2"] = m1, m2
            continue
        out[name + " momentum_buffer"] = g
        A = g + MOMENTUM * g
        A = A.reshape(3, -1, A.shape[1]) if "c_attn" in name else A[None]
        if arm not in DEFLATED:
            polar[name] = _plain64(A, arm).reshape(p.shape)
            continue
        wide = A.shape[-2] < A.shape[-1]
        A = A.mT if wide else A
        groups.setdefault(tuple(A.shape[-2:]), []).append((name, A, wide))
    for i, (_, es) in enumerate(sorted(groups.items())):
        A = torch.cat([e[1] for e in es])
        U, _, _ = _group64(A, _generator((1009 + i * 9176867) % (2 ** 62)), arm)
        for (name, A, wide), u in zip(es, U.split([len(e[1]) for e in es])):
            polar[name] = (u.mT if wide else u).reshape(params[name].shape)
    for name, u in polar.items():
        p = params[name].double()
        lr = LR * math.sqrt(p.shape[0] / p.shape[1])
        out[name] = p * (1 - LR * WEIGHT_DECAY) - lr * u
    return out
