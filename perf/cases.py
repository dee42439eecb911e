"""Performance cases of the optimizer framework, through its public entry points.

A case is one call (or the few calls of one training iteration) that a
training program makes: an optimizer step over a parameter list, gradient
clipping with it, the read-out of the diagnostics, and the collection of the
tau order statistics.  The model sizes are those of the repository's own
benchmark and smoke test; ``draw`` spreads over the same ranges.

Parameters, gradients and optimizer state are views of flat buffers (one per
kind, each tensor on a 1,024-element boundary, as the optimizer's own slabs
have them), so that a pass returns them whole in a few tensors.  A case starts
in the middle of a run (``start`` steps taken): moments and tau hold what such
a run has in them, and gradients have a global norm of ``grad_norm``.

Fields of a case:
  path         "step" or "tau"
  optimizer    "adana" (clipsnr 0: ADana, else Dana-MK4) or "star" (Dana-Star)
  state        "fp32"; "master" (bfloat16 parameters, float32 master and
               moments); "bf16" (bfloat16 parameters and moments)
  foreach, eager   use_foreach=True; numerics="eager"
  clip         "none"; "fused" (the optimizer's clip_grad_norm_, applied by
               its step); "call" (the function, in place, before the step)
  log          whether the diagnostics are read out after the step
  list         "gpt" (vocab, d, layers, ln_bias), "mixed" (tensors 1-D tensors
               of lo..hi elements, log-uniform), "matrix" (rows x d), "small"
"""
import functools
import math
import random

import numpy as np
import torch

import adana_amd

ALIGN = 1024                      # elements: each tensor starts on such a boundary of its flat buffer
DELTA, EPS, LR = 8.0, 1e-8, 1e-3
WD_TS = 100.0
DIAG = ("current_alpha", "gradient_norm", "auto_factor_mean", "current_kappa_factor", "m_norm")
FEW = 8                           # up to so many tensors, their 0-d diagnostics are outputs too

BASE = dict(path="step", optimizer="star", clipsnr=2.0, kappa=0.85, state="fp32", foreach=False, eager=False,
            clip="none", max_norm=0.5, grad_norm=0.3, log=False, start=1000)
GPT_51M = dict(list="gpt", vocab=50304, d=512, layers=8, ln_bias=True)
GPT_1B = dict(list="gpt", vocab=50304, d=2048, layers=24, ln_bias=False)
GPT_2B = dict(list="gpt", vocab=50304, d=2560, layers=32, ln_bias=False)
SMALL_TENSORS = dict(list="mixed", tensors=10000, lo=64, hi=65536, sizes=5)


def listed():
    def case(name, *parts, **more):
        c = dict(BASE, name=name)
        for p in parts:
            c.update(p)
        c.update(more)
        return c

    return [
        # the smallest call: a toy model's four tensors (20,000 values), all launches and host work
        case("toy_adana", dict(list="small"), optimizer="adana", clipsnr=0.0),
        # one weight matrix of 4M values (also what a flat-parameter shard looks like)
        case("matrix_adana", dict(list="matrix", rows=1024, d=4096), optimizer="adana", clipsnr=0.0),
        # a 51M-parameter GPT in 67 tensors, the step alone, Dana-MK4
        case("gpt51m_mk4", GPT_51M, optimizer="adana"),
        # the same model's logging iteration: clip (not binding, as in most steps of a run), step, read-out
        case("gpt51m_clip_log", GPT_51M, clip="fused", log=True),
        # the same model on the reference's foreach path with bfloat16 parameters and state
        case("gpt51m_foreach_bf16", GPT_51M, state="bf16", foreach=True),
        # 10,000 tensors of 64 to 65,536 values: many small parameters
        case("small_tensors", SMALL_TENSORS),
        # the same list with a binding clip before the step
        case("small_tensors_clip", SMALL_TENSORS, clip="fused", grad_norm=2.0),
        # a 1.3B-parameter GPT, float32, Dana-Star-MK4
        case("gpt1b_star", GPT_1B),
        # the same model with bfloat16 parameters and float32 master weights, clipped in place before the step
        case("gpt1b_master_clip", GPT_1B, optimizer="adana", clipsnr=0.0, state="master", clip="call", grad_norm=2.0),
        # the largest: a 2.6B-parameter GPT with bfloat16 parameters and state
        case("gpt2b_star_bf16", GPT_2B, state="bf16"),
        # tau order statistics of one matrix
        case("tau_matrix", dict(list="matrix", rows=1024, d=4096), path="tau"),
        # and of the 1.3B-parameter model's whole state (collected at evaluation steps)
        case("tau_gpt1b", GPT_1B, path="tau"),
    ]


def _log_uniform(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999))))


def draw(rng):
    """One more case: the same paths and options over the whole range of sizes,
    from a thousand values to the largest listed case's bytes."""
    while True:
        c = dict(BASE, path="tau" if rng.random() < 0.2 else "step")
        if c["path"] == "step":
            c["optimizer"] = rng.choice(["adana", "star", "star"])
            c["state"] = rng.choice(["fp32", "fp32", "master", "bf16"])
            c["foreach"] = rng.random() < 0.2
            c["eager"] = rng.random() < 0.15
            c["kappa"] = rng.choice([0.75, 0.85, 0.85, 1.0])
            c["clip"] = rng.choice(["none", "fused", "call"])
            c["grad_norm"] = rng.choice([0.1, 0.3, 2.0])
            c["log"] = rng.random() < 0.2
            if c["optimizer"] == "adana" or rng.random() < 0.3:
                c["clipsnr"] = rng.choice([0.0, 2.0]) if c["optimizer"] == "adana" else 1.0
        c["start"] = _log_uniform(rng, 10, 50000)
        kind = rng.choice(["gpt", "gpt", "mixed", "matrix"])
        c["list"] = kind
        if kind == "gpt":
            d = _log_uniform(rng, 48, 2560)
            c.update(vocab=_log_uniform(rng, 1000, 50304), d=d, layers=rng.randint(1, 32), ln_bias=rng.random() < 0.5)
        elif kind == "mixed":
            lo, hi = sorted(_log_uniform(rng, 1, 200000) for _ in range(2))
            c.update(tensors=_log_uniform(rng, 1, 10000), lo=lo, hi=hi, sizes=rng.randrange(1 << 20))
        else:
            c.update(rows=_log_uniform(rng, 1, 50304), d=_log_uniform(rng, 33, 10240))
        if 1000 <= sum(math.prod(s) for s, _ in _shapes(c)) and _cost(c) <= _cost(dict(BASE, **GPT_2B, state="bf16")):
            return c


def _shapes(case):
    """[(shape, decayed)] of the case's parameters, the decayed group first."""
    if case["list"] == "small":
        return [((64, 33), True), ((1000,), False), ((5,), False), ((16384 + 7,), False)]
    if case["list"] == "matrix":
        return [((case["rows"], case["d"]), True)]
    if case["list"] == "mixed":
        r = random.Random(case["sizes"])
        return [((_log_uniform(r, case["lo"], case["hi"]),), True) for _ in range(case["tensors"])]
    d, norms = case["d"], 2 if case["ln_bias"] else 1
    decay = [(3 * d, d), (d, d), (4 * d, d), (d, 4 * d)] * case["layers"]
    rest = [(case["vocab"], d)] + [(d,)] * (norms * (2 * case["layers"] + 1))
    return [(s, True) for s in decay] + [(s, False) for s in rest]


def _layout(case):
    """[(offset, shape, decayed)] and the flat buffers' length."""
    out, off = [], 0
    for s, decayed in _shapes(case):
        out.append((off, s, decayed))
        off += -(-math.prod(s) // ALIGN) * ALIGN
    return out, off


def _elems(case):
    return sum(math.prod(s) for s, _ in _shapes(case))


def _bytes_per_elem(case):
    """Each input read once and each output written once."""
    if case["path"] == "tau":
        return 4
    star = case["optimizer"] == "star"
    if case["state"] == "master":
        b = 28 + (8 if star else 0)      # master, m, v [, tau] 4 + 4 each, gradient 2, parameter 2
        g = 2
    else:
        g = 2 if case["state"] == "bf16" else 4
        b = g * (9 if star else 7)       # p, m, v [, tau] in and out, gradient in
    return b + (g if case["clip"] != "none" else 0)   # the clipped gradient is written


def _cost(case):
    return _elems(case) * _bytes_per_elem(case)


def work(case):
    n = _elems(case)
    if case["path"] == "tau":
        return {"bytes": 4.0 * n, "flops": 1.0 * n}
    return {"bytes": float(_cost(case)), "flops": (60.0 if case["optimizer"] == "star" else 28.0) * n}


def _inputs(case, seed):
    """The flat buffers before the pass: p, g, m, v[, tau][, master]."""
    lay, total = _layout(case)
    n = sum(math.prod(s) for _, s, _ in lay)
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    rng = random.Random(seed)
    low = torch.float32 if case["state"] == "fp32" else torch.bfloat16      # parameter and gradient
    mom = torch.bfloat16 if case["state"] == "bf16" else torch.float32      # moments and tau
    a = DELTA / (DELTA + case["start"])
    sd = case["grad_norm"] / math.sqrt(n)
    star = case["optimizer"] == "star"
    tau_only = case["path"] == "tau"

    def normal(dtype, mean, std):
        return torch.empty(total, dtype=dtype, device=dev).normal_(mean, std, generator=gen)

    b = {}
    if not tau_only:
        if case["state"] == "master":
            b["master"] = normal(torch.float32, 0.0, 0.02)
            b["p"] = b["master"].to(torch.bfloat16)
        else:
            b["p"] = normal(low, 0.0, 0.02)
        b["g"] = normal(low, 0.0, sd)
        b["m"] = normal(mom, 0.0, sd * math.sqrt(a / 2))
        b["v"] = normal(mom, 0.0, 0.3).exp_().mul_(sd * sd)
    if star:
        # |g| / (|g| + sqrt(v)) averaged over the last steps
        b["tau"] = normal(mom, 0.4, 0.2 * math.sqrt(a / 2)).clamp_(0.0, 1.0)
    for i, (off, s, _) in enumerate(lay):
        m = math.prod(s)
        if case["list"] == "gpt" and len(s) == 2 and s[0] == case["vocab"]:
            # embedding rows are met by frequency: few have a gradient now, the state of rare ones is small
            f = torch.pow(10.0, -3.0 * torch.rand((s[0], 1), device=dev, generator=gen))
            hit = (torch.rand((s[0], 1), device=dev, generator=gen) < 0.1)
            for k in ("m", "v", "tau"):
                if k in b:
                    b[k][off:off + m].view(s).mul_(f.to(b[k].dtype))
            if "g" in b:
                b["g"][off:off + m].view(s).mul_(hit.to(low))
        elif case["list"] == "gpt" and star:
            b["tau"][off:off + m].mul_(rng.uniform(0.5, 1.1))        # layers differ
        elif case["list"] == "mixed" and "g" in b and rng.random() < 0.05:
            b["g"][off:off + m].zero_()
    return b, lay


def _hyper(case):
    return dict(lr=LR, delta=DELTA, kappa=case["kappa"], epsilon=EPS, clipsnr=case["clipsnr"] or None,
                wd_decaying=True, wd_ts=WD_TS)


def prepare(case, seed):
    b, lay = _inputs(case, seed)
    if case["path"] == "tau":
        taus = [b["tau"][off:off + math.prod(s)].view(s) for off, s, _ in lay]
        params = [torch.nn.Parameter(torch.empty(0, device="cuda")) for _ in taus] if len(taus) > 1 else []
        opt = None
        if params:
            opt = adana_amd.DANA_STAR_MK4(params, **_hyper(case))
            for p, t in zip(params, taus):
                opt.state[p] = {"step": case["start"], "tau": t}
        return {"case": case, "opt": opt, "taus": taus, "params": params}
    groups = {True: [], False: []}
    params, held = [], []
    for off, s, decayed in lay:
        n = math.prod(s)
        p = torch.nn.Parameter(b["p"][off:off + n].view(s))
        p.grad = b["g"][off:off + n].view(s)
        st = {"step": case["start"]}
        for k in ("m", "v", "tau", "master"):
            if k in b:
                st[k] = b[k][off:off + n].view(s)
        groups[decayed].append(p)
        params.append(p)
        held.append(st)
    wd = 4.0 / WD_TS
    cls = adana_amd.DANA_STAR_MK4 if case["optimizer"] == "star" else adana_amd.ADana
    opt = cls([dict(params=ps, weight_decay=wd if d else 0.0) for d, ps in groups.items() if ps],
              use_foreach=case["foreach"], master_weights=case["state"] == "master",
              numerics="eager" if case["eager"] else "compiled", **_hyper(case))
    for p, st in zip(params, held):
        opt.state[p] = st
    return {"case": case, "opt": opt, "params": params, "buffers": b}


def run(state):
    case, opt = state["case"], state["opt"]
    if case["path"] == "tau":
        if opt is None:
            largest, smallest = adana_amd.compute_tau_order_statistics(state["taus"][0])
            return {"largest": largest, "smallest": smallest}
        stats = list(adana_amd.extract_tau_statistics(opt).values())
        return {"largest": np.concatenate([s["largest_order_stats"] for s in stats]),
                "smallest": np.concatenate([s["smallest_order_stats"] for s in stats])}
    out = dict(state["buffers"])
    if case["clip"] == "fused":
        out["total_norm"] = opt.clip_grad_norm_(case["max_norm"])
    elif case["clip"] == "call":
        out["total_norm"] = adana_amd.clip_grad_norm_(state["params"], case["max_norm"])
    opt.step()
    if case["log"]:
        out["diagnostics"] = opt.diagnostics_host()[1]
    elif len(state["params"]) <= FEW:
        for i, p in enumerate(state["params"]):
            out["diagnostics%d" % i] = [opt.state[p][k] for k in DIAG]
    return out


def tolerance(case):
    """Selected values are the tensors' own.  Steps, about four times the error
    against 64 bits: float32 1e-7 to 2.5e-7; with bfloat16 storage 2.2e-3 (single
    values half a unit of 8 significant bits per pass, 4e-3)."""
    if case["path"] == "tau":
        return "exact"
    if case["state"] == "fp32":
        return {"rel": 1e-6, "max": 4e-6}
    return {"rel": 9e-3, "max": 2e-2}


@functools.lru_cache(maxsize=None)
def _ranks(n):
    """Positions read from a sorted tau of n values (both ends)."""
    k = int(np.ceil(np.log(n) / np.log(1.1)))
    return np.minimum(np.unique(np.int32(1.1 ** np.arange(k + 1)) - 1), n - 1)


def exact(case, seed):
    b, lay = _inputs(case, seed)
    if case["path"] == "tau":
        large, small = [], []
        for off, s, _ in lay:
            n = math.prod(s)
            x = torch.sort(b["tau"][off:off + n])[0]
            at = torch.from_numpy(_ranks(n).astype(np.int64)).to(x.device)
            small.append(x[at].double())
            large.append(x[n - 1 - at].double())
        return {"largest": torch.cat(large), "smallest": torch.cat(small)}
    star, master = case["optimizer"] == "star", "master" in b
    t = case["start"] + 1
    a, expo = DELTA / (DELTA + t), 1.0 - case["kappa"]
    sums = torch.zeros(len(lay), 4, dtype=torch.float64, device="cuda")
    coef, out = 1.0, {}
    if case["clip"] != "none":
        sq = torch.zeros((), dtype=torch.float64, device="cuda")
        for off, s, _ in lay:
            sq += b["g"][off:off + math.prod(s)].double().square().sum()
        out["total_norm"] = sq.sqrt()
        coef = min(1.0, case["max_norm"] / (float(sq.sqrt()) + 1e-6))
    names = ["p", "m", "v"] + (["tau"] if star else []) + (["master"] if master else [])
    new = {k: b[k].double() for k in names}        # padding stays as it is
    if case["clip"] != "none":
        new["g"] = b["g"].double()
    for i, (off, s, decayed) in enumerate(lay):
        n = math.prod(s)
        for lo in range(off, off + n, 1 << 26):
            cut = slice(lo, min(lo + (1 << 26), off + n))
            g = b["g"][cut].double() * coef
            m = new["m"][cut]
            m = m + a * (g - m)
            v = (1.0 - a) * new["v"][cut] + a * g * g
            root = v.sqrt()
            if star:
                tau = new["tau"][cut]
                tau = tau + a * (g.abs() / (g.abs() + root + EPS) - tau)
                half = tau.clamp(max=0.5)
                reg = (half / (1.0 - half)).clamp(min=1.0 / (1.0 + t))
                nt = reg.sqrt() / (root + EPS)
                mfac = m.abs() * nt / reg
                af = (tau * t).clamp(min=1.0) ** expo * mfac
                new["tau"][cut] = tau
            else:
                reg = 1.0
                nt = 1.0 / (root + EPS)
                mfac = m.abs() * nt
                af = (1.0 + t) ** expo * mfac
            if case["clipsnr"]:
                af = af.clamp(max=case["clipsnr"])
            src = new["master" if master else "p"][cut]
            wdf = -(4.0 / WD_TS if decayed else 0.0) / (1.0 + t / WD_TS)
            p = (src - LR * (g * nt + (m.sign() * reg * af + m * nt))) * (1.0 + wdf)
            new["m"][cut], new["v"][cut], new["p"][cut] = m, v, p
            if master:
                new["master"][cut] = p
            if "g" in new:
                new["g"][cut] = g
            sums[i] += torch.stack([af.sum(), g.square().sum(), mfac.sum(), m.square().sum()])
    out.update(new)
    out.setdefault("g", None)                      # unchanged without a clip
    count = torch.tensor([math.prod(s) for _, s, _ in lay], dtype=torch.float64, device="cuda")
    mean_af, mean_mfac = sums[:, 0] / count, sums[:, 2] / count
    diag = torch.stack([mean_af, sums[:, 1].sqrt(), mean_mfac, mean_af / mean_mfac, sums[:, 3].sqrt()], 1)
    if case["log"]:
        out["diagnostics"] = diag
    elif len(lay) <= FEW:
        for i in range(len(lay)):
            out["diagnostics%d" % i] = list(diag[i])
    return out
