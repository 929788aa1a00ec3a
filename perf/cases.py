"""Workloads that time this package's transforms through its public Python calls.

A case is a dict of plain values: `op` names the call or pair of calls, `L`
and `lmax` the grid and truncation degrees, `n` the upper index, `real` the
value kind, `batch` the fields per call and `precision` the arithmetic mode.
`listed()` gives the fixed cases, `draw()` others of the same ranges;
`prepare()`, `run()`, `work()` and `exact()` build, execute, cost and verify
one.  The arithmetic behind `exact()` is plain numpy and torch in 64 bits.
"""
import math

import numpy as np
import torch

import gshtrans_amd as G
from gshtrans_amd.autograd import synthesize

NMAX = 2


def listed():
    return [
        # One small complex field there and back, outputs allocated by the
        # calls: a low-degree model evaluated inside a program's inner loop.
        dict(name="single_l64", op="roundtrip", L=64, lmax=64, n=0, real=False, batch=1,
             precision="fp64", keep=False),
        # One complex field for each upper index -2 .. 2: the canonical
        # components of a tensor field, each a call of its own.
        dict(name="components_l512", op="components", L=512, lmax=512, n=0, real=False, batch=1,
             precision="fp64", keep=True),
        # Three scalar fields on a grid of odd degree whose ring length is not
        # a power of two: a model given at a degree of its author's choice.
        dict(name="scalar_l301", op="roundtrip", L=301, lmax=301, n=0, real=True, batch=3,
             precision="fp64", keep=True),
        # Expansion of sampled data of ordinary resolution: analysis only,
        # white noise on a smooth field, ring length 2000.
        dict(name="data_l1000", op="analysis", L=1000, lmax=1000, n=2, real=False, batch=6,
             precision="fp64", keep=True),
        # The residual and gradient of a least-squares fit of 16 fields.
        dict(name="fit_l512", op="gradient", L=512, lmax=512, n=1, real=False, batch=16,
             precision="fp64", keep=False),
        # Products of two expansions of degree 256 on a grid of degree 384
        # (3/2 of it, so the product does not alias).
        dict(name="product_l384", op="product", L=384, lmax=256, n=1, real=False, batch=8,
             precision="fp64", keep=False),
        # Evaluation of an ordinary batch of scalar fields below the grid's
        # degree, FP32 products.
        dict(name="maps_l512_fp32", op="synthesis", L=512, lmax=400, n=0, real=True, batch=24,
             precision="fp32", keep=True),
        # Spin-one fields in the split modes at a degree of no special form.
        dict(name="mixed_l360", op="roundtrip", L=360, lmax=360, n=-1, real=False, batch=20,
             precision="bf16x3", keep=True),
        # The headline workload's two batches in FP64 ...
        dict(name="scalars_l1024", op="roundtrip", L=1024, lmax=1024, n=0, real=True, batch=64,
             precision="fp64", keep=True),
        dict(name="spin2_l1024", op="roundtrip", L=1024, lmax=1024, n=2, real=False, batch=64,
             precision="fp64", keep=True),
        # ... and both in one step in its headline mode.
        dict(name="headline_bf16x6", op="headline", L=1024, lmax=1024, n=2, real=False, batch=64,
             precision="bf16x6", keep=True),
        # 256 fields of uneven degree and upper index as one replayed plan.
        dict(name="plan_256", op="plan", L=1024, lmax=1024, n=0, real=False, batch=256,
             precision="fp64", keep=True, storage="fp32", lo=32),
    ]


def draw(rng):
    op = rng.choice(["roundtrip", "roundtrip", "synthesis", "analysis", "gradient", "product",
                     "components", "plan"])
    top = 512 if op == "plan" else 1024
    L = int(round(math.exp(rng.uniform(math.log(24), math.log(top)))))
    if rng.random() < 0.35:
        L = 1 << min(10, max(5, int(round(math.log2(L)))))
        L = min(L, top)
    lmax = L if rng.random() < 0.6 else max(8, int(L * rng.uniform(0.5, 1.0)))
    n = rng.choice([0, 0, 1, -1, 2, -2])
    real = rng.random() < (0.6 if n == 0 else 0.1)
    precision = rng.choice(["fp64"] * 6 + ["bf16x6", "bf16x6", "bf16x3", "fp32"])
    batch = int(round(math.exp(rng.uniform(0.0, math.log(64)))))
    batch = max(1, min(batch, int(40 * (1024 / L) ** 3)))
    case = dict(op=op, L=L, lmax=lmax, n=n, real=real, batch=batch, precision=precision,
                keep=rng.random() < 0.5)
    if op == "components":
        case.update(n=0, real=False, precision="fp64", batch=min(batch, 4), keep=True)
    elif op == "product":
        case.update(n=0 if real else rng.choice([0, 1, -1]))
    elif op == "gradient":
        case.update(precision="fp64", keep=False)
    elif op == "plan":
        case.update(n=0, lmax=L, real=real, precision=rng.choice(["fp64", "fp64", "bf16x6"]),
                    batch=rng.randint(9, 96), storage=rng.choice(["fp32", "fp64"]),
                    lo=max(4, L // 16), keep=True)
    return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed):
    g = torch.Generator(device=_device())
    g.manual_seed(int(seed))
    return g


def _csize(lmax, n, real):
    na = abs(n)
    if real:
        return (lmax + 1) * (lmax + 2) // 2 - na * (na + 1) // 2
    return (lmax + 1) ** 2 - na * na


def _degrees_orders(lmax, n, real):
    """Degree and order of every coefficient, in the order of the layout."""
    l = np.repeat(np.arange(abs(n), lmax + 1),
                  [(i + 1 if real else 2 * i + 1) for i in range(abs(n), lmax + 1)])
    first = np.concatenate([[0], np.cumsum(np.bincount(l, minlength=lmax + 1))])[l]
    m = np.arange(l.size) - first - (0 if real else l)
    return torch.from_numpy(l).to(_device()), torch.from_numpy(m).to(_device())


def _coefficients(seed, L, lmax, n, real, batch):
    """Normal coefficients of (l + 1)^-1 decay with the masks of the
    reference's generator (GSHTrans/src/GridBase.h:115-172)."""
    l, m = _degrees_orders(lmax, n, real)
    c = torch.randn((batch, l.numel()), dtype=torch.complex128, device=_device(),
                    generator=_generator(seed))
    c *= math.sqrt(2.0) / (l + 1.0)
    if real:
        c.imag[:, m == 0] = 0.0
        if lmax == L:
            c.imag[:, -1] = 0.0
    elif lmax == L:
        c[:, -1] = 0.0
    return c


def _samples(seed, L, real, batch):
    """Sampled data: a dozen smooth waves and white noise of a tenth of their size."""
    g = _generator(seed)
    dev = _device()
    th = torch.linspace(0.0, math.pi, L + 1, dtype=torch.float64, device=dev)
    ph = torch.arange(2 * L, dtype=torch.float64, device=dev) * (math.pi / L)
    k = torch.arange(12, device=dev)
    a = torch.randn((batch, L + 1, 12), dtype=torch.complex128, device=dev, generator=g) * 0.02
    a += torch.randn((batch, 1, 12), dtype=torch.complex128, device=dev, generator=g) * \
        torch.cos(th[:, None] * (k + 1))
    f = torch.matmul(a.reshape(-1, 12), torch.exp(1j * k[:, None] * ph)).reshape(batch, L + 1, -1)
    f += 0.1 * torch.randn(f.shape, dtype=torch.complex128, device=dev, generator=g)
    return f.real.contiguous() if real else f


def _plan_fields(case, seed):
    """Degrees (log-uniform), upper indices and coefficients of a plan's fields."""
    rng = np.random.default_rng(case["L"] * 1000 + case["batch"])
    lmax = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["L"]), case["batch"]))
    lmax = np.clip(np.rint(lmax).astype(int), case["lo"], case["L"])
    n = rng.integers(-NMAX, NMAX + 1, case["batch"])
    sizes = [_csize(int(a), int(b), case["real"]) for a, b in zip(lmax, n)]
    dtype = torch.complex64 if case["storage"] == "fp32" else torch.complex128
    c = torch.zeros((case["batch"], max(sizes)), dtype=dtype, device=_device())
    for i, s in enumerate(sizes):
        c[i, :s] = _coefficients(seed * 4096 + i, case["L"], int(lmax[i]), int(n[i]),
                                 case["real"], 1)[0]
    return lmax, n, sizes, c


def _inputs(case, seed):
    """The tensors that a case's calls read."""
    op, L, lmax, n = case["op"], case["L"], case["lmax"], case["n"]
    real, batch = case["real"], case["batch"]
    if op == "components":
        return {"c": [_coefficients(seed * 8 + k, L, lmax, k - NMAX, False, batch)
                      for k in range(2 * NMAX + 1)]}
    if op == "headline":
        return {"cr": _coefficients(2 * seed, L, lmax, 0, True, batch),
                "cc": _coefficients(2 * seed + 1, L, lmax, n, False, batch)}
    if op == "product":
        return {"u": _coefficients(2 * seed, L, lmax, n, real, batch),
                "v": _coefficients(2 * seed + 1, L, lmax, n, real, batch)}
    if op == "plan":
        return dict(zip(("lmax", "n", "sizes", "c"), _plan_fields(case, seed)))
    d = {}
    if op != "analysis":
        d["c"] = _coefficients(2 * seed, L, lmax, n, real, batch)
    if op in ("analysis", "gradient"):
        d["f"] = _samples(2 * seed + 1, L, real, batch)
    return d


# ---------------------------------------------------------------------------
# The calls
# ---------------------------------------------------------------------------
def prepare(case, seed):
    L = case["L"]
    s = dict(_inputs(case, seed), case=case, grid=G.GaussLegendreGrid(L, NMAX))
    op, n, real, batch = case["op"], case["n"], case["real"], case["batch"]
    need = {"components": range(-NMAX, NMAX + 1), "headline": (0, n), "product": (n, 2 * n),
            "plan": sorted(set(int(k) for k in s["n"])) if op == "plan" else ()}
    for k in need.get(op, (n,)):
        s["grid"].prepare(k)
    if op == "plan":
        s["plan"] = G.BatchPlan(s["grid"], s["lmax"], s["n"], real=real,
                                precision=case["precision"], storage=case["storage"])

    def field(r, b=batch, dtype=None):
        dtype = dtype or (torch.float64 if r else torch.complex128)
        return torch.zeros((b, L + 1, 2 * L), dtype=dtype, device="cuda")

    if case["keep"]:  # outputs that the program keeps from call to call
        if op == "components":
            s["fo"] = [field(False) for _ in s["c"]]
            s["co"] = [torch.zeros_like(c) for c in s["c"]]
        elif op == "headline":
            s.update(fr=field(True), fc=field(False), or_=torch.zeros_like(s["cr"]),
                     oc=torch.zeros_like(s["cc"]))
        elif op == "plan":
            s.update(fo=field(real, dtype=s["plan"].field_dtype()), co=torch.zeros_like(s["c"]))
        elif op != "product":
            s["fo"] = field(real) if op != "analysis" else None
            s["co"] = torch.zeros((batch, _csize(case["lmax"], n, real)), dtype=torch.complex128,
                                  device="cuda") if op != "synthesis" else None
    if op == "gradient":
        s["c"].requires_grad_(True)
    return s


def run(s):
    case, g = s["case"], s["grid"]
    op, lmax, n = case["op"], case["lmax"], case["n"]
    kw = dict(real=case["real"], precision=case["precision"])
    if op == "roundtrip":
        f = g.inverse(lmax, n, s["c"], field=s.get("fo"), **kw)
        return {"field": f, "coeffs": g.forward(lmax, n, f, coeffs=s.get("co"), **kw)}
    if op == "synthesis":
        return {"field": g.inverse(lmax, n, s["c"], field=s.get("fo"), **kw)}
    if op == "analysis":
        return {"coeffs": g.forward(lmax, n, s["f"], coeffs=s.get("co"), **kw)}
    if op == "gradient":
        f = synthesize(g, lmax, n, s["c"], **kw)
        r = f - s["f"]
        return {"residual": r.detach(), "gradient": torch.autograd.grad(f, s["c"], r.detach())[0]}
    if op == "product":
        return {"coeffs": g.product(lmax, s["u"], n, s["v"], n, **kw)}
    if op == "components":
        for k, c in enumerate(s["c"]):
            g.inverse(lmax, k - NMAX, c, field=s["fo"][k])
            g.forward(lmax, k - NMAX, s["fo"][k], coeffs=s["co"][k])
        return {"field": s["fo"], "coeffs": s["co"]}
    if op == "headline":
        p = case["precision"]
        g.inverse(lmax, 0, s["cr"], field=s["fr"], real=True, precision=p)
        g.forward(lmax, 0, s["fr"], coeffs=s["or_"], real=True, precision=p)
        g.inverse(lmax, n, s["cc"], field=s["fc"], real=False, precision=p)
        g.forward(lmax, n, s["fc"], coeffs=s["oc"], real=False, precision=p)
        return {"field_r": s["fr"], "coeffs_r": s["or_"], "field_c": s["fc"], "coeffs_c": s["oc"]}
    s["plan"].inverse(s["c"], field=s["fo"], graph=True)
    s["plan"].forward(s["fo"], coeffs=s["co"], graph=True)
    return {"field": s["fo"], "coeffs": s["co"]}


# ---------------------------------------------------------------------------
# Costs
# ---------------------------------------------------------------------------
def _transform(L, lmax, n, real, batch):
    """Operations of one batched transform, fewest known: the Legendre sums
    (over half the colatitudes for upper index 0, by parity) and ring FFTs."""
    nt, N = L + 1, 2 * L
    leg = 4.0 * ((nt + 1) // 2 if n == 0 else nt) * _csize(lmax, n, real)
    return batch * (leg + 5.0 * N * math.log2(N) * nt * (0.5 if real else 1.0))


def work(case):
    op, L, lmax, n = case["op"], case["L"], case["lmax"], case["n"]
    real, batch = case["real"], case["batch"]
    field = (L + 1) * 2 * L * (8.0 if real else 16.0) * batch
    co = 16.0 * _csize(lmax, n, real) * batch
    one = _transform(L, lmax, n, real, batch)
    if op == "roundtrip":
        return {"bytes": 2 * (field + co), "flops": 2 * one}
    if op in ("synthesis", "analysis"):
        return {"bytes": field + co, "flops": one}
    if op == "gradient":
        return {"bytes": 3 * field + 2 * co, "flops": 2 * one}
    if op == "product":
        return {"bytes": 3 * co, "flops": 2 * one + _transform(L, lmax, 2 * n, real, batch)}
    if op == "components":
        ks = range(-NMAX, NMAX + 1)
        return {"bytes": sum(2 * (field + 16.0 * _csize(lmax, k, False) * batch) for k in ks),
                "flops": sum(2 * _transform(L, lmax, k, False, batch) for k in ks)}
    if op == "headline":
        cr = 16.0 * _csize(lmax, 0, True) * batch
        return {"bytes": 2 * (field + field / 2 + co + cr),
                "flops": 2 * (one + _transform(L, lmax, 0, True, batch))}
    rng = np.random.default_rng(L * 1000 + batch)
    lm = np.exp(rng.uniform(math.log(case["lo"]), math.log(L), batch))
    lm = np.clip(np.rint(lm).astype(int), case["lo"], L)
    ns = rng.integers(-NMAX, NMAX + 1, batch)
    half = 0.5 if case["storage"] == "fp32" else 1.0
    return {"bytes": half * 2 * (field + sum(16.0 * _csize(int(a), int(b), real)
                                             for a, b in zip(lm, ns))),
            "flops": sum(2 * _transform(L, int(a), int(b), real, 1) for a, b in zip(lm, ns))}


# ---------------------------------------------------------------------------
# Results in plain 64-bit arithmetic
# ---------------------------------------------------------------------------
def _nodes(L):
    """Colatitudes and weights of the (L + 1)-point Gauss-Legendre rule, by
    Newton's method in extended precision."""
    k = np.arange(L + 1)
    x = np.cos(np.pi * (k + 0.75) / (L + 1.5)).astype(np.longdouble)
    for _ in range(6):
        p0, p1 = np.ones_like(x), x.copy()
        for j in range(2, L + 2):
            p0, p1 = p1, ((2 * j - 1) * x * p1 - (j - 1) * p0) / j
        dp = (L + 1) * (x * p1 - p0) / (x * x - 1)
        x = x - p1 / dp
    return np.arccos(x), 2 / ((1 - x * x) * dp * dp)


class _Functions:
    """d^l_{mn}(theta_i) sqrt((2l + 1) / 4 pi) for all l <= lmax and all orders
    (m >= 0 if real): table[order][l][theta], from the closed form at l =
    max(|m|, |n|) and the three-term recurrence over l."""

    def __init__(self, L, lmax, n, real):
        dev = _device()
        self.L, self.lmax, self.n, self.real = L, lmax, n, real
        th, w = _nodes(L)
        self.w = torch.from_numpy((w * (np.longdouble(np.pi) / L)).astype(np.float64)).to(dev)
        m = np.arange(0 if real else -lmax, lmax + 1)
        l0 = np.maximum(np.abs(m), abs(n))
        lg = np.concatenate([[0.0], np.cumsum(np.log(np.arange(1, 2 * lmax + 2,
                                                               dtype=np.longdouble)))])
        # d^{l0}_{mn} = sign sqrt((2 l0)! / ((l0+a)! (l0-a)!)) cos^p sin^q
        # of theta / 2, p = l0 + a', q = l0 - a', a the smaller index.
        a = np.where(np.abs(m) >= abs(n), n, m)
        top = np.where(np.abs(m) >= abs(n), m, n)
        p = np.where(top >= 0, l0 + a, l0 - a)
        q = 2 * l0 - p
        odd = np.where(np.abs(m) >= abs(n), np.where(m >= 0, m - n, 0),
                       np.where(n >= 0, 0, m - n))
        sign = np.where(odd % 2 == 0, 1.0, -1.0)
        c, s = np.log(np.cos(th / 2)), np.log(np.sin(th / 2))
        half = np.longdouble(0.5)
        log = half * (lg[2 * l0] - lg[l0 + a] - lg[l0 - a])[:, None] + p[:, None] * c + \
            q[:, None] * s + half * np.log((2 * l0 + 1) / (4 * np.longdouble(np.pi)))[:, None]
        seed = torch.from_numpy((sign[:, None] * np.exp(log)).astype(np.float64)).to(dev)
        x = torch.from_numpy(np.cos(th).astype(np.float64)).to(dev)
        ll, mm = np.arange(lmax + 1, dtype=np.longdouble)[:, None], m.astype(np.longdouble)
        nn = np.longdouble(n)
        with np.errstate(all="ignore"):
            den = np.sqrt((ll * ll - nn * nn) * (ll * ll - mm * mm))
            A = (2 * ll - 1) * ll / den
            B = np.where(m * n == 0, 0, (2 * ll - 1) * mm * nn / ((ll - 1) * den))
            C = ll * np.sqrt(((ll - 1) ** 2 - nn * nn) * ((ll - 1) ** 2 - mm * mm)) / \
                ((ll - 1) * den)
            r1 = np.sqrt((2 * ll + 1) / (2 * ll - 1))
            r2 = np.sqrt((2 * ll + 1) / (2 * ll - 3))
            A, B, C = A * r1, B * r1, np.where(ll >= l0 + 2, C * r2, 0)
        live = ll > l0
        A, B, C = (torch.from_numpy(np.where(live, v, 0).astype(np.float64)).to(dev)[:, :, None]
                   for v in (A, B, C))
        start = torch.from_numpy(l0).to(dev)[:, None]
        self.table = torch.empty((m.size, lmax + 1, th.size), dtype=torch.float64, device=dev)
        e0 = torch.zeros_like(seed)
        e1 = torch.zeros_like(seed)
        for l in range(lmax + 1):
            e = (A[l] * x - B[l]) * e0 - C[l] * e1
            e = torch.where(start == l, seed, e)
            self.table[:, l] = e
            e1, e0 = e0, e
        l, k = _degrees_orders(lmax, n, real)
        self.at = (k - int(m[0])) * (lmax + 1) + l
        self.m = torch.from_numpy(m).to(dev)

    def synthesis(self, c):
        b, M, N = c.shape[0], self.m.numel(), 2 * self.L
        dense = torch.zeros((M * (self.lmax + 1), b), dtype=torch.complex128, device=c.device)
        dense[self.at] = c.to(torch.complex128).T
        dense = torch.view_as_real(dense).reshape(M, self.lmax + 1, 2 * b)
        F = torch.bmm(self.table.transpose(1, 2).contiguous(), dense)
        del dense
        F = torch.view_as_complex(F.reshape(M, -1, b, 2)).permute(2, 1, 0)
        if self.real:
            X = torch.zeros((b, self.L + 1, self.L + 1), dtype=torch.complex128, device=c.device)
            X[:, :, :M] = F
            X.imag[:, :, 0] = 0.0
            X.imag[:, :, self.L] = 0.0
            return torch.fft.irfft(X, n=N, norm="forward")
        X = torch.zeros((b, self.L + 1, N), dtype=torch.complex128, device=c.device)
        X[:, :, :self.lmax + 1] += F[:, :, self.lmax:]
        X[:, :, N - self.lmax:] += F[:, :, :self.lmax]
        return torch.fft.ifft(X, norm="forward")

    def analysis(self, f, adjoint=False):
        b, M = f.shape[0], self.m.numel()
        if self.real:
            X = torch.fft.rfft(f.to(torch.float64))
            if adjoint:
                X *= 2.0
                X[:, :, 0] = X[:, :, 0].real / 2
                X[:, :, self.L] = X[:, :, self.L].real / 2
        else:
            X = torch.fft.fft(f.to(torch.complex128))
        X = X[:, :, self.m % (2 * self.L)]
        if not adjoint:
            X = X * self.w[:, None]
        X = torch.view_as_real(X.permute(2, 1, 0).contiguous()).reshape(M, -1, 2 * b)
        c = torch.bmm(self.table, X)
        c = torch.view_as_complex(c.reshape(M * (self.lmax + 1), b, 2))[self.at].T.contiguous()
        if not adjoint and not self.real and self.lmax == self.L:
            c[:, -1] = 0.0
        return c


def exact(case, seed):
    op, L, lmax, n = case["op"], case["L"], case["lmax"], case["n"]
    real = case["real"]
    d = _inputs(case, seed)
    if op in ("roundtrip", "synthesis"):
        t = _Functions(L, lmax, n, real)
        f = t.synthesis(d["c"])
        return {"field": f} if op == "synthesis" else {"field": f, "coeffs": t.analysis(f)}
    if op == "analysis":
        return {"coeffs": _Functions(L, lmax, n, real).analysis(d["f"])}
    if op == "gradient":
        t = _Functions(L, lmax, n, real)
        r = t.synthesis(d["c"]) - d["f"]
        return {"residual": r, "gradient": t.analysis(r, adjoint=True)}
    if op == "product":
        t = _Functions(L, lmax, n, real)
        f = t.synthesis(d["u"]) * t.synthesis(d["v"])
        return {"coeffs": _Functions(L, lmax, 2 * n, real).analysis(f)}
    if op == "components":
        out = {"field": [], "coeffs": []}
        for k, c in enumerate(d["c"]):
            t = _Functions(L, lmax, k - NMAX, False)
            out["field"].append(t.synthesis(c))
            out["coeffs"].append(t.analysis(out["field"][-1]))
        return out
    if op == "headline":
        t = _Functions(L, lmax, 0, True)
        out = {"field_r": t.synthesis(d["cr"])}
        out["coeffs_r"] = t.analysis(out["field_r"])
        t = _Functions(L, lmax, n, False)
        out["field_c"] = t.synthesis(d["cc"])
        out["coeffs_c"] = t.analysis(out["field_c"])
        return out
    # A plan: by upper index, each field's coefficients widened to the group's degree.
    ftype = (torch.float64 if real else torch.complex128)
    out = {"field": torch.zeros((case["batch"], L + 1, 2 * L), dtype=ftype, device=_device()),
           "coeffs": torch.zeros(d["c"].shape, dtype=torch.complex128, device=_device())}
    for k in sorted(set(int(v) for v in d["n"])):
        own = [i for i in range(case["batch"]) if int(d["n"][i]) == k]
        top = max(int(d["lmax"][i]) for i in own)
        t = _Functions(L, top, k, real)
        c = torch.zeros((len(own), _csize(top, k, real)), dtype=torch.complex128, device=_device())
        for j, i in enumerate(own):
            c[j, :d["sizes"][i]] = d["c"][i, :d["sizes"][i]]
        f = t.synthesis(c)
        back = t.analysis(f)
        for j, i in enumerate(own):
            out["field"][i] = f[j]
            out["coeffs"][i, :d["sizes"][i]] = back[j, :d["sizes"][i]]
        del t
    return out
