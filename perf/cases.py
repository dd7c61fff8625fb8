"""Measured cases of the library: the calls a pricing, risk or calibration program makes.

A case is a dict of plain values; ``kind`` names the entry point:

  dropin            calculate_exposure_multi_gpu, the reference's own call: everything from
                    the market to the EE profile in one call
  reference         a ReferencePlan kept by the program; a pass is one ``execute``
  greeks            cva_greeks: CVA and its sensitivities in one call
  portfolio         a PortfolioPlan kept by the program; a pass is one ``execute``
  portfolio_greeks  portfolio_cva_greeks: the book's CVA and sensitivities in one call
  calibration       calibrate_pca over rolling windows of a curve history

The seed of ``prepare`` moves the curve, the loadings, the deal terms, the book and the
generator's key. Results of FP32 runs are returned in single precision, the precision they
are computed in (the float overload of the drop-in returns that by itself); FP64 results in
double. ``exact`` states the same quantities with torch in 64 bits, from the published
Philox4x32-10 and the library's documented stream layout on.
"""
import math

import numpy as np
import torch

import cva_hjm_cuda_amd as hjm

TENORS, STRIDE, DT, DTAU = 51, 50, 0.01, 0.5
EXACT_PATH_STEPS = 1.0e9   # beyond this exact() would take too long


def listed():
    return [
        # the reference's recorded CPU run (5000 scenarios, 25y) through its own call: a
        # program ported as it is, one call per curve
        dict(name="dropin_f64_5000x25y", kind="dropin", paths=5000, expiry=25.0, fp64=True),
        # the reference driver's default, -scenarios 100000 over 25y, float overload
        dict(name="dropin_f32_100000x25y", kind="dropin", paths=100000, expiry=25.0, fp64=False),
        # the smallest configuration, 1000 paths of a 5y swap in FP64: an interactive quote
        dict(name="quote_f64_1000x5y", kind="reference", paths=1000, expiry=5.0, fp64=True,
             quantile=0.975),
        # an ordinary quote in FP32, an odd number of paths
        dict(name="quote_f32_10007x10y", kind="reference", paths=10007, expiry=10.0, fp64=False,
             quantile=0.975),
        # the benchmark's headline: 131072 paths x 1000 steps, FP32 compensated
        dict(name="headline_f32_131072x10y", kind="reference", paths=131072, expiry=10.0,
             fp64=False, quantile=0.975),
        # the same in FP64, the API's default precision
        dict(name="headline_f64_131072x10y", kind="reference", paths=131072, expiry=10.0,
             fp64=True, quantile=0.975),
        # CVA + 204 Greeks of one deal at the adjoint configuration's size
        dict(name="greeks_f32_65536x10y", kind="greeks", paths=65536, expiry=10.0, fp64=False),
        # a desk's small book, odd sizes throughout
        dict(name="book_f32_57x11_10007", kind="portfolio", swaps=57, sets=11, paths=10007,
             horizon=30.0, fp64=False, quantile=0.975, graph=False),
        # the batched configuration, replayed as a graph as the benchmark does
        dict(name="batched_f32_256x32_262144", kind="portfolio", swaps=256, sets=32, paths=262144,
             horizon=30.0, fp64=False, quantile=0.975, graph=True),
        # the full configuration: the largest forward run
        dict(name="full_f32_1024x128_1048576", kind="portfolio", swaps=1024, sets=128,
             paths=1048576, horizon=30.0, fp64=False, quantile=0.975, graph=False),
        # CVA + 204 Greeks of the full book at the path count its FP64 check runs
        dict(name="bookgreeks_f32_1024x128_65536", kind="portfolio_greeks", swaps=1024, sets=128,
             paths=65536, horizon=30.0, fp64=False),
        # every 500-day window of ten years of daily curves
        dict(name="calibration_2101x500", kind="calibration", windows=2101, window=500, step=1,
             fit=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dropin", "reference", "reference", "greeks", "portfolio", "portfolio",
                       "portfolio_greeks", "calibration"])
    half_years = lambda lo, hi: 0.5 * rng.randint(int(2 * lo), int(2 * hi))  # noqa: E731
    if kind == "dropin":
        return dict(kind=kind, paths=_log_uniform(rng, 1000, 100000), expiry=half_years(2, 25),
                    fp64=rng.random() < 0.5)
    if kind == "reference":
        return dict(kind=kind, paths=_log_uniform(rng, 500, 262144), expiry=half_years(2, 25),
                    fp64=rng.random() < 0.5, quantile=rng.choice([0.95, 0.975, 0.99]))
    if kind == "greeks":
        return dict(kind=kind, paths=_log_uniform(rng, 1000, 65536), expiry=half_years(2, 15),
                    fp64=rng.random() < 0.25)
    if kind == "calibration":
        window = rng.randint(60, 500)
        return dict(kind=kind, windows=_log_uniform(rng, 20, 2101), window=window,
                    step=rng.choice([1, 1, 5]), fit=rng.random() < 0.5)
    sets = _log_uniform(rng, 3, 128)
    case = dict(kind=kind, swaps=sets * rng.randint(2, 8) + rng.randint(0, 3), sets=sets,
                paths=_log_uniform(rng, 2000, 262144 if kind == "portfolio" else 65536),
                horizon=rng.choice([10.0, 20.0, 30.0]), fp64=rng.random() < 0.25)
    if kind == "portfolio":
        case.update(quantile=rng.choice([0.95, 0.975, 0.99]), graph=rng.random() < 0.5)
    return case


# ---- inputs ---------------------------------------------------------------------------
def _simpson(y):
    """Cumulative Simpson integral on the tenor grid (1/3 rule to even nodes, 3/8 on the last
    three intervals for odd ones, the 3-point quadratic on the first)."""
    h, out = DTAU, np.zeros(TENORS)
    for j in range(1, TENORS):
        if j == 1:
            out[j] = h / 12.0 * (5.0 * y[0] + 8.0 * y[1] - y[2])
            continue
        e = j if j % 2 == 0 else j - 3
        s = sum(h / 3.0 * (y[i] + 4.0 * y[i + 1] + y[i + 2]) for i in range(0, e, 2))
        if j % 2:
            s += 3.0 * h / 8.0 * (y[j - 3] + 3.0 * y[j - 2] + 3.0 * y[j - 1] + y[j])
        out[j] = s
    return out


def _market(rng):
    """A Nelson-Siegel curve and three parametric loadings around the benchmark market's, with
    the HJM drift of the loadings."""
    tau = np.arange(TENORS) * DTAU
    x = tau / rng.uniform(1.6, 2.4)
    b = np.array([0.03, -0.02, 0.01]) * rng.uniform(0.85, 1.15, 3)
    spot = b[0] + b[1] * np.exp(-x) + b[2] * x * np.exp(-x)
    s = rng.uniform(0.9, 1.1, 3)
    vols = np.stack([np.full(TENORS, 0.0064 * s[0]),
                     s[1] * (-0.0036 + 0.0006 * tau - 2e-5 * tau ** 2),
                     s[2] * (-0.0047 + 0.0018 * tau - 1.5e-4 * tau ** 2 + 3e-6 * tau ** 3)])
    drift = sum(v * _simpson(v) for v in vols)
    return spot, drift, vols, np.full(TENORS, 0.5)


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    d = dict(key=int(rng.integers(1, 1 << 40)))
    d["spot"], d["drift"], d["vols"], d["accrual"] = _market(rng)
    kind = case["kind"]
    if kind == "calibration":
        n = (case["windows"] - 1) * case["step"] + case["window"]
        d["curves"] = hjm.synthetic_history(d["vols"], n, seed=int(rng.integers(1 << 30)),
                                            noise=2e-5, base=d["spot"])
    elif kind.startswith("portfolio"):
        pf = hjm.synthetic_portfolio(case["swaps"], case["sets"], seed=int(rng.integers(1 << 30)))
        pf.periods = np.minimum(pf.periods, int(round(case["horizon"] / DTAU))).astype(np.int32)
        d["book"] = pf
    else:
        d["notional"], d["rate"] = 1e6 * rng.uniform(0.5, 2.0), rng.uniform(0.02, 0.03)
        d["hazard"] = rng.uniform(0.01, 0.03)
        if kind == "dropin":
            d["key"] = 1234   # the call's own seed
            d["hazard"] = 0.0
            if not case["fp64"]:
                # the float overload's inputs are floats
                for k in ("spot", "drift", "vols", "accrual"):
                    d[k] = d[k].astype(np.float32)
                d["notional"], d["rate"] = float(np.float32(d["notional"])), float(np.float32(d["rate"]))
    return d


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    state = dict(case=case, **d)
    if kind == "calibration":
        return state
    precision = hjm.FP64 if case["fp64"] else hjm.FP32_KAHAN
    state["precision"] = precision
    if kind == "dropin":
        state["swap"] = hjm.InterestRateSwap(d["notional"], d["rate"], case["expiry"])
        state["ee"] = np.zeros(TENORS, np.float64 if case["fp64"] else np.float32)
        return state
    state["market"] = hjm.Market(d["spot"], d["drift"], d["vols"], d["accrual"])
    if kind in ("reference", "greeks"):
        state["swap"] = hjm.InterestRateSwap(d["notional"], d["rate"], case["expiry"])
    if kind == "reference":
        state["plan"] = hjm.ReferencePlan(state["market"], state["swap"], case["paths"], DT,
                                          precision=precision, seed=d["key"], hazard=d["hazard"],
                                          pfe_quantile=case["quantile"])
    elif kind == "portfolio":
        state["plan"] = hjm.PortfolioPlan(state["market"], d["book"], case["paths"],
                                          horizon=case["horizon"], dt=DT, precision=precision,
                                          seed=d["key"], pfe_quantile=case["quantile"],
                                          tuning=hjm.Tuning(use_graph=case["graph"]))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "calibration":
        c = hjm.calibrate_pca(state["curves"], window=case["window"], step=case["step"],
                              nwindows=case["windows"], fit_degrees=(0, 2, 3) if case["fit"] else None)
        return dict(eigenvalues=c.eigenvalues, volatilities=c.volatilities, drifts=c.drifts,
                    raw_loadings=c.raw_loadings)
    if kind == "dropin":
        hjm.calculate_exposure_multi_gpu(state["ee"], state["swap"], state["accrual"], state["spot"],
                                         state["drift"], state["vols"].reshape(-1), 1.0, 1,
                                         case["paths"], DT)
        return dict(ee=state["ee"])
    own = np.float64 if case["fp64"] else np.float32
    if kind == "reference":
        p = state["plan"].execute()
        return dict(ee=p.ee.astype(own), pfe=p.pfe.astype(own), cva=p.cva.astype(own),
                    cva_stderr=p.se.astype(own))
    if kind == "portfolio":
        r = state["plan"].execute()
        return dict(ee=r.expected_exposure.astype(own), pfe=r.pfe.astype(own), cva=r.cva.astype(own),
                    cva_stderr=r.cva_stderr.astype(own))
    if kind == "greeks":
        g = hjm.cva_greeks(state["market"], state["swap"], case["paths"], DT,
                           precision=state["precision"], seed=state["key"], hazard=state["hazard"])
    else:
        g = hjm.portfolio_cva_greeks(state["market"], state["book"], case["paths"],
                                     horizon=case["horizon"], dt=DT, precision=state["precision"],
                                     seed=state["key"])
    return dict(cva=np.array([g.cva]).astype(own), d_spot=g.d_spot.astype(own),
                d_vol=g.d_vol.astype(own), d_drift=g.d_drift.astype(own),
                d_vol_total=g.d_vol_total.astype(own))


def work(case):
    """Bytes: the inputs read and the results written once. Operations: the Euler steps' (51
    tenors of subtraction, 4 FMAs, addition and accumulation; 5 FMAs and a short-rate sum for
    the portfolio), the reverse sweep's (per tenor 3 gradient FMAs and the 2 of the transposed
    step), the valuation's FMAs, the covariances' and one orthogonal reduction's."""
    market = 8 * (3 * TENORS + 3 * TENORS)
    kind = case["kind"]
    if kind == "calibration":
        w, n = case["windows"], (case["windows"] - 1) * case["step"] + case["window"]
        return dict(bytes=8 * TENORS * n + 8 * w * TENORS * (1 + 3 + 1 + 3),
                    flops=w * (case["window"] * TENORS * (TENORS + 1) + 9 * TENORS ** 3))
    p = case["paths"]
    if kind.startswith("portfolio"):
        dates = int(round(case["horizon"] / DTAU)) + 1
        steps = STRIDE * (dates - 1)
        fl = p * (512 * steps + dates * case["sets"] * dates)
        if kind == "portfolio_greeks":
            fl += p * (10 * TENORS * steps + dates * case["sets"] * dates)
            return dict(bytes=market + 8 * (1 + 2 * TENORS + 6 * TENORS), flops=fl)
        return dict(bytes=market + 16 * case["sets"] * (dates + 1), flops=fl)
    steps = int(round(case["expiry"] / DT)) - STRIDE
    fl = 561 * p * steps
    if kind == "greeks":
        fl += 10 * TENORS * p * steps
        return dict(bytes=market + 8 * (1 + 2 * TENORS + 6 * TENORS), flops=fl)
    return dict(bytes=market + 8 * (2 * TENORS + 2), flops=fl)


# ---- the same quantities in 64 bits -----------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


_LOW = 0xFFFFFFFF


def _block_normals(key, block, ids):
    """Shocks [50][3][paths] of one date block: class g = s % 4 of step s draws from the stream
    (path, block, g); call c of a stream is one Philox4x32-10 block with counter (block, path,
    g, c), whose four words are two Box-Muller pairs, shocks 4c .. 4c + 3; shock 3q + k of a
    stream is factor k of the class's q-th step."""
    dev = ids.device
    shape = (4, 10, ids.numel())
    c0 = torch.full(shape, block, dtype=torch.int64, device=dev)
    c1 = ids.view(1, 1, -1).expand(shape)
    c2 = torch.arange(4, device=dev).view(4, 1, 1).expand(shape)
    c3 = torch.arange(10, device=dev).view(1, 10, 1).expand(shape)
    k0, k1 = key & _LOW, (key >> 32) & _LOW
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = (((p1 >> 32) & _LOW) ^ c1 ^ k0, p1 & _LOW, ((p0 >> 32) & _LOW) ^ c3 ^ k1,
                          p0 & _LOW)
        k0, k1 = (k0 + 0x9E3779B9) & _LOW, (k1 + 0xBB67AE85) & _LOW

    def pair(a, b):
        u = (a.to(torch.float32).double() * 2.0 ** -32 + 2.0 ** -33).to(torch.float32).double()
        t = b.to(torch.float32).double() * (2.0 ** -32 * 2.0 * math.pi)
        r = torch.sqrt(-2.0 * torch.log(u))
        return r * torch.cos(t), r * torch.sin(t)

    z = torch.stack(pair(c0, c1) + pair(c2, c3), dim=2).reshape(4, 40, -1)
    z = z[:, :39].reshape(4, 13, 3, -1).permute(1, 0, 2, 3).reshape(52, 3, -1)
    return z[:STRIDE]


class _Steps:
    """Euler steps of the forward curve [51][paths] and their transpose."""

    def __init__(self, d, dev):
        t = lambda a: torch.as_tensor(np.asarray(a, np.float64), device=dev)  # noqa: E731
        self.drift = t(d["drift"]).view(-1, 1) * DT
        self.vols = t(d["vols"]).T.contiguous() * math.sqrt(DT)
        self.spot = t(d["spot"])
        self.c = DT / DTAU

    def forward(self, f, z):
        g = torch.empty_like(f)
        torch.sub(f[1:], f[:-1], out=g[:-1])
        g[-1] = f[-1] - f[-2]
        return f + self.c * g + self.drift + self.vols @ z

    def transposed(self, lam):
        out = (1.0 - self.c) * lam
        out[1:] += self.c * lam[:-1]
        out[-1] += 2.0 * self.c * lam[-1]
        out[-2] -= self.c * lam[-1]
        return out


def _weights(hazard, recovery, n):
    w = np.zeros(n)
    for i in range(1, n):
        pd = math.exp(-hazard * (i - 1) * DTAU) - math.exp(-hazard * i * DTAU)
        w[i - 1] += 0.5 * (1.0 - recovery) * pd
        w[i] += 0.5 * (1.0 - recovery) * pd
    return w


def _stderr(x):
    n = x.shape[-1]
    return torch.sqrt(x.var(dim=-1, unbiased=True) / n) if n > 1 else torch.zeros_like(x[..., 0])


def _kth(rows, q):
    n = rows.shape[-1]
    k = min(max(int(math.ceil(q * n)), 1), n)
    return torch.sort(rows, dim=-1).values[..., k - 1]


def _reference_paths(case, d, dev):
    """Numeraire pairs x, y [dates + 1][paths] (slot 0 unused) of the reference semantics."""
    ids = torch.arange(case["paths"], dtype=torch.int64, device=dev)
    dates = int(round(case["expiry"] / DTAU))
    st = _Steps(d, dev)
    f = st.spot.view(-1, 1).repeat(1, case["paths"])
    a = STRIDE * f
    x, y = torch.zeros((2, dates + 1, case["paths"]), dtype=torch.float64, device=dev)
    x[1], y[1] = f[1], torch.exp(-a[1] * DT)
    for b in range(1, dates):
        z = _block_normals(d["key"], b, ids)
        for s in range(STRIDE):
            f = st.forward(f, z[s])
            a += f
        x[b + 1], y[b + 1] = f[b + 1], torch.exp(-a[b + 1] * DT)
    return st, ids, dates, x, y


def _cash_flows(d, x, y, dates):
    m = 1.0 / DTAU
    acc = torch.as_tensor(np.asarray(d["accrual"], np.float64), device=x.device)[: dates + 1].view(-1, 1)
    base = y * d["notional"] * acc
    cf = base * (m * (torch.exp(x / m) - 1.0) - d["rate"])
    v = torch.flip(torch.cumsum(torch.flip(cf[1:], [0]), 0), [0])   # V_t, t = 0 .. dates - 1
    return base, cf, v


def _exact_reference(case, d):
    dev = _device()
    _, _, dates, x, y = _reference_paths(case, d, dev)
    _, _, v = _cash_flows(d, x, y, dates)
    e = torch.clamp(v, min=0.0)
    ee = np.zeros(TENORS)
    ee[:dates] = e.mean(dim=1).cpu().numpy()
    if case["kind"] == "dropin":
        return dict(ee=ee)
    w = _weights(d["hazard"], 0.4, TENORS)
    pfe = np.zeros(TENORS)
    pfe[:dates] = _kth(e, case["quantile"]).cpu().numpy()
    per_path = torch.as_tensor(w[:dates], device=dev) @ e
    return dict(ee=ee, pfe=pfe, cva=np.array([float(w @ ee)]),
                cva_stderr=np.array([float(_stderr(per_path))]))


def _with_drift(d, dv, dm):
    """d_vol plus the drift's share through the cumulative Simpson drift of the loadings."""
    unit = np.stack([_simpson(e) for e in np.eye(TENORS)])   # [l][j]
    out = dv.copy()
    for k, s in enumerate(np.asarray(d["vols"], np.float64)):
        out[k] += dm * _simpson(s) + unit @ (dm * s)
    return out


def _sensitivities(d, cva, ds, dv, dm):
    return dict(cva=np.array([cva]), d_spot=ds, d_vol=dv.reshape(-1), d_drift=dm,
                d_vol_total=_with_drift(d, dv, dm).reshape(-1))


def _exact_greeks(case, d):
    dev = _device()
    st, ids, dates, x, y = _reference_paths(case, d, dev)
    base, cf, v = _cash_flows(d, x, y, dates)
    n = case["paths"]
    w = _weights(d["hazard"], 0.4, TENORS)
    wt = torch.as_tensor(w[:dates], device=dev).view(-1, 1)
    u = torch.cumsum(wt * (v > 0), 0)                 # u[i - 1]: the weight of cash flow i
    gx = torch.zeros_like(x)
    ga = torch.zeros_like(x)
    gx[1:] = u * base[1:] * torch.exp(x[1:] * DTAU)
    ga[1:] = -u * DT * cf[1:]
    lam = torch.zeros((TENORS, n), dtype=torch.float64, device=dev)
    mu = torch.zeros_like(lam)
    dv = torch.zeros((3, TENORS), dtype=torch.float64, device=dev)
    dm = torch.zeros(TENORS, dtype=torch.float64, device=dev)
    for b in range(dates - 1, 0, -1):
        lam[b + 1] += gx[b + 1] + ga[b + 1]
        mu[b + 1] += ga[b + 1]
        z = _block_normals(d["key"], b, ids)
        for s in range(STRIDE - 1, -1, -1):
            dv += z[s] @ lam.T
            dm += lam.sum(dim=1)
            lam = st.transposed(lam) + mu
    spot = lam + (STRIDE - 1) * mu
    spot[1] += gx[1] + STRIDE * ga[1]
    cva = float((wt * torch.clamp(v, min=0.0)).sum() / n)
    host = lambda t: (t / n).cpu().numpy()  # noqa: E731
    return _sensitivities(d, cva, host(spot.sum(dim=1)), math.sqrt(DT) * host(dv), DT * host(dm))


def _book_tables(pf, date, dates):
    """Set values at a date as a - gamma P: [sets], [sets][dates - 1]."""
    a, gam = np.zeros(pf.nsets), np.zeros((pf.nsets, dates - 1))
    for n, s, k, g in zip(pf.periods - date, pf.sign_notional, pf.fixed_rate, pf.set_of):
        if n > 0:
            a[g] += s
            gam[g, n - 1] += s
            gam[g, :n] += s * k * pf.dtau
    return a, gam


def _bonds(f, periods):
    """P(t, t + k dtau), k = 1 .. periods, from the trapezoid integral, flat past the grid."""
    inc = 0.5 * DTAU * (f[1:] + f[:-1])
    if periods > TENORS - 1:
        inc = torch.cat([inc, DTAU * f[-1:].expand(periods - TENORS + 1, -1)])
    return torch.exp(-torch.cumsum(inc[:periods], 0))


def _book_dates(case, d, dev):
    """(date, curve [51][paths], log bank account [paths]) at every date."""
    ids = torch.arange(case["paths"], dtype=torch.int64, device=dev)
    st = _Steps(d, dev)
    f = st.spot.view(-1, 1).repeat(1, case["paths"])
    lnb = torch.zeros(case["paths"], dtype=torch.float64, device=dev)
    dates = int(round(case["horizon"] / DTAU)) + 1
    for e in range(dates):
        yield e, f, lnb
        if e + 1 < dates:
            z = _block_normals(d["key"], e, ids)
            lnb = lnb.clone()
            for s in range(STRIDE):
                lnb += f[0] * DT
                f = st.forward(f, z[s])


def _exact_portfolio(case, d):
    dev, pf = _device(), d["book"]
    dates = int(round(case["horizon"] / DTAU)) + 1
    w = torch.as_tensor(np.stack([_weights(h, 0.4, dates) for h in pf.hazard]), device=dev)
    ee, pfe = np.zeros((2, pf.nsets, dates))
    per_path = torch.zeros((pf.nsets, case["paths"]), dtype=torch.float64, device=dev)
    for e, f, lnb in _book_dates(case, d, dev):
        a, gam = (torch.as_tensor(t, device=dev) for t in _book_tables(pf, e, dates))
        v = a.view(-1, 1) - gam @ _bonds(f, dates - 1)
        x = torch.clamp(v, min=0.0) * torch.exp(-lnb)
        ee[:, e] = x.mean(dim=1).cpu().numpy()
        pfe[:, e] = _kth(x, case["quantile"]).cpu().numpy()
        per_path += w[:, e].view(-1, 1) * x
    return dict(ee=ee, pfe=pfe, cva=(w.cpu().numpy() * ee).sum(axis=1),
                cva_stderr=_stderr(per_path).cpu().numpy())


def _exact_portfolio_greeks(case, d):
    dev, pf = _device(), d["book"]
    n, periods = case["paths"], int(round(case["horizon"] / DTAU))
    dates = periods + 1
    w = torch.as_tensor(np.stack([_weights(h, 0.4, dates) for h in pf.hazard]), device=dev)
    cva, gbar, beta = 0.0, [], []
    for e, f, lnb in _book_dates(case, d, dev):
        a, gam = (torch.as_tensor(t, device=dev) for t in _book_tables(pf, e, dates))
        bonds, disc = _bonds(f, periods), torch.exp(-lnb)
        v = a.view(-1, 1) - gam @ bonds
        u = w[:, e].view(-1, 1) * (v > 0) * disc
        beta.append(-(u * v).sum(dim=0))
        cva -= float(beta[-1].sum()) / n
        iota = bonds * (gam.T.contiguous() @ u)                  # dJ / d integral to period k
        suffix = torch.flip(torch.cumsum(torch.flip(iota, [0]), 0), [0])
        g = torch.zeros((TENORS, n), dtype=torch.float64, device=dev)
        inside = min(periods, TENORS - 1)
        g[:inside] += 0.5 * DTAU * suffix[:inside]
        g[1: inside + 1] += 0.5 * DTAU * suffix[:inside]
        if periods > inside:
            g[-1] += DTAU * suffix[inside:].sum(dim=0)
        gbar.append(g)
    st, ids = _Steps(d, dev), torch.arange(n, dtype=torch.int64, device=dev)
    lam = gbar[-1]
    mu = torch.zeros(n, dtype=torch.float64, device=dev)
    dv = torch.zeros((3, TENORS), dtype=torch.float64, device=dev)
    dm = torch.zeros(TENORS, dtype=torch.float64, device=dev)
    for e in range(dates - 2, -1, -1):
        mu = mu + DT * beta[e + 1]
        z = _block_normals(d["key"], e, ids)
        for s in range(STRIDE - 1, -1, -1):
            dv += z[s] @ lam.T
            dm += lam.sum(dim=1)
            lam = st.transposed(lam)
            lam[0] += mu
        lam += gbar[e]
    host = lambda t: (t / n).cpu().numpy()  # noqa: E731
    return _sensitivities(d, cva, host(lam.sum(dim=1)), math.sqrt(DT) * host(dv), DT * host(dm))


def _exact_calibration(case, d):
    diffs = np.diff(d["curves"], axis=0)
    n, step, nd = case["windows"], case["step"], case["window"] - 1
    cov = np.stack([np.cov(diffs[i * step: i * step + nd], rowvar=False) for i in range(n)]) * 252.0
    ev, vec = np.linalg.eigh(cov)
    ev, vec = ev[:, ::-1], vec[:, :, ::-1]
    raw = np.transpose(vec[:, :, :3], (0, 2, 1)) * np.sqrt(ev[:, :3, None])
    raw = raw * np.where(raw.sum(axis=2, keepdims=True) > 0, 1.0, -1.0)
    vols = raw.copy()
    if case["fit"]:
        x = np.arange(TENORS) / (TENORS - 1.0)
        for k, deg in enumerate((0, 2, 3)):
            basis = np.vander(x, deg + 1)
            vols[:, k] = raw[:, k] @ (basis @ np.linalg.pinv(basis)).T
    unit = np.stack([_simpson(e) for e in np.eye(TENORS)])
    drifts = (vols * (vols @ unit)).sum(axis=1)
    flat = lambda a: np.ascontiguousarray(a.reshape(n, -1))  # noqa: E731
    return dict(eigenvalues=np.ascontiguousarray(ev), volatilities=flat(vols), drifts=drifts,
                raw_loadings=flat(raw))


def exact(case, seed):
    kind = case["kind"]
    d = _inputs(case, seed)
    if kind == "calibration":
        return _exact_calibration(case, d)
    steps = case["horizon" if kind.startswith("portfolio") else "expiry"] / DT
    if case["paths"] * steps > EXACT_PATH_STEPS:
        return None
    return {"dropin": _exact_reference, "reference": _exact_reference, "greeks": _exact_greeks,
            "portfolio": _exact_portfolio, "portfolio_greeks": _exact_portfolio_greeks}[kind](case, d)
