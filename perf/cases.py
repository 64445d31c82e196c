"""The work that users of holodeck_amd have it do, as cases that can be timed and compared.

``listed()`` holds the fixed cases, ``draw(rng)`` makes more of the same ranges.  A case is a dict
of plain values whose ``"kind"`` names the path:

gwb       parameters -> model -> loud sources and background (``Semi_Analytic_Model.gwb``)
sample    one sample of a parameter-space library (``librarian.run_model``)
evolve    binary evolution, bin integration and strain on device arrays (``engine``)
scatter   M-Mbulge scatter of a binary density (``scatter.add_scatter_to_masses_device``)
counts    loud-source walk over given counts (``engine.realize``)
eccen     harmonic sums of an eccentric population (``cyutils.sam_calc_gwb_single_eccen``)
discrete  the same with Poisson counts (``cyutils.sam_calc_gwb_single_eccen_discrete``)
predict   surrogate inference (``surrogate.MLPSurrogate.predict``)
fit       surrogate training, one epoch (``surrogate.MLPSurrogate.fit``)
"""
import os

import numpy as np
import torch

import holodeck_amd as holo
from holodeck_amd import _lib, configs, cyutils, engine, librarian, scatter, surrogate, utils
from holodeck_amd import device as D
from holodeck_amd.constants import GYR, MSOL, PC, YR
from holodeck_amd.sams.components import density_params

DATA = os.path.join(os.path.dirname(holo.__file__), "data")
WEIGHTS = {"classic": "surrogate_classic_uniform_91x81x101_f30_r500.npz",
           "eccen": "surrogate_eccen_classic_61x51x61_f40_h100.npz"}
DURATION = 16.03 * YR    # PTA duration; the frequencies are its harmonics


def listed():
    return [
        # a first look at a GW-driven model on a coarse grid: every stage is a handful of blocks
        dict(name="gwb coarse GW-driven", kind="gwb", hard="gw", M=17, Q=15, Z=13, F=6, R=64, L=3, params=False),
        # the GW-driven workload with the loud sources' and background's parameters
        dict(name="gwb 61x51x41 parameters", kind="gwb", hard="gw", M=61, Q=51, Z=41, F=20, R=100, L=5, params=True),
        # the flagship spectrum: full grid, 2PL 500 realizations, 10 loudest
        dict(name="gwb 91x81x101 full", kind="gwb", hard="2pl", M=91, Q=81, Z=101, F=40, R=500, L=10, params=False),
        # a library sample at an uneven grid: split and independent Poisson background
        dict(name="sample 67x59x83", kind="sample", M=67, Q=59, Z=83, F=30, R=100, L=5),
        # the deterministic half of the flagship spectrum, resident on the device
        dict(name="evolve 91x81x101", kind="evolve", M=91, Q=81, Z=101, F=40),
        # scatter of the full-size density
        dict(name="scatter 91x81x101", kind="scatter", M=91, Q=81, Z=101),
        # given counts (a comparison with another sampler's draws)
        dict(name="counts 61x51x41", kind="counts", M=61, Q=51, Z=41, F=20, R=50, L=5, mode="sorted"),
        # one spectrum of the eccentric library
        dict(name="eccen 61x51x61", kind="eccen", M=61, Q=51, Z=61, F=40, H=100, E=123, e0=0.5),
        # realizations of an eccentric population
        dict(name="discrete 41x31x41", kind="discrete", M=41, Q=31, Z=41, F=20, H=30, E=123, R=100, e0=0.5),
        # one step of a sampler that holds 64 walkers
        dict(name="predict 64", kind="predict", net="classic", rows=64, width=0, layers=0, outs=0),
        # a whole prior volume at once
        dict(name="predict 100000", kind="predict", net="classic", rows=100000, width=0, layers=0, outs=0),
        # an epoch over a small library
        dict(name="fit 4096", kind="fit", rows=4096, batch=1024, width=256, layers=4, outs=90),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["gwb", "gwb", "sample", "evolve", "scatter", "counts", "eccen", "discrete", "predict", "fit"])
    grid = dict(M=rng.randint(13, 91), Q=rng.randint(11, 81), Z=rng.randint(9, 101))
    if kind == "gwb":
        return dict(kind=kind, hard=rng.choice(["gw", "2pl"]), **grid, F=rng.randint(3, 40), R=_log_int(rng, 20, 500),
                    L=rng.choice([1, 3, 5, 10]), params=rng.random() < 0.3)
    if kind == "sample":
        return dict(kind=kind, M=rng.randint(41, 91), Q=rng.randint(41, 81), Z=rng.randint(41, 101),
                    F=rng.randint(20, 40), R=rng.randint(50, 200), L=rng.choice([1, 5, 10]))
    if kind == "evolve":
        return dict(kind=kind, **grid, F=rng.randint(3, 40))
    if kind == "scatter":
        return dict(kind=kind, **grid)
    if kind == "counts":
        return dict(kind=kind, M=rng.randint(13, 61), Q=rng.randint(11, 51), Z=rng.randint(9, 41), F=rng.randint(3, 20),
                    R=_log_int(rng, 5, 50), L=rng.choice([1, 3, 5, 10]), mode=rng.choice(["sorted", "argmax", "none"]))
    if kind == "eccen":
        return dict(kind=kind, M=rng.randint(13, 61), Q=rng.randint(11, 51), Z=rng.randint(9, 61), F=rng.randint(3, 40),
                    H=_log_int(rng, 10, 100), E=rng.randint(60, 150), e0=round(rng.uniform(0.05, 0.9), 3))
    if kind == "discrete":
        return dict(kind=kind, M=rng.randint(11, 41), Q=rng.randint(9, 31), Z=rng.randint(9, 41), F=rng.randint(3, 20),
                    H=_log_int(rng, 6, 30), E=rng.randint(60, 150), R=_log_int(rng, 10, 100),
                    e0=round(rng.uniform(0.1, 0.9), 3))
    if kind == "predict":
        net = rng.choice(["classic", "eccen", "fresh"])
        fresh = net == "fresh"
        return dict(kind=kind, net=net, rows=_log_int(rng, 1, 100000), width=rng.choice([64, 128, 256]) if fresh else 0,
                    layers=rng.randint(1, 4) if fresh else 0, outs=3 * rng.randint(5, 40) if fresh else 0)
    return dict(kind=kind, rows=_log_int(rng, 300, 4096), batch=rng.choice([128, 256, 512, 1024]),
                width=rng.choice([64, 128, 256]), layers=rng.randint(2, 4), outs=3 * rng.randint(5, 40))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _spec(case, rng, hard):
    """Model specification of a case: the benchmark's components with parameters from the seed."""
    make = configs.spec_config2 if hard == "2pl" else configs.spec_config1
    s = make(shape=(case["M"], case["Q"], case["Z"]), nfreq=case.get("F", 20))
    s["gsmf"]["phi0"] += rng.uniform(-0.3, 0.3)
    s["mmbulge"]["mamp_log10"] += rng.uniform(-0.2, 0.2)
    s["gmt"]["time_norm"] *= rng.uniform(0.7, 1.3)
    if hard == "2pl":
        s["hard"]["time"] = rng.uniform(0.5, 5.0) * GYR
    return s


def _cosmo(spec):
    cos = holo.Cosmology(h=spec["cosmo"]["h"], Om0=spec["cosmo"]["Om0"])
    cos.device_tables()
    return cos


def _static(spec, cos):
    """Device grids and static density (no scatter) of a specification."""
    sam = configs.make_sam(spec, scatter=0.0, cosmo=cos)
    par = density_params(sam._gsmf, sam._gpf, sam._gmt, sam._gmr, sam._mmbulge, cos)
    grids = [D.to_dev(g) for g in sam.edges]
    dens, zprime, gmt = engine.static_density(*grids, par, cos)
    return sam, grids, dens, zprime, gmt


def _peters_evolution(e0, a0, a1, num):
    """Separations from a0 to a1 and the GW-driven eccentricities along them (Peters 1964, Eq. 5.11)."""
    ee = e0 * 10.0 ** np.linspace(-16.0, 0.0, 40000)
    la = np.log(ee ** (12 / 19) / (1 - ee**2) * (1 + 121 / 304 * ee**2) ** (870 / 2299))
    sepa = np.logspace(np.log10(a0), np.log10(a1), num)
    return sepa, np.exp(np.interp(np.log(sepa / a0) + la[-1], la, np.log(ee)))


def _eccen_inputs(case, seed):
    """Host arrays of the eccentric entry points: a Schechter-like density that fades with redshift."""
    rng = np.random.default_rng([seed, 5])
    mtot = np.logspace(4, 12, case["M"]) * MSOL
    mrat = np.logspace(-3, 0, case["Q"])
    redz = np.logspace(-3, 1, case["Z"])
    lm = np.log10(mtot / MSOL)[:, None, None]
    q, z = mrat[None, :, None], redz[None, None, :]
    knee, slope = rng.uniform(8.2, 9.0), rng.uniform(0.2, 0.5)
    ndens = 10 ** (rng.uniform(-3.5, -2.5) - slope * (lm - 8)) * np.exp(-(10 ** (lm - knee)))
    ndens = ndens * q ** rng.uniform(-0.3, 0.3) * (1 + z) ** 0.5 * np.exp(-z / rng.uniform(1.0, 2.5))
    ndens = np.where(z > rng.uniform(5.0, 8.0), 0.0, ndens)     # mergers that stall past today
    zz = np.linspace(0.0, 10.5, 20001)
    ez = 1.0 / np.sqrt(0.31 * (1 + zz) ** 3 + 0.69)
    dcom = np.concatenate([[0.0], np.cumsum(0.5 * (ez[1:] + ez[:-1]) * np.diff(zz))]) * 299792.458 / 67.7
    sepa, eccen = _peters_evolution(case["e0"], PC, 3 * 2.953e5 * 1e4, case["E"])
    fobs = np.arange(1, case["F"] + 1) / DURATION
    return ndens, np.log10(mtot), mrat, redz, np.interp(redz, zz, dcom), fobs, sepa, eccen


def _net(case, seed):
    if case.get("net") in WEIGHTS:
        return surrogate.MLPSurrogate.load(os.path.join(DATA, WEIGHTS[case["net"]]))
    return surrogate.MLPSurrogate(n_in=6, hidden=(case["width"],) * case["layers"], n_out=case["outs"], seed=seed % 997)


def _train_set(case, seed):
    """Parameters in the unit box and smooth log10 spectra of them, falling with frequency."""
    rng = np.random.default_rng([seed, 7])
    X = rng.random((case["rows"], 6))
    freq = np.linspace(0.0, 1.5, case["outs"])[None, :]
    Y = -14.5 + X @ rng.uniform(-0.6, 0.6, (6, 1)) - (0.67 + 0.2 * X[:, :1]) * freq
    return X, Y + 0.2 * np.sin(3 * X[:, 1:2] + freq) + 0.02 * rng.standard_normal(Y.shape[:1] + (1,))


def _count_inputs(case, seed):
    """Bins' strains and Poisson counts on the device, lambda over many decades and mostly below one."""
    B, F, R = (case["M"] - 1) * (case["Q"] - 1) * (case["Z"] - 1), case["F"], case["R"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    mass = torch.rand(B, 1, generator=gen, device="cuda", dtype=torch.float64)
    freq = torch.arange(1, F + 1, device="cuda", dtype=torch.float64)[None, :]
    lam = 10.0 ** (3.0 - 9.0 * mass) * freq ** (-8.0 / 3.0)
    noise = torch.rand(B, F, generator=gen, device="cuda", dtype=torch.float64)
    h2fdf = 1e-36 * 10.0 ** (9.0 * mass) * freq ** (4.0 / 3.0) * (0.5 + noise)
    counts = torch.poisson(lam[:, :, None].expand(B, F, R).contiguous(), generator=gen)
    return lam, h2fdf, counts


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng([seed, 3])
    if kind == "gwb":
        spec = _spec(case, rng, case["hard"])
        return dict(case=case, spec=spec, cosmo=_cosmo(spec), edges=configs.fobs_gw_edges(spec), seed=seed)
    if kind == "sample":
        space = librarian.PS_Classic_Phenom_Uniform(sam_shape=(case["M"], case["Q"], case["Z"]))
        return dict(case=case, space=space, params=space.normalized_params(0.1 + 0.8 * rng.random(6)), seed=seed)
    if kind == "evolve":
        spec = _spec(case, rng, "2pl")
        cos = _cosmo(spec)
        sam, grids, dens, zprime, gmt = _static(spec, cos)
        engine.zero_stalled(dens, zprime)
        orb = configs.fobs_gw_edges(spec) / 2.0
        cents, width = utils.midpoints(orb), np.diff(orb)
        return dict(case=case, cosmo=cos, hard=configs.make_hard(spec, sam), grids=grids, dens=dens, gmt=gmt,
                    fobs=D.to_dev(cents), dlnf=D.to_dev(np.diff(np.log(orb))), fcdf=D.to_dev(cents / width),
                    log10_mtot=D.to_dev(np.log10(sam.mtot)), mt_cent=D.to_dev(utils.midpoints(sam.mtot)),
                    mr_cent=D.to_dev(utils.midpoints(sam.mrat)))
    if kind == "scatter":
        spec = _spec(case, rng, "2pl")
        sam, _, dens, _, _ = _static(spec, _cosmo(spec))
        return dict(case=case, mtot=sam.mtot, mrat=sam.mrat, dens=dens, scatter=rng.uniform(0.1, 0.6))
    if kind == "counts":
        lam, h2fdf, counts = _count_inputs(case, seed)
        order = engine.order_desc(h2fdf, col=0) if case["mode"] == "sorted" else None
        return dict(case=case, number=lam, h2fdf=h2fdf, counts=counts, order=order)
    if kind in ("eccen", "discrete"):
        return dict(case=case, args=_eccen_inputs(case, seed), seed=seed)
    net = _net(case, seed)
    if kind == "predict":
        X = net.x_lo + (net.x_hi - net.x_lo) * rng.random((case["rows"], net.sizes[0]))
        return dict(case=case, net=net, X=X)
    X, Y = _train_set(case, seed)
    return dict(case=case, net=net, X=X, Y=Y, seed=seed)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
MODES = {"sorted": _lib.HD_SEL_SORTED, "argmax": _lib.HD_SEL_ARGMAX, "none": _lib.HD_SEL_NONE}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gwb":
        sam = configs.make_sam(state["spec"], cosmo=state["cosmo"])
        hard = configs.make_hard(state["spec"], sam)
        return sam.gwb(state["edges"], hard=hard, realize=case["R"], loudest=case["L"], params=case["params"],
                       seed=state["seed"])
    if kind == "sample":
        sam, hard = state["space"].model_for_params(state["params"])
        out = librarian.run_model(sam, hard, nfreqs=case["F"], nreals=case["R"], nloudest=case["L"], seed=state["seed"])
        return {key: out[key] for key in ("hc_ss", "hc_bg", "gwb")}
    if kind == "evolve":
        hard, (mtot, mrat, redz), cos = state["hard"], state["grids"], state["cosmo"]
        rf, dn = engine.dbn_2pwl(state["fobs"], True, hard._sepa_init, hard._num_steps, hard._norm_dev, hard._rchar,
                                 hard._gamma_inner, hard._gamma_outer, state["dens"], mtot, mrat, redz, state["gmt"], cos)
        number = engine.integrate_3dx1d(state["log10_mtot"], mrat, redz, state["dlnf"], dn)
        h2fdf = engine.h2fdf_redz(state["mt_cent"], state["mr_cent"], state["fobs"], state["fcdf"], rf, cos)
        return rf, dn, number, h2fdf
    if kind == "scatter":
        dens = state["dens"].clone()      # the call works in place
        sweeps = scatter.add_scatter_to_masses_device(state["mtot"], state["mrat"], dens, state["scatter"])
        return dens, sweeps
    if kind == "counts":
        hc2ss, ssidx, hc2bg, _ = engine.realize(state["number"], state["h2fdf"], case["R"], case["L"],
                                                MODES[case["mode"]], order=state["order"], counts=state["counts"])
        return hc2ss, ssidx, hc2bg
    if kind == "eccen":
        return cyutils.sam_calc_gwb_single_eccen(*state["args"], nharms=case["H"])
    if kind == "discrete":
        return cyutils.sam_calc_gwb_single_eccen_discrete(*state["args"], case["H"], case["R"], seed=state["seed"])
    net = state["net"]
    if kind == "predict":
        return net.predict(state["X"])
    loss = net.fit(state["X"], state["Y"], epochs=1, batch=case["batch"], lr=1e-3, seed=state["seed"] % 1009)
    return dict(loss=loss.astype(np.float32), W=list(net.W), b=list(net.b))


def work(case):
    """Bytes: inputs read and outputs written once.  Flops: the operations of the method itself."""
    kind = case["kind"]
    if kind in ("predict", "fit"):
        sizes = {"classic": [6, 256, 256, 256, 256, 90], "eccen": [7, 256, 256, 256, 256, 120]}.get(case.get("net"))
        sizes = sizes or [6] + [case["width"]] * case["layers"] + [case["outs"]]
        weights = sum(a * b + b for a, b in zip(sizes[:-1], sizes[1:]))
        if kind == "predict":
            return dict(bytes=8.0 * case["rows"] * (sizes[0] + sizes[-1]) + 2.0 * weights, flops=2.0 * case["rows"] * weights)
        seen = case["rows"] // case["batch"] * case["batch"] or case["rows"]
        steps = max(1, case["rows"] // case["batch"])
        return dict(bytes=8.0 * seen * (6 + case["outs"]) + 24.0 * weights * steps, flops=6.0 * seen * weights)
    M, Q, Z = case["M"], case["Q"], case["Z"]
    nodes, bins = M * Q * Z, (M - 1) * (Q - 1) * (Z - 1)
    smooth = 2.0 * (4 * M) ** 3 * Z               # the scatter's matrix product
    if kind == "scatter":
        return dict(bytes=16.0 * nodes, flops=smooth)
    F = case["F"]
    steps = 150.0 * nodes * F                     # evolution, integration and strain of one (node, frequency)
    if kind == "evolve":
        return dict(bytes=16.0 * nodes + 16.0 * F * (nodes + bins), flops=steps)
    if kind == "eccen":
        # two Bessel values by a backward recurrence from just above the harmonic, then closed forms
        terms = float(M * Z * F * case["H"])
        return dict(bytes=8.0 * (nodes + F * case["H"]), flops=terms * (4.0 * (case["H"] / 2 + 20) + 100.0))
    if kind == "discrete":
        cols = F * case["H"]
        return dict(bytes=8.0 * (nodes + cols * case["R"]), flops=10.0 * nodes * cols * case["R"])
    R, L = case["R"], case["L"]
    if kind == "counts":
        loud = 0 if case["mode"] == "none" else 16.0 * F * R * L
        return dict(bytes=8.0 * bins * F * (R + 1) + 8.0 * F * R + loud, flops=2.0 * bins * F * R)
    # a dense draw (a word and a search) for about one cell in six and realization
    draws = 30.0 * bins * F * R / 6
    out = 8.0 * F * R * (1 + L)
    if kind == "sample":
        return dict(bytes=out + 8.0 * F * R, flops=smooth + steps + 2 * draws)
    return dict(bytes=out + (8.0 * F * R * (7 + 4 * L) if case["params"] else 0.0), flops=smooth + steps + draws)


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain numpy and torch
# ---------------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "counts":
        return _exact_counts(case, seed)
    if kind == "eccen":
        return _exact_eccen(case, seed)
    if kind == "predict":
        net = prepare(case, seed)["net"]
        rng = np.random.default_rng([seed, 3])
        x01 = torch.from_numpy(rng.random((case["rows"], net.sizes[0])))
        y = x01.cuda()
        for k, (W, b) in enumerate(zip(net.W, net.b)):
            y = y @ W.double().T + b.double()
            y = torch.nn.functional.silu(y) if k < len(net.W) - 1 else y
        return y.cpu().numpy() * net.y_std + net.y_mean
    if kind == "fit":
        return _exact_fit(case, seed)
    return None        # draws of the library's own streams, or a chain of its own stages


def _exact_counts(case, seed):
    """The first L instances of the bins in order of strain; the rest is background."""
    lam, h, counts = _count_inputs(case, seed)
    (B, F, R), L = counts.shape, case["L"]
    ss = torch.zeros(F, R, L, dtype=torch.float64, device=h.device)
    idx = torch.full((F, R, L), -1, dtype=torch.int64, device=h.device)
    bg = torch.zeros(F, R, dtype=torch.float64, device=h.device)
    for f in range(F):
        bg[f] = (counts[:, f] * h[:, f, None]).sum(0)
        if case["mode"] == "none":
            continue
        order = torch.sort(h[:, 0 if case["mode"] == "sorted" else f], descending=True, stable=True).indices
        total = counts[order, f].cumsum(0).T.contiguous()
        at = torch.searchsorted(total, torch.arange(1.0, L + 1, dtype=torch.float64, device=h.device).expand(R, L).contiguous())
        have = at < B
        bins = order[at.clamp(max=B - 1)]
        idx[f] = torch.where(have, bins, -1)
        ss[f] = torch.where(have, h[:, f][bins], 0.0)
        bg[f] -= ss[f].sum(1)
    if case["mode"] == "none":
        return ss[..., :0], idx[..., :0], bg
    return ss, idx, bg


def _exact_eccen(case, seed):
    """Sum over masses, ratios and redshifts of the harmonic strain; Bessel functions by their integral."""
    G, C, MPC = 6.6742999e-08, 29979245800.0, 3.08567758e24
    ndens, lm, mrat, redz, dcom, fobs, sepa, eccen = (torch.from_numpy(np.asarray(a)).cuda() for a in _eccen_inputs(case, seed))
    H, F = case["H"], case["F"]

    def width(g):
        w = torch.empty_like(g)
        w[1:-1] = 0.5 * (g[2:] - g[:-2])
        w[0], w[-1] = 0.5 * (g[1] - g[0]), 0.5 * (g[-1] - g[-2])
        return w

    mt = (10.0**lm)[:, None]
    q = mrat[None, :]
    m1 = mt / (1 + q)
    m2 = mt - m1
    mc = mt * q**0.6 / (1 + q) ** 1.2
    gsrc = 8 * G ** (5 / 3) * np.pi ** (2 / 3) / np.sqrt(10) / C**4
    per_q = (gsrc * mc * (2 * mc) ** (2 / 3)) ** 2 / (m1 * m2 * mt) * width(mrat)[None, :]
    pair = torch.einsum("iqz,iq->iz", ndens, per_q) * width(lm)[:, None] * width(redz)[None, :]
    pair = pair * (4 * np.pi * C / MPC) * dcom**2 * (1 + redz) / (dcom * MPC) ** 2
    pref = np.sqrt(G) / (2 * np.pi) / sepa**1.5
    tau = (torch.arange(160 + 2 * H, device="cuda", dtype=torch.float64) + 0.5) * np.pi / (160 + 2 * H)
    out = torch.zeros(F, H, dtype=torch.float64, device="cuda")
    for n in range(1, H + 1):
        fr = fobs[None, None, :] * (1 + redz)[None, :, None] / n
        x = (fr / mt.sqrt()[:, :, None]).contiguous()
        ok = (x >= pref[0]) & (x <= pref[-1]) & (pair[:, :, None] != 0)
        ii, zz, ff = ok.nonzero(as_tuple=True)
        if not len(ii):
            continue
        x, fr = x[ok], fr.expand(ok.shape)[ok]
        e = (torch.searchsorted(pref, x) - 1).clamp(0, len(pref) - 2)
        ecc = eccen[e] + (x - pref[e]) * (eccen[e + 1] - eccen[e]) / (pref[e + 1] - pref[e])
        J = []
        for k in range(n - 2, n + 3):
            J.append(torch.cat([torch.cos(k * tau - (n * p)[:, None] * torch.sin(tau)).mean(1) for p in ecc.split(1 << 16)]))
        aa = J[0] - 2 * ecc * J[1] + 2 / n * J[2] + 2 * ecc * J[3] - J[4]
        bb = J[0] - 2 * ecc * J[2] + J[4]
        g = n**4 / 32 * (aa**2 + (1 - ecc**2) * bb**2 + 4 / (3 * n**2) * J[2] ** 2)
        g = torch.where(ecc < 1e-12, 1.0 if n == 2 else 0.0, g)
        Fe = (1 + 73 / 24 * ecc**2 + 37 / 96 * ecc**4) / (1 - ecc**2) ** 3.5
        a4 = (G / (2 * np.pi) ** 2 * mt[ii, 0] / fr**2) ** (4 / 3)
        A = a4 / (64 * G**3 / 5 / C**5 * Fe) * g * (4 / n**2) * fr ** (4 / 3)
        out[:, n - 1].index_add_(0, ff, A * pair[ii, zz])
    return out


def _exact_fit(case, seed):
    """One epoch of Adam on the mean squared error of the standardised targets."""
    net = _net(case, seed)
    X, Y = _train_set(case, seed)
    x_lo, x_hi = X.min(0), X.max(0)
    X = torch.from_numpy((X - x_lo) / (x_hi - x_lo)).cuda()
    Y = torch.from_numpy((Y - Y.mean(0)) / np.maximum(Y.std(0), 1e-6)).cuda()
    par = [p.double().clone().requires_grad_() for p in [*net.W, *net.b]]
    n = len(net.W)
    opt = torch.optim.Adam(par, lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
    rows, batch = case["rows"], case["batch"]
    perm = torch.randperm(rows, generator=torch.Generator(device="cpu").manual_seed(seed % 1009)).cuda()
    losses = []
    for s in range(0, rows - batch + 1 if rows >= batch else 1, batch):
        at = perm[s:s + batch]
        y = X[at]
        for k in range(n):
            y = y @ par[k].T + par[n + k]
            y = torch.nn.functional.silu(y) if k < n - 1 else y
        loss = ((y - Y[at]) ** 2).mean()
        opt.zero_grad()
        loss.backward()
        opt.step()
        losses.append(float(loss))
    par = [p.detach() for p in par]
    return dict(loss=np.array([np.mean(losses)]), W=par[:n], b=par[n:])
