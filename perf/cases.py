"""Performance cases: the calls a user of optifax_amd makes, over the sizes,
directions, precisions and options they are made with.

Kinds (all through the package's public entry points):
  pass     OPOmexBatch: one crystal pass on host arrays, the call that
           OpticalSim.run makes once per round trip through the MEX gateway
  ring     OPOBatch: one device-resident round trip of one cavity
  batch    OPOBatch: one round trip of many uneven cavities in one launch
  fibre    gnlsefib / gnlse_batch: fibre GNLSE solves
  qpm      zsum: the mismatch sums of a phase-matching gain map
  forward  SurrogateMLP.forward: inference on host rows
  grads    SurrogateMLP.gradients: loss and parameter gradients
  train    SurrogateMLP.train: Adam steps on an uploaded set, then get_params

`listed()` names the cases that are tracked, `draw(rng)` takes another one
from the same ranges.  `exact(case, seed)` is the same result in plain numpy
or torch at 64 bits.
"""
import math

import numpy as np
import torch

from optifax_amd import fibre
from optifax_amd import physics as ph
from optifax_amd import qpm
from optifax_amd.solver import Context, OPOBatch, OPOmexBatch
from optifax_amd.surrogate import SurrogateMLP, layer_shapes

_AREA = math.pi * (50e-6) ** 2


def listed():
    return [
        # one pass of a thin crystal on a small grid: the quick check and the
        # parameter scan, where a step's latency is everything
        dict(name="pass_512", kind="pass", n=512, window_ps=3.0, length_um=300, period_um=30.0,
             energy_nj=0.2, area_um2=20.0, batch=1, method="heun", precision="single", plots=5),
        # a single SHG/OPG pass with the third-order solver at tight tolerance
        dict(name="pass_rk23_8192", kind="pass", n=8192, window_ps=10.0, length_um=200,
             period_um=30.0, energy_nj=0.1, area_um2=5.0, batch=1, method="rk23",
             precision="single", plots=5),
        # three fields at once in FP64: the accurate mode of the solver handle
        dict(name="pass_f64_2048x3", kind="pass", n=2048, window_ps=6.0, length_um=400,
             period_um=29.5, energy_nj=0.2, area_um2=20.0, batch=3, method="heun",
             precision="double", plots=4),
        # the ring OPO of the headline benchmark: one round trip from noise
        dict(name="ring_32768", kind="ring", n=32768, window_ps=12.0, length_um=5000,
             period_um=30.5, energy_nj=2.0, fwhm_fs=200, delay_fs=300.0, sync=False, band=False,
             fixed=False, method="heun", precision="single"),
        # a detuned 8 mm-type cavity (here 1 mm) solved to its steady state in
        # FP64 with fixed steps, as the warm-start study does
        dict(name="ring_f64_16384", kind="ring", n=16384, window_ps=16.0, length_um=1000,
             period_um=30.0, energy_nj=4.0, fwhm_fs=1000, delay_fs=80.0, sync=True, band=True,
             fixed=True, method="heun", precision="double"),
        # a scan over periods, crystal lengths, grids and detunings in one
        # launch: the device is full and throughput counts
        dict(name="batch_32", kind="batch", count=32, lg_lo=14, lg_hi=16, length_lo_um=100,
             length_hi_um=1000, precision="single"),
        # one fibre in FP64 (gnlsefib's default): the supercontinuum example
        dict(name="fibre_f64_4096", kind="fibre", n=4096, count=1, length_mm=60.0, saves=40,
             raman=True, shock=True, precision="double"),
        # a pump-power scan of fibres in one launch with FP32 fields
        dict(name="fibre_8192x96", kind="fibre", n=8192, count=96, length_mm=20.0, saves=4,
             raman=True, shock=True, precision="single"),
        # the gain map of a chirped 12 mm grating
        dict(name="qpm_120000", kind="qpm", n_out=120000, length_mm=12.0, period_um=30.0,
             chirped=True),
        # the warm start's inference on a ragged number of instances
        dict(name="forward_200", kind="forward", n_in=2050, width=2048, n_out=2048, batch=200),
        # gradients of the surrogate for an outer optimiser
        dict(name="grads_512", kind="grads", n_in=2050, width=2048, n_out=2048, batch=512),
        # training the surrogate on a device-resident set
        dict(name="train_512", kind="train", n_in=2050, width=2048, n_out=2048, batch=512,
             steps=100, rows=2048),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["pass", "pass", "pass", "ring", "ring", "batch", "fibre", "fibre", "qpm",
                       "forward", "grads", "train"])
    if kind == "pass":
        lg = rng.randint(8, 15)
        method = rng.choice(["heun", "heun", "rk23"])
        return dict(kind="pass", n=2 ** lg, window_ps=round(3.0 * 2.0 ** ((lg - 9) / 3.0), 3),
                    length_um=int(_log(rng, 60, 400 if method == "heun" else 100)),
                    period_um=round(rng.uniform(28.0, 32.0), 3), energy_nj=0.1,
                    area_um2=round(rng.uniform(20.0, 60.0), 1), batch=rng.choice([1, 1, 1, 2, 3, 5]),
                    method=method, precision=rng.choice(["single", "double"]),
                    plots=rng.randint(2, 9))
    if kind == "ring":
        lg = rng.randint(11, 16)
        return dict(kind="ring", n=2 ** lg, window_ps=round(12.0 * 2.0 ** ((lg - 15) / 3.0), 3),
                    length_um=int(_log(rng, 200, 1500)), period_um=round(rng.uniform(28.0, 32.0), 3),
                    energy_nj=round(rng.uniform(1.0, 3.0), 3),
                    fwhm_fs=rng.choice([150, 200, 300, 1000]),
                    delay_fs=round(rng.uniform(-60.0, 110.0), 2), sync=rng.random() < 0.7,
                    band=rng.random() < 0.7, fixed=rng.random() < 0.4,
                    method=rng.choice(["heun", "heun", "heun", "rk23"]),
                    precision=rng.choice(["single", "double"]))
    if kind == "batch":
        lo = rng.randint(12, 15)
        return dict(kind="batch", count=int(_log(rng, 6, 40)), lg_lo=lo, lg_hi=min(16, lo + 2),
                    length_lo_um=100, length_hi_um=int(_log(rng, 150, 700)),
                    precision=rng.choice(["single", "single", "double"]))
    if kind == "fibre":
        precision = rng.choice(["single", "double"])
        lg = rng.randint(8, 13 if precision == "single" else 12)
        return dict(kind="fibre", n=2 ** lg, count=int(_log(rng, 1, 96)),
                    length_mm=round(_log(rng, 4.0, 20.0), 2), saves=rng.randint(3, 8),
                    raman=rng.random() < 0.75, shock=rng.random() < 0.75, precision=precision)
    if kind == "qpm":
        return dict(kind="qpm", n_out=int(_log(rng, 2000, 120000)),
                    length_mm=round(_log(rng, 1.0, 12.0), 2),
                    period_um=round(rng.uniform(7.0, 32.0), 2), chirped=rng.random() < 0.5)
    width = 64 * rng.randint(4, 32)
    sizes = dict(n_in=rng.randint(100, 2100), width=width, n_out=64 * rng.randint(2, 32))
    if kind == "forward":
        return dict(kind="forward", batch=rng.randint(1, 512), **sizes)
    if kind == "grads":
        return dict(kind="grads", batch=64 * rng.randint(1, 8), **sizes)
    return dict(kind="train", batch=64 * rng.randint(2, 8), steps=rng.randint(20, 100), rows=2048,
                **sizes)


# ---------------------------------------------------------------- inputs
def _pass_inputs(c, seed):
    """The arrays of one OPOmexBatch call: sech^2 pump plus one-photon noise."""
    sw = ph.SimWindow(1040e-9, c["n"], c["window_ps"] * 1e-12)
    area = c["area_um2"] * 1e-12
    si = ph.NonlinearCrystal(c["period_um"] * 1e-6, c["length_um"] * 1e-6,
                             chi2=np.pi * 14e-12).solver_inputs(sw)
    pump = ph.sech_pump(sw, 200e-15, c["energy_nj"] * 1e-9, area)
    E = np.stack([np.fft.fftshift(pump + ph.quantum_noise(sw, area, seed * 16 + b))
                  for b in range(c["batch"])], axis=1)
    cdt, rdt = ((np.complex128, np.float64) if c["precision"] == "double"
                else (np.complex64, np.float32))
    tol = (1e-4, 5e-6) if c["method"] == "rk23" else (5e-2, 2.5e-3)
    sel = float(math.ceil(si["nSteps"] / (c["plots"] - 1)))
    ap_shape = (c["n"], c["plots"] - 1) + ((c["batch"],) if c["batch"] > 1 else ())
    return dict(Et=np.ascontiguousarray(E.astype(cdt)) if c["batch"] > 1 else E[:, 0].astype(cdt),
                alpha=si["alpha_w"].astype(rdt), G=si["G33"].astype(rdt), w0=si["w0"],
                bdiffw0=si["bdiffw0"], h=si["h"], nsteps=si["nSteps"], dt=si["dt"],
                beta=si["beta_op"].astype(rdt), max_err=tol[0], min_err=tol[1], sel=sel,
                apft=np.zeros(ap_shape, cdt), stepmods=np.zeros(si["nSteps"], rdt))


def _ring_config(c, seed):
    return ph.OPOConfig(n=c["n"], window=c["window_ps"] * 1e-12, period=c["period_um"] * 1e-6,
                        length=c["length_um"] * 1e-6, pump_energy=c["energy_nj"] * 1e-9,
                        pump_fwhm=c["fwhm_fs"] * 1e-15, delay=c["delay_fs"] * 1e-15,
                        delay_mode="sync" if c["sync"] else "absolute",
                        oc_band=(1.2e-6, 1.8e-6) if c["band"] else None, area=_AREA,
                        error_bounds=(0.0, 1e30) if c["fixed"] else (2.5e-3, 5e-2),
                        noise_seed=seed)


def _instance(cfg, method="heun"):
    b = cfg.build()
    ops = b["ops"]
    return dict(solver=b["solver"], field0=ops["field0"], pump=ops["pump"], cav=ops["cav"],
                ocm=ops["ocm"], delay=b["delay"], method=method)


def _batch_configs(c, seed):
    """Uneven cavities at one time step: grids 2^lo .. 2^hi in turn, periods
    28-32 um, lengths spread over their range, +-50 fs from synchronism."""
    rng = np.random.default_rng(seed)
    out = []
    for i in range(c["count"]):
        lg = c["lg_lo"] + i % (c["lg_hi"] - c["lg_lo"] + 1)
        length = c["length_lo_um"] + (c["length_hi_um"] - c["length_lo_um"]) * \
            ((i * 0.6180339887) % 1.0)
        out.append(ph.OPOConfig(n=2 ** lg, window=12e-12 * 2.0 ** (lg - 15), progress_plots=2,
                                period=float(rng.uniform(28e-6, 32e-6)), length=length * 1e-6,
                                delay=float(rng.uniform(-50e-15, 50e-15)), delay_mode="sync",
                                noise_seed=int(rng.integers(1 << 30))))
    return out


_BETAS = [-11.830e-3, 8.1038e-5, -9.5205e-8, 2.0737e-10, -5.3943e-13, 1.3486e-15, -2.5495e-18,
          3.0524e-21, -1.7140e-24]   # ps^k / m, the photonic-crystal fibre of the example


def _fibre_inputs(c, seed):
    """The supercontinuum example's pulse and fibre (835 nm, 28.4 fs sech,
    12.5 ps window), peak powers 5-10 kW over the fibres of a batch."""
    rng = np.random.default_rng(seed)
    T = np.linspace(-6.25, 6.25, c["n"])
    fields = [np.sqrt(p) / np.cosh(T / 0.0284) *
              np.exp(1j * rng.uniform(0, 2 * np.pi)) * (1 + 1e-3 * rng.standard_normal())
              for p in (np.linspace(5000.0, 10000.0, c["count"]) if c["count"] > 1 else [10000.0])]
    w0 = 2 * np.pi * 299792.458 / 835.0 if c["shock"] else 0.0
    RT = fibre.raman_response(T, 0.0122, 0.032) if c["raman"] else 0.0
    return dict(T=T, fields=fields, w0=w0, gamma=0.11, RT=RT, fr=0.18 if c["raman"] else 0.0)


def _qpm_inputs(c, seed):
    """Mismatches of a signal-pump map around the grating's vector and the
    sampled poling (1 um samples), uniform or linearly chirped domains."""
    rng = np.random.default_rng(seed)
    L = c["length_mm"] * 1e-3
    nz = int(round(1e6 * L))
    z = np.linspace(0.0, L, nz)
    per = c["period_um"] * 1e-6
    edges, x = [], 0.0
    while x < L:
        x += 0.5 * per * (1.0 + (0.15 * (x / L - 0.5) if c["chirped"] else 0.0)) * \
            (1.0 + (0.02 * rng.standard_normal() if c["chirped"] else 0.0))
        edges.append(x)
    P = 1.0 - 2.0 * (np.searchsorted(edges, z, side="right") % 2)
    dk = 2 * np.pi / per * rng.uniform(0.2, 1.8, c["n_out"])
    return dict(dk=dk, z=z, w=P * z[1])


def _mlp_params(c, seed):
    """He-normal weights, small biases, in the public layout."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    parts = []
    for l, (o, i) in enumerate(layer_shapes(c["n_in"], c["width"], c["n_out"])):
        sc = math.sqrt(2.0 / i) * (0.5 if l == 3 else 1.0)
        parts += [torch.randn(o * i, generator=g, device="cuda") * sc,
                  torch.randn(o, generator=g, device="cuda") * 0.01]
    return torch.cat(parts).cpu().numpy()


def _mlp_rows(c, rows, seed):
    """Rows as the features are: inputs of order one, targets correlated with them."""
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    x = torch.randn(rows, c["n_in"], generator=g, device="cuda")
    mix = torch.randn(c["n_in"], c["n_out"], generator=g, device="cuda") / math.sqrt(c["n_in"])
    t = torch.tanh(x @ mix) + 0.1 * torch.randn(rows, c["n_out"], generator=g, device="cuda")
    return x.cpu().numpy(), t.cpu().numpy()


# ---------------------------------------------------------------- prepare / run
_shared = {}


def _context():
    if "ctx" not in _shared:
        _shared["ctx"] = Context(0)
    return _shared["ctx"]


def prepare(case, seed):
    c, k = case, case["kind"]
    if k == "pass":
        return dict(case=c, a=_pass_inputs(c, seed), ctx=_context())
    if k == "ring":
        inst = _instance(_ring_config(c, seed), c["method"])
        return dict(case=c, field=inst["field0"],
                    run=OPOBatch([inst], precision=c["precision"], ctx=_context()))
    if k == "batch":
        insts = [_instance(cfg) for cfg in _batch_configs(c, seed)]
        return dict(case=c, fields=[i["field0"] for i in insts],
                    run=OPOBatch(insts, precision=c["precision"], ctx=_context()))
    if k == "fibre":
        f = _fibre_inputs(c, seed)
        if c["count"] > 1:
            f["op"] = fibre.operators(f["T"], f["w0"], f["gamma"], _BETAS, 0.0, f["fr"], f["RT"])
        return dict(case=c, f=f)
    if k == "qpm":
        return dict(case=c, q=_qpm_inputs(c, seed))
    batch = max(64, -(-c["batch"] // 64) * 64)
    net = SurrogateMLP(c["n_in"], c["width"], c["n_out"], max_batch=batch,
                       params=_mlp_params(c, seed))
    s = dict(case=c, net=net)
    if k == "train":
        net.upload_dataset(*_mlp_rows(c, c["rows"], seed))
    else:
        s["x"], s["t"] = _mlp_rows(c, c["batch"], seed)
    return s


def _cx(c):
    return np.complex128 if c["precision"] == "double" else np.complex64


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "pass":
        a = s["a"]
        return list(OPOmexBatch(a["Et"], a["alpha"], a["G"], a["w0"], a["bdiffw0"], a["h"],
                                a["nsteps"], a["dt"], a["beta"], a["max_err"], a["min_err"],
                                a["sel"], a["apft"], a["stepmods"], ctx=s["ctx"],
                                precision=c["precision"], method=c["method"]))
    if k == "ring":
        b = s["run"]
        b.write_field(0, s["field"])
        b.launch(1)
        b.sync()
        r = b.read(0)
        # (read() widens to FP64; the fields are held in the run's precision)
        return [r["field"].astype(_cx(c)), r["oc_spec"].astype(_cx(c)),
                r["apft"].astype(_cx(c)), r["stepmods"].astype(np.int32)]
    if k == "batch":
        b = s["run"]
        for i, f in enumerate(s["fields"]):
            b.write_field(i, f)
        b.launch(1)
        b.sync()
        out = [b.read(i) for i in range(b.n_inst)]
        return [np.concatenate([r["field"] for r in out]).astype(_cx(c)),
                np.concatenate([r["oc_spec"] for r in out]).astype(_cx(c))]
    if k == "fibre":
        f = s["f"]
        if c["count"] == 1:
            Z, AT, AW, _, _ = fibre.gnlsefib(f["T"], f["fields"][0], f["w0"], f["gamma"], _BETAS,
                                             0.0, f["fr"], f["RT"], c["length_mm"] * 1e-3,
                                             c["saves"], precision=c["precision"])
            return [AT.astype(_cx(c)), AW.astype(_cx(c))]
        _, AWz, _, _ = fibre.gnlse_batch(f["T"], f["fields"], [f["op"]] * c["count"],
                                         c["length_mm"] * 1e-3, c["saves"], c["precision"])
        return [AWz.astype(_cx(c))]
    if k == "qpm":
        q = s["q"]
        return [qpm.zsum(q["dk"], q["z"], q["w"])]
    net = s["net"]
    if k == "forward":
        return [net.forward(s["x"])]
    if k == "grads":
        loss, g = net.gradients(s["x"], s["t"])
        return [np.float32(loss), g]
    losses, _ = net.train(c["steps"], batch=c["batch"], lr=1e-4, seed=1)
    return [losses, net.get_params()]


# ---------------------------------------------------------------- work
def _nee_flops(n, steps):
    # a split step: two transforms and about 200 operations a point
    return steps * (10.0 * n * math.log2(n) + 200.0 * n)


def work(case):
    """Each input read once and each output written once; the arithmetic of
    the accepted steps at their usual length (4 minimal steps)."""
    c, k = case, case["kind"]
    if k == "pass":
        sz = 16.0 if c["precision"] == "double" else 8.0
        ns, n, b = c["length_um"] * 10, c["n"], c["batch"]
        return dict(bytes=b * n * sz * (2 + c["plots"] - 1) + n * sz + ns * 1.5 * sz,
                    flops=b * _nee_flops(n, ns / 4 if c["method"] == "heun" else ns))
    if k == "ring":
        sz = 16.0 if c["precision"] == "double" else 8.0
        n, ns = c["n"], c["length_um"] * 10
        return dict(bytes=n * sz * (2 + 3 + 1 + 4) + n * 16.0 + ns * 12.0,
                    flops=_nee_flops(n, ns / 4))
    if k == "batch":
        sz = 16.0 if c["precision"] == "double" else 8.0
        by = fl = 0.0
        for cfg in _batch_configs(c, 0):
            by += cfg.n * sz * 6 + cfg.n * 16.0 + cfg.length * 1e7 * 12.0
            fl += _nee_flops(cfg.n, cfg.length * 1e7 / 4)
        return dict(bytes=by, flops=fl)
    if k == "fibre":
        n, B = c["n"], c["count"]
        evals = 6.0 * (30 + 8.0 * c["length_mm"])
        per = (20.0 if c["raman"] else 10.0) * n * math.log2(n) + 120.0 * n
        return dict(bytes=B * n * 16.0 * (c["saves"] + 3), flops=B * evals * per)
    if k == "qpm":
        runs = 2 * c["length_mm"] * 1e3 / c["period_um"]
        return dict(bytes=c["n_out"] * 24.0, flops=c["n_out"] * runs * 50.0)
    p = sum(o * i + o for o, i in layer_shapes(c["n_in"], c["width"], c["n_out"]))
    w = sum(o * i for o, i in layer_shapes(c["n_in"], c["width"], c["n_out"]))
    B = c["batch"]
    io = 4.0 * B * (c["n_in"] + c["n_out"])
    if k == "forward":
        return dict(bytes=2.0 * p + io, flops=2.0 * B * w)
    dgrad = w - c["width"] * c["n_in"]
    if k == "grads":
        return dict(bytes=8.0 * p + io, flops=2.0 * B * (2 * w + dgrad))
    return dict(bytes=c["steps"] * (28.0 * p + io) + 4.0 * p,
                flops=c["steps"] * 2.0 * B * (2 * w + dgrad))


# ---------------------------------------------------------------- exact
class _Nee:
    """The nonlinear envelope equation's split step in torch at 64 bits."""

    def __init__(self, n, dt, w0, bdiffw0, h, beta, alpha, G):
        f64 = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()  # noqa: E731
        self.n, self.dt, self.w0, self.bdw, self.h = n, dt, w0, bdiffw0, h
        t = np.fft.fftshift((np.arange(n) - n // 2) * dt)
        self.wt = f64(np.remainder(w0 * t, 2 * np.pi))
        tr = (n - 1) * dt
        at2 = np.abs(2 * t)
        sh = 1.0 / np.cosh(np.clip(24.0 * (1.0 - at2 / tr), -700, 700))
        self.absorb = f64(np.where(tr - at2 < 0.25 * tr, 1.0 - sh ** 2, 1.0))
        self.beta, self.alpha = f64(beta), f64(alpha)
        self.G = np.asarray(G, np.float64)

    def slope(self, A, s, Gk, z):
        e = torch.polar(torch.ones_like(self.wt), self.wt - self.bdw * z * self.h)
        nl = A * A * e + 2 * (A.abs() ** 2) * e.conj()
        d = torch.roll(nl, -1) - torch.roll(nl, 1)
        return -1j * (s * self.h * Gk) * (nl - 1j * (0.5 / self.dt / self.w0) * d)

    def disperse(self, E, s):
        S = torch.fft.fft(E * self.absorb)
        S = S * torch.polar(self.alpha ** s, -self.beta * s)
        return torch.fft.ifft(S), S

    def heun(self, A, max_err, min_err, sel, cols):
        ns, k, s = self.G.size, 1.0, 4.0
        ap = [torch.zeros_like(A)] * cols
        chunk, nch = 1, ns / sel
        while chunk <= nch:
            S = None
            while k < chunk * sel and k <= ns:
                Gk = self.G[int(k) - 1]
                k1 = self.slope(A, s, Gk, k - 1.0)
                A1 = A + k1
                E = A + 0.5 * k1 + 0.5 * self.slope(A1, s, Gk, k - 1.0 + s)
                err = 0.0
                if max_err < 1e29:
                    err = 100.0 * float(((E - A1).abs() / (E.abs() + 1.0)).max())
                if err > max_err and s > 1:
                    s -= 1.0
                    continue
                A, S = self.disperse(E, s)
                if err < min_err:
                    s += 1.0
                if k < ns and k + s > ns:
                    s = ns - k
                k += s
            if chunk <= cols:
                ap[chunk - 1] = S if S is not None else torch.fft.fft(A)
            chunk += 1
        return A, ap

    def rk23(self, A, max_err, min_err, sel, cols):
        ns, k, prev, s = self.G.size, 0.0, 4.0, 4.0
        sel = int(sel)
        ap = [torch.zeros_like(A)] * cols
        K1 = self.slope(A, s, self.G[0], 0.0)
        for chunk in range(ns // sel):
            s, cend = prev, float((chunk + 1) * sel)
            S = None
            while k < cend:
                Gk = self.G[int(k)]
                K2 = self.slope(A + 0.5 * K1, s, Gk, k + 0.5 * s)
                K3 = self.slope(A + 0.75 * K2, s, Gk, k + 0.75 * s)
                E = A + (4 / 9 * K3 + 1 / 3 * K2) + 2 / 9 * K1
                K4 = self.slope(E, s, Gk, k + s)
                A1 = A + (1 / 8 * K4 + 1 / 3 * K3) + 1 / 4 * K2 + 7 / 24 * K1
                err = 400.0 * float((0.5 * (A1 - E).abs() / (E.abs() + 1.0)).max())
                if err >= max_err and s > 1 and k - s > 0:
                    k -= s
                    s -= 1.0
                    prev = s
                    K1 = self.slope(A, s, self.G[int(k)], k + s)
                    k += s
                    continue
                A, S = self.disperse(E, s)
                K1 = K4
                if k + s >= cend and k < cend - 1:
                    prev, s = s, cend - k - 1
                else:
                    if err < min_err and k + 2 * s < cend - 1:
                        s *= 2
                    prev = s
                k += s
            if chunk < cols:
                ap[chunk] = S
        return A, ap


def _solve(eq, method, A, max_err, min_err, sel, cols):
    return (eq.rk23 if method == "rk23" else eq.heun)(A, max_err, min_err, sel, cols)


def _host(x):
    return x.cpu().numpy()


def _exact_pass(c, seed):
    a = _pass_inputs(c, seed)
    eq = _Nee(c["n"], a["dt"], a["w0"], a["bdiffw0"], a["h"], a["beta"], a["alpha"], a["G"])
    E, ap = [], []
    for b in range(c["batch"]):
        e0 = a["Et"] if c["batch"] == 1 else a["Et"][:, b]
        A = torch.from_numpy(np.ascontiguousarray(e0.astype(np.complex128))).cuda()
        A, cols = _solve(eq, c["method"], A, a["max_err"], a["min_err"], a["sel"],
                            c["plots"] - 1)
        E.append(_host(A))
        ap.append([_host(x) for x in cols])
    ap_out = np.stack([np.stack(cols, axis=1) for cols in ap], axis=2)
    ap_out = ap_out[:, :, 0] if c["batch"] == 1 else ap_out
    # (the step record is a list of whole numbers: no 64-bit value of its own)
    return [E[0] if c["batch"] == 1 else np.stack(E, axis=1), ap_out, None]


def _exact_ring(c, seed):
    i = _instance(_ring_config(c, seed), c["method"])
    s = i["solver"]
    n = c["n"]
    eq = _Nee(n, s["dt"], s["w0"], s["bdiffw0"], s["h"], s["beta_op"], s["alpha_w"], s["G33"])
    A = torch.from_numpy(np.ascontiguousarray(i["field0"], dtype=np.complex128)).cuda()
    A, ap = _solve(eq, c["method"], A, s["maxErr"], s["minErr"], s["sel"], s["n_cols"])
    S = np.fft.fft(_host(A))
    dw = 2 * np.pi * np.fft.fftfreq(n, s["dt"])
    nxt = np.fft.ifft(S * np.asarray(i["cav"]) * np.exp(-1j * i["delay"] * dw) +
                      np.asarray(i["pump"]))
    return [nxt, S * np.asarray(i["ocm"]), np.stack([_host(x) for x in ap], axis=1), None]


_DP_A = [0.2, 0.3, 0.8, 8 / 9, 1.0, 1.0]
_DP_B = [[1 / 5], [3 / 40, 9 / 40], [44 / 45, -56 / 15, 32 / 9],
         [19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729],
         [9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656],
         [35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84]]
_DP_E = [71 / 57600, 0, -71 / 16695, 71 / 1920, -17253 / 339200, 22 / 525, -1 / 40]
_DP_I = [[1, -183 / 64, 37 / 12, -145 / 128], [0, 0, 0, 0],
         [0, 1500 / 371, -1000 / 159, 1000 / 371], [0, -125 / 32, 125 / 12, -375 / 64],
         [0, 9477 / 3392, -729 / 106, 25515 / 6784], [0, -11 / 7, 11 / 3, -55 / 28],
         [0, 3 / 2, -4, 5 / 2]]


def _dormand_prince(rhs, Z, y, rtol=1e-5, atol=1e-12):
    """The 5(4) pair with the norm-controlled steps and outputs of ode45."""
    comb = lambda f, w: sum(a * b for a, b in zip(w, f) if a)  # noqa: E731
    norm = np.linalg.norm
    t, tf, thr = Z[0], Z[-1], atol / rtol
    out = [y]
    f = [rhs(t, y)]
    hmax = 0.1 * abs(tf - t)
    h = min(hmax, abs(Z[1] - Z[0]))
    rh = norm(f[0]) / max(norm(y), thr) / (0.8 * rtol ** 0.2)
    if h * rh > 1:
        h = 1.0 / rh
    done = False
    while not done:
        h = min(hmax, max(16 * np.spacing(t), h))
        if 1.1 * h >= abs(tf - t):
            h, done = tf - t, True
        first = True
        while True:
            f = f[:1]
            for k in range(5):
                f.append(rhs(t + h * _DP_A[k], y + h * comb(f, _DP_B[k])))
            tn = tf if done else t + h
            h = tn - t
            yn = y + h * comb(f, _DP_B[5])
            f.append(rhs(tn, yn))
            err = h * norm(comb(f, _DP_E)) / max(norm(y), norm(yn), thr)
            if err <= rtol:
                break
            h = h * max(0.1, 0.8 * (rtol / err) ** 0.2) if first else 0.5 * h
            first = done = False
        while len(out) < len(Z) and tn >= Z[len(out)]:
            s = (Z[len(out)] - t) / h
            out.append(yn if Z[len(out)] == tn else
                       y + h * comb(f, [b[0] * s + b[1] * s ** 2 + b[2] * s ** 3 + b[3] * s ** 4
                                        for b in _DP_I]))
        if first:
            g = 1.25 * (err / rtol) ** 0.2
            h = h / g if g > 0.2 else 5.0 * h
        t, y, f = tn, yn, [f[6]]
    return np.stack(out)


def _exact_fibre(c, seed):
    if c["count"] * c["n"] * c["length_mm"] > 4096 * 130:
        return None     # too many right-hand sides for a host solve
    f = _fibre_inputs(c, seed)
    T, n = f["T"], c["n"]
    dT = T[1] - T[0]
    V = 2 * np.pi * np.arange(-(n // 2), n - n // 2) / (n * dT)
    B = sum(b / math.factorial(i + 2) * V ** (i + 2) for i, b in enumerate(_BETAS))
    L = np.fft.fftshift(1j * B)
    W, g = (np.fft.fftshift(V + f["w0"]), f["gamma"] / f["w0"]) if c["shock"] else (1.0, f["gamma"])
    RW = n * np.fft.ifft(np.fft.fftshift(f["RT"])) if c["raman"] else None
    fr = f["fr"]

    def rhs(z, AW):
        AT = np.fft.fft(AW * np.exp(L * z))
        IT = np.abs(AT) ** 2
        M = AT * IT if RW is None else \
            AT * ((1 - fr) * IT + dT * fr * np.fft.fft(np.fft.ifft(IT) * RW))
        return 1j * g * W * np.fft.ifft(M) * np.exp(-L * z)

    Z = np.linspace(0.0, c["length_mm"] * 1e-3, c["saves"])
    got = [_dormand_prince(rhs, Z, np.fft.ifft(a)) for a in f["fields"]]
    if c["count"] > 1:
        return [np.stack(got)]
    a = got[0] * np.exp(L[None, :] * Z[:, None])
    return [np.fft.fft(a, axis=1), np.fft.fftshift(a, axes=1) * dT * n]


def _exact_mlp(c, seed):
    """The network, its loss and (for training) Adam in FP64."""
    shapes = layer_shapes(c["n_in"], c["width"], c["n_out"])
    p = torch.from_numpy(_mlp_params(c, seed)).cuda().double().requires_grad_(c["kind"] != "forward")

    def net(x):
        at = 0
        for l, (o, i) in enumerate(shapes):
            w = p[at:at + o * i].view(o, i)
            at += o * i
            x = torch.addmm(p[at:at + o], x, w.t())
            at += o
            if l < 3:
                x = torch.nn.functional.gelu(x)
        return x

    def loss_of(x, t):
        return ((net(x) - t).norm(dim=1) / t.norm(dim=1)).mean()

    rows = c["rows"] if c["kind"] == "train" else c["batch"]
    x, t = (torch.from_numpy(v).cuda().double() for v in _mlp_rows(c, rows, seed))
    if c["kind"] == "forward":
        return [net(x).cpu().numpy()]
    if c["kind"] == "grads":
        loss = loss_of(x, t)
        loss.backward()
        return [float(loss), p.grad.cpu().numpy()]
    rng, idx = np.random.default_rng(1), []
    while sum(len(v) for v in idx) < c["steps"] * c["batch"]:
        idx.append(rng.permutation(rows))
    idx = torch.from_numpy(np.concatenate(idx)).cuda()
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
    for s in range(c["steps"]):
        pick = idx[s * c["batch"]:(s + 1) * c["batch"]]
        loss = loss_of(x[pick], t[pick])
        g, = torch.autograd.grad(loss, p)
        losses.append(float(loss))
        with torch.no_grad():
            m.mul_(0.9).add_(g, alpha=0.1)
            v.mul_(0.999).addcmul_(g, g, value=0.001)
            p -= 1e-4 * (m / (1 - 0.9 ** (s + 1))) / ((v / (1 - 0.999 ** (s + 1))).sqrt() + 1e-8)
    return [np.array(losses), p.detach().cpu().numpy()]


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "pass":
        return _exact_pass(c, seed)
    if k == "ring":
        return _exact_ring(c, seed)
    if k == "batch":
        return None     # tens of cavities of thousands of steps: minutes in plain torch
    if k == "fibre":
        return _exact_fibre(c, seed)
    if k == "qpm":
        # the literal sum over the samples, a slice of the outputs at a time
        q = _qpm_inputs(c, seed)
        z, w = (torch.from_numpy(q[v]).cuda() for v in ("z", "w"))
        out = []
        for dk in torch.from_numpy(q["dk"]).cuda().split(4096):
            ph_ = dk[:, None] * z[None, :]
            out.append(torch.complex(ph_.cos() @ w, ph_.sin() @ w))
        return [torch.cat(out).cpu().numpy()]
    return _exact_mlp(c, seed)
