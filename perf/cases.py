"""Performance cases: what programs do with this package, through its public entry points.

listed() names the cases, draw(rng) gives more of the same ranges, prepare()
makes what a program holds before the call (inputs on the GPU, or host arrays
where the entry point takes those; plans), run() is one pass, work() the bytes
and operations a pass cannot do without, and exact() the same outputs from
plain torch in 64 bits.

Kinds of case:
  sir     one array of rectangular elements (torch_ops.arr_rect)
  batch   many uneven arrays of rectangles in one launch (torch_ops.SirBatch)
  annular an annular array (torch_ops.arr_annu)
  att     an array in an attenuating medium (torch_ops.sir_attenuated)
  tfm     a total-focusing image from device data (torch_ops.DasPlan.forward)
  host    an image from host arrays, the reference's Python call (das.das, das_f.das)
  train   image and gradients of a loss on it (torch_ops.das_diff)
  conv    many signals through an electrical impulse response (torch_ops.conv_sum)

Units are the package's: mm, us, m/s; sampling frequencies in MHz.
"""
import math

import numpy as np
import torch

from dream_amd import das as das_f64
from dream_amd import das_f as das_f32
from dream_amd import torch_ops

CP = 1500.0
F0, BANDWIDTH = 5.0, 0.6                      # transducer pulse: MHz, fraction
SIGMA = math.sqrt(2.0 * math.log(2.0)) / (math.pi * BANDWIDTH * F0)      # us
EXACT_CONTRIBUTIONS = 2.0e9                   # of a batch's problems in exact()


def listed():
    return [
        # The smallest call: one array's response at a line of points on its
        # axis, as a simulation script asks for it inside a loop.
        dict(name="sir_axis_f64", kind="sir", points=64, elements=16, a=0.9, b=10.0, pitch=1.0,
             step=0.05, dt=0.025, nt=400, plane=False, focus="off", apod="off", out="f64"),
        # The field of a focused, apodized array over a plane.
        dict(name="sir_plane_f64", kind="sir", points=16384, elements=32, a=0.4, b=10.0,
             pitch=0.5, step=0.05, dt=0.02, nt=1200, plane=True, focus="x", apod="hann",
             out="f64"),
        # Arrays of every size in one launch: the rows of a system model.
        dict(name="sir_batch_f32", kind="batch", problems=24, points_lo=256, points_hi=8192,
             elements_lo=8, elements_hi=128, nt_lo=500, nt_hi=4000, out="f32"),
        # The annular array of the reference's own test over a plane.
        dict(name="annular_plane_f64", kind="annular", points=4096, rings=5, r0=3.5, width=0.9,
             step=0.05, dt=0.25, nt=300, cp=1000.0, focus="x", out="f64"),
        # The same small array in an attenuating medium.
        dict(name="attenuated_axis_f64", kind="att", points=64, elements=16, a=0.9, b=10.0,
             pitch=1.0, step=0.05, dt=0.025, nt=400, alpha=5.0, out="f64"),
        # One frame of full-matrix capture to an image: the usual inspection.
        dict(name="tfm_image_f32", kind="tfm", elements=64, pitch=0.5, samples=2048, fs=50.0,
             nx=256, nz=256, pixel=0.125, frames=1, precision="f32", interp="nearest",
             two_arrays=False, apod=False, delay=0.0),
        # The reference's Python call on host arrays, a system delay set.
        dict(name="host_tfm_f64", kind="host", elements=48, pitch=0.5, samples=1800, fs=40.0,
             nx=200, nz=180, pixel=0.15, precision="f64", method="tfm", delay=0.35),
        # A training step through the TFM image: gradients in data and weights.
        dict(name="tfm_train_f32", kind="train", method="tfm", elements=48, pitch=0.5,
             samples=1536, fs=40.0, nx=192, ny=1, nz=160, pixel=0.16, frames=1, precision="f32",
             interp="linear", grad_y=True, grad_cp=False),
        # Calibration of a synthetic-aperture image: gradients in data, weights and speed.
        dict(name="saft_train_f32", kind="train", method="saft", elements=128, pitch=0.3,
             samples=4096, fs=50.0, nx=512, ny=1, nz=512, pixel=0.06, frames=1, precision="f32",
             interp="linear", grad_y=True, grad_cp=True),
        # A row-column array's volumes over several frames, its weights being learned.
        dict(name="rca_train_f32", kind="train", method="rca_rowtx", elements=64, pitch=0.2,
             samples=2560, fs=40.0, nx=64, ny=64, nz=128, pixel=0.2, frames=8, precision="f32",
             interp="nearest", grad_y=False, grad_cp=False),
        # Responses of many points through the transducer's pulse.
        dict(name="conv_pulse_f32", kind="conv", columns=4096, length=2000, taps=300,
             precision="f32", per_column=False),
        # The same through a long coded excitation.
        dict(name="conv_code_f64", kind="conv", columns=1024, length=2000, taps=2000,
             precision="f64", per_column=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sir", "sir", "batch", "annular", "att", "tfm", "tfm", "host", "train",
                       "train", "train", "conv", "conv"])
    if kind == "sir":
        plane = rng.random() < 0.7
        a = round(rng.uniform(0.2, 1.0), 3)
        return dict(kind=kind, points=_log_int(rng, 32, 16384), elements=_log_int(rng, 2, 64),
                    a=a, b=round(rng.uniform(2.0, 12.0), 3), pitch=round(a + 0.1, 3), step=0.05,
                    dt=rng.choice([0.02, 0.025]), nt=_log_int(rng, 200, 1600), plane=plane,
                    focus=rng.choice(["off", "x", "ud"]),
                    apod=rng.choice(["off", "hann"]), out=rng.choice(["f64", "f64", "f32"]))
    if kind == "batch":
        return dict(kind=kind, problems=_log_int(rng, 3, 48), points_lo=16,
                    points_hi=_log_int(rng, 64, 2048), elements_lo=4,
                    elements_hi=_log_int(rng, 8, 96), nt_lo=200, nt_hi=_log_int(rng, 400, 4000),
                    out=rng.choice(["f32", "f32", "f64"]))
    if kind == "annular":
        return dict(kind=kind, points=_log_int(rng, 64, 4096), rings=rng.randint(1, 5),
                    r0=round(rng.uniform(0.8, 3.5), 2), width=round(rng.uniform(0.4, 1.1), 2),
                    step=0.05, dt=rng.choice([0.05, 0.25]), nt=_log_int(rng, 200, 1000),
                    cp=rng.choice([1000.0, 1500.0]), focus=rng.choice(["off", "x"]),
                    out=rng.choice(["f64", "f32"]))
    if kind == "att":
        return dict(kind=kind, points=_log_int(rng, 4, 64), elements=_log_int(rng, 1, 16),
                    a=round(rng.uniform(0.3, 0.9), 2), b=round(rng.uniform(2.0, 10.0), 2),
                    pitch=1.0, step=0.05, dt=rng.choice([0.02, 0.025, 0.04]),
                    nt=_log_int(rng, 150, 450), alpha=round(rng.uniform(0.5, 6.0), 2),
                    out=rng.choice(["f64", "f32"]))
    if kind in ("tfm", "host"):
        c = dict(kind=kind, elements=_log_int(rng, 8, 64), pitch=0.5,
                 samples=rng.randint(500, 2048), fs=rng.choice([25.0, 40.0, 50.0]),
                 nx=_log_int(rng, 24, 256), nz=_log_int(rng, 24, 256), pixel=0.125,
                 precision=rng.choice(["f32", "f64"]),
                 delay=rng.choice([0.0, 0.0, 0.25]))
        if kind == "host":
            return dict(c, method=rng.choice(["tfm", "saft"]))
        return dict(c, frames=rng.choice([1, 1, 3]), interp=rng.choice(["nearest", "linear"]),
                    two_arrays=rng.random() < 0.3, apod=rng.random() < 0.5)
    if kind == "train":
        method = rng.choice(["tfm", "saft", "rca_rowtx", "rca_coltx"])
        rca = method.startswith("rca")
        interp = rng.choice(["nearest", "linear"])
        return dict(kind=kind, method=method,
                    elements=_log_int(rng, 12, 128 if method == "saft" else 48), pitch=0.25,
                    samples=rng.randint(700, 2600), fs=rng.choice([25.0, 40.0]),
                    nx=_log_int(rng, 16, 48 if rca else 200),
                    ny=_log_int(rng, 12, 48) if rca else 1,
                    nz=_log_int(rng, 16, 64 if rca else 160), pixel=0.2,
                    frames=rng.choice([1, 2, 5]) if rca else 1,
                    precision=rng.choice(["f32", "f32", "f64"]),
                    interp=interp, grad_y=rng.random() < 0.6,
                    grad_cp=interp == "linear" and rng.random() < 0.5)
    return dict(kind=kind, columns=_log_int(rng, 16, 4096), length=_log_int(rng, 200, 3000),
                taps=_log_int(rng, 16, 1200), precision=rng.choice(["f32", "f64"]),
                per_column=rng.random() < 0.25)


# ------------------------------------------------------------------ geometry

def _linear_array(n, pitch):
    x = (np.arange(n) - (n - 1) / 2.0) * pitch
    return np.c_[x, np.zeros(n), np.zeros(n)]


def _dtype(name):
    return torch.float64 if name == "f64" else torch.float32


def _centres(width, step):
    """Sub-element centres along a side, accumulated as the package's are."""
    s, out = -width / 2.0 + step / 2.0, []
    while s <= width / 2.0:
        out.append(s)
        s += step
    return np.array(out)


def _sir_problem(case, seed, rng):
    """Points, elements and per-point delays of one array of rectangles."""
    n, pitch = case["elements"], case["pitch"]
    G = _linear_array(n, pitch)
    half = G[-1, 0] + case["a"] / 2
    P = case["points"]
    if case.get("plane", False):
        Ro = np.c_[rng.uniform(-half - 2, half + 2, P), np.zeros(P), rng.uniform(8.0, 60.0, P)]
    else:
        Ro = np.c_[np.zeros(P), np.zeros(P), np.sort(rng.uniform(20.0, 60.0, P))]
    near = np.maximum(np.abs(Ro[:, :1] - G[None, :, 0]) - case["a"] / 2, 0.0)
    delay = np.sqrt(near ** 2 + Ro[:, 2:] ** 2).min(axis=1) * 1000.0 / CP - 0.5
    focal = 0.0
    if case.get("focus") == "ud":
        r = np.hypot(G[:, 0] - rng.uniform(-half, half), 30.0)
        focal = (r.max() - r) * 1000.0 / CP
        delay = delay - focal.max()
    elif case.get("focus") == "x":
        focal = 30.0
        delay = delay - float(np.max(_focal_delays(case, G, focal)))
    return dict(Ro=torch.tensor(Ro.T.copy(), dtype=torch.float64, device="cuda"), G=G,
                delay=torch.tensor(delay, dtype=torch.float64, device="cuda"), focal=focal,
                a=case["a"], b=case["b"], dx=case["step"], dy=case["step"], dt=case["dt"],
                nt=case["nt"], v=1.0, cp=CP, foc_met=case.get("focus", "off"),
                apod_met=case.get("apod", "off"), err_level="ignore")


def _batch_cases(case, rng):
    """The batch's problems as 'sir' cases, uneven in every size."""
    out = []
    for _ in range(case["problems"]):
        a = float(rng.uniform(0.2, 1.0))
        points = math.exp(rng.uniform(math.log(case["points_lo"]), math.log(case["points_hi"])))
        out.append(dict(points=int(round(points)),
                        elements=int(rng.integers(case["elements_lo"], case["elements_hi"] + 1)),
                        a=a, b=float(rng.uniform(5.0, 15.0)), pitch=a + 0.1, step=0.05, dt=0.02,
                        nt=int(rng.integers(case["nt_lo"], case["nt_hi"] + 1)), plane=True,
                        focus="ud", apod="hann"))
    return out


def _batch_rng(case):
    """Sizes of a batch are the case's; the points and delays in them the seed's."""
    return np.random.default_rng(case["problems"] * 100003 + case["points_hi"])


def _radii(case):
    """Centre disc, then (inner, outer) pairs with a 0.1 mm gap."""
    r = [case["r0"]]
    for _ in range(case["rings"] - 1):
        r += [r[-1] + 0.1, r[-1] + 0.1 + case["width"]]
    return r


def _sector(case):
    """Image pixels under the array, z fastest."""
    nx, ny, nz, d = case["nx"], case.get("ny", 1), case["nz"], case["pixel"]
    x = (np.arange(nx) - nx / 2.0) * d
    y = (np.arange(ny) - ny / 2.0) * d if ny > 1 else np.zeros(1)
    z = 5.0 + d * np.arange(nz)
    X, Y, Z = np.meshgrid(x, y, z, indexing="ij")
    return np.c_[X.ravel(), Y.ravel(), Z.ravel()]


def _arrays(case):
    """Transmit and receive elements (columns and rows of a row-column array)."""
    n = case["elements"]
    Gt = _linear_array(n, case["pitch"])
    method = case.get("method", "tfm")
    if method == "saft":
        return Gt, None
    if method.startswith("rca"):
        return Gt, Gt[:, [1, 0, 2]]
    if case.get("two_arrays", False):
        return Gt, Gt + np.array([0.5 * case["pitch"], 0.0, 0.0])
    return Gt, Gt


def _echoes(case, seed, dtype):
    """A-scans of point scatterers plus noise: (frames, A-scans, samples)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    Gt, Gr = _arrays(case)
    Ro, K, fs = _sector(case), case["samples"], case["fs"]
    S = Ro[rng.integers(0, Ro.shape[0], 24)] + rng.normal(0.0, 0.02, (24, 3)) * [1, 0, 1]
    amp = torch.tensor(rng.uniform(0.5, 1.0, 24), device="cuda")
    method = case.get("method", "tfm")

    def legs(G, x=True, y=True):
        d = G[:, None, :] - S[None, :, :]
        return np.sqrt((d[..., 0] * x) ** 2 + (d[..., 1] * y) ** 2 + d[..., 2] ** 2) * 1000.0 / CP

    if method == "saft":
        tau = 2.0 * legs(Gt)
    elif method == "tfm":
        tau = (legs(Gt)[:, None, :] + legs(Gr)[None, :, :]).reshape(-1, 24)
    else:
        c, r = legs(Gt, y=False), legs(Gr, x=False)
        c, r = (c, r) if method == "rca_coltx" else (r, c)
        tau = (c[:, None, :] + r[None, :, :]).reshape(-1, 24)
    tau = torch.tensor(tau, device="cuda")
    n_a = tau.shape[0]
    half = int(math.ceil(5 * SIGMA * fs)) + 1
    offs = torch.arange(-half, half + 1, device="cuda", dtype=torch.float64)
    Y = torch.zeros((n_a, K), dtype=torch.float64, device="cuda")
    for s in range(24):
        k = torch.floor(tau[:, s:s + 1] * fs) + offs
        t = k / fs - tau[:, s:s + 1]
        val = amp[s] * torch.exp(-0.5 * (t / SIGMA) ** 2) * torch.cos(2 * math.pi * F0 * t)
        ok = (k >= 0) & (k < K)
        Y.scatter_add_(1, torch.where(ok, k, 0.0).long(), torch.where(ok, val, 0.0))
    F = case.get("frames", 1)
    out = torch.empty((F, n_a, K), dtype=dtype, device="cuda")
    for f in range(F):
        out[f] = Y + 0.02 * torch.randn(Y.shape, generator=gen, dtype=torch.float64,
                                        device="cuda")
    return out


# ------------------------------------------------------------------ cases

def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind in ("sir", "att"):
        return dict(case=case, problem=_sir_problem(case, seed, rng))
    if kind == "batch":
        problems = [_sir_problem(c, seed, rng) for c in _batch_cases(case, _batch_rng(case))]
        return dict(case=case, batch=torch_ops.SirBatch(problems, out_dtype=_dtype(case["out"])))
    if kind == "annular":
        n = case["points"]
        Ro = np.c_[rng.uniform(-10, 10, n), np.zeros(n), rng.uniform(10, 50, n)]
        return dict(case=case, Ro=torch.tensor(Ro.T.copy(), device="cuda"), radii=_radii(case),
                    delay=0.0 if case["dt"] > 0.1 else 5.0)
    if kind == "tfm":
        dt = _dtype(case["precision"])
        Gt, Gr = _arrays(case)
        plan = torch_ops.DasPlan("tfm", case["samples"], _sector(case), Gt, Gr,
                                 precision=case["precision"])
        Y = _echoes(case, seed, dt)
        n = case["elements"]
        w = [torch.tensor(rng.uniform(0.6, 1.0, n), dtype=dt, device="cuda") if case["apod"]
             else None for _ in range(2)]
        return dict(case=case, plan=plan, Y=Y if case["frames"] > 1 else Y[0], w=w)
    if kind == "host":
        Gt, Gr = _arrays(case)
        Y = _echoes(case, seed, _dtype(case["precision"]))[0].cpu().numpy().T
        dt = Y.dtype
        return dict(case=case, Y=Y, Gt=np.asfortranarray(Gt, dtype=dt),
                    Gr=None if Gr is None else np.asfortranarray(Gr, dtype=dt),
                    Ro=np.asfortranarray(_sector(case), dtype=dt))
    if kind == "train":
        dt = _dtype(case["precision"])
        Gt, Gr = _arrays(case)
        Ro = _sector(case)
        plan = torch_ops.DasPlan(case["method"], case["samples"], Ro, Gt, Gr,
                                 precision=case["precision"])
        Y = _echoes(case, seed, dt)
        n = case["elements"]
        w = [torch.tensor(rng.uniform(0.6, 1.0, n), dtype=dt, device="cuda", requires_grad=True)
             for _ in range(1 if Gr is None else 2)]
        if case["frames"] == 1:
            Y = Y[0].contiguous()
        Y.requires_grad_(case["grad_y"])
        cp = CP
        if case["grad_cp"]:
            cp = torch.tensor(CP, dtype=dt, requires_grad=True)
        gen = torch.Generator(device="cuda").manual_seed(seed + 1)
        g = torch.randn(Y.shape[:-2] + (Ro.shape[0],), generator=gen, dtype=dt, device="cuda")
        return dict(case=case, plan=plan, Y=Y, w=w, cp=cp, g=g)
    if kind == "conv":
        dt = _dtype(case["precision"])
        gen = torch.Generator(device="cuda").manual_seed(seed)
        N, m, t = case["columns"], case["length"], case["taps"]
        A = torch.randn((N, m), generator=gen, dtype=dt, device="cuda")
        k = torch.arange(t, device="cuda", dtype=torch.float64) - t / 2.0
        pulse = torch.exp(-0.5 * (k / (t / 6.0)) ** 2) * torch.cos(0.63 * k)
        shape = (N, t) if case["per_column"] else (t,)
        B = (pulse * (1.0 + 0.1 * torch.randn(shape, generator=gen, dtype=torch.float64,
                                              device="cuda"))).to(dt).contiguous()
        return dict(case=case, A=A, B=B)
    raise ValueError(f"unknown kind {kind!r}")


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "sir":
        p = state["problem"]
        return torch_ops.arr_rect(p["Ro"], p["a"], p["b"], p["dx"], p["dy"], p["dt"], p["nt"],
                                  p["delay"], p["v"], p["cp"], p["G"], foc_met=p["foc_met"],
                                  focal=p["focal"], apod_met=p["apod_met"], err_level="ignore",
                                  out_dtype=_dtype(case["out"]))
    if kind == "batch":
        return state["batch"].run()
    if kind == "annular":
        return torch_ops.arr_annu(state["Ro"], state["radii"], case["step"], case["step"],
                                  case["dt"], case["nt"], state["delay"], 1.0, case["cp"],
                                  foc_met=case["focus"], focal=25.0, err_level="ignore",
                                  out_dtype=_dtype(case["out"]))
    if kind == "att":
        return torch_ops.sir_attenuated(state["problem"], case["alpha"],
                                        out_dtype=_dtype(case["out"]))
    if kind == "tfm":
        return state["plan"].forward(state["Y"], 1.0 / case["fs"], case["delay"], CP, *state["w"],
                                     interp=case["interp"])
    if kind == "host":
        das = das_f64.das if case["precision"] == "f64" else das_f32.das
        return das(state["Y"], state["Gt"], state["Gr"], state["Ro"], 1.0 / case["fs"],
                   case["delay"], CP, case["method"], "ignore")
    if kind == "train":
        w = state["w"]
        Im = torch_ops.das_diff(state["plan"], state["Y"], w[0], w[1] if len(w) > 1 else None,
                                state["cp"], 1.0 / case["fs"], 0.0, case["interp"])
        leaves = list(w)
        if case["grad_y"]:
            leaves.append(state["Y"])
        if case["grad_cp"]:
            leaves.append(state["cp"])
        return [Im.detach(), *torch.autograd.grad(Im, leaves, state["g"])]
    return torch_ops.conv_sum(state["A"], state["B"])


def _sir_contributions(c):
    return (float(c["points"]) * c["elements"] * len(_centres(c["a"], c["step"]))
            * len(_centres(c["b"], c["step"])))


def work(case):
    kind = case["kind"]
    size = 8 if case.get("out", case.get("precision")) == "f64" else 4
    # Of a sub-element's contribution: squared distance, root, sample, amplitude, sum.
    ops = 10.0
    if kind in ("sir", "att"):
        P = case["points"]
        flops = ops * _sir_contributions(case)
        if kind == "att":
            flops += 5.0 * P * case["nt"] * math.log2(case["nt"])
        return dict(bytes=P * (case["nt"] * size + 32.0), flops=flops)
    if kind == "batch":
        cs = _batch_cases(case, _batch_rng(case))
        return dict(bytes=sum(c["points"] * (c["nt"] * size + 32.0) for c in cs),
                    flops=ops * sum(map(_sir_contributions, cs)))
    if kind == "annular":
        area = sum(math.pi * r * r for r in _radii(case)) / case["step"] ** 2
        return dict(bytes=case["points"] * (case["nt"] * size + 24.0),
                    flops=ops * area * case["points"])
    if kind == "conv":
        N, m, t = case["columns"], case["length"], case["taps"]
        n = 1 << (m + t - 2).bit_length()
        direct = 2.0 * m * t * N
        fft = 5.0 * n * math.log2(n) * N
        return dict(bytes=size * (N * (m + m + t - 1.0) + t * (N if case["per_column"] else 1)),
                    flops=min(direct, fft))
    n = case["elements"]
    n_a = n if case.get("method") == "saft" else n * n
    pixels = float(case["nx"] * case.get("ny", 1) * case["nz"])
    frames = case.get("frames", 1)
    data = size * frames * n_a * float(case["samples"])
    image = size * frames * pixels
    if kind == "train":
        # Forward and adjoint; the data read by both, the data's gradient written.
        return dict(bytes=(2 + case["grad_y"]) * data + 2 * image + 48.0 * pixels,
                    flops=(4.0 + 3.0 * frames) * 2 * pixels * n_a)
    return dict(bytes=data + image + 24.0 * pixels, flops=(2.0 + frames) * pixels * n_a)


# ------------------------------------------------------------------ exact

def _focal_delays(case, G, focal):
    if case.get("focus") == "ud":
        return np.asarray(focal)
    if case.get("focus") == "x":
        x = np.abs(G[:, 0])
        return (math.sqrt(x.max() ** 2 + focal ** 2) - np.sqrt(x ** 2 + focal ** 2)) * 1e3 / CP
    return np.zeros(G.shape[0])


def _element_weights(case, G):
    if case.get("apod") != "hann":
        return np.ones(G.shape[0])
    r = np.abs(G[:, 0])
    return 0.5 * (1.0 - np.cos((r + r.max()) * math.pi / r.max()))


def _add_responses(H, Ro, xs, ys, shift, weight, ds, dt, cp):
    """H[p] += the sums over sub-elements (xs, ys) of one element, shift[p] its delay."""
    P, nt = H.shape
    # Divisors as tensors: torch multiplies by the reciprocal of a number.
    dt, cp = (torch.tensor(v, dtype=torch.float64, device="cuda") for v in (dt, cp))
    chunk = max(1, (1 << 25) // xs.numel())
    for p0 in range(0, P, chunk):
        R = Ro[p0:p0 + chunk]
        rx, ry, rz = R[:, 0:1] - xs, R[:, 1:2] - ys, R[:, 2:3]
        r = torch.sqrt((rx * rx + ry * ry) + rz * rz)
        it = torch.round(((r * 1000.0) / cp - shift[p0:p0 + chunk, None]) / dt)
        ai = (weight * ds) / (2 * math.pi * r) / dt * 1000.0
        ok = (it >= 0) & (it < nt)
        H[p0:p0 + chunk].scatter_add_(1, torch.where(ok, it, 0.0).long(),
                                      torch.where(ok, ai, 0.0))


def _sir_exact(case, problem):
    Ro = problem["Ro"].t().contiguous()
    G = problem["G"]
    foc, w = _focal_delays(case, G, problem["focal"]), _element_weights(case, G)
    X, Yc = np.meshgrid(_centres(case["a"], case["step"]), _centres(case["b"], case["step"]))
    X = torch.tensor(X.ravel(), device="cuda")
    Yc = torch.tensor(Yc.ravel(), device="cuda")
    H = torch.zeros((case["points"], case["nt"]), dtype=torch.float64, device="cuda")
    for e in range(G.shape[0]):
        R = Ro - torch.tensor(G[e], device="cuda")
        _add_responses(H, R, X, Yc, problem["delay"] - foc[e], float(w[e]),
                       case["step"] * case["step"], case["dt"], CP)
    return H


def _disc(radius, step):
    xs, ys, y = [], [], -radius + step / 2.0
    while y <= radius:
        half = math.sqrt(radius * radius - y * y)
        x = -half + step / 2.0
        while x <= half:
            xs.append(x)
            ys.append(y)
            x += step
        y += step
    return tuple(torch.tensor(v, dtype=torch.float64, device="cuda") for v in (xs, ys))


def _annular_exact(case, seed):
    s = prepare(case, seed)
    Ro, nt, dt, cp = s["Ro"].t().contiguous(), case["nt"], case["dt"], case["cp"]
    shift = torch.full((case["points"],), s["delay"], dtype=torch.float64, device="cuda")
    radii = s["radii"]
    discs = []
    for r in radii:
        D = torch.zeros((case["points"], nt), dtype=torch.float64, device="cuda")
        xs, ys = _disc(r, case["step"])
        if xs.numel():
            _add_responses(D, Ro, xs, ys, shift, 1.0, case["step"] ** 2, dt, cp)
        discs.append(D)
    rings = (len(radii) + 1) // 2
    mid = [0.0] + [(radii[2 * n] + radii[2 * n - 1]) / 2.0 for n in range(1, rings)]
    H = torch.zeros_like(discs[0])
    for n in range(rings):
        D = discs[0] if n == 0 else discs[2 * n] - discs[2 * n - 1]
        foc = 0.0
        if case["focus"] == "x":
            foc = (math.sqrt(mid[-1] ** 2 + 625.0) - math.sqrt(mid[n] ** 2 + 625.0)) * 1000 / cp
        k = int(np.rint(foc / dt)) + 1
        if k < nt:
            H[:, k:] += D[:, :nt - k]
    return H


def _attenuated_exact(case, problem):
    Ro, G, nt, dt = problem["Ro"].t().contiguous(), problem["G"], case["nt"], case["dt"]
    X, Yc = np.meshgrid(_centres(case["a"], case["step"]), _centres(case["b"], case["step"]))
    ys = torch.tensor(Yc.ravel(), device="cuda")
    gx = torch.tensor(G[:, 0:1], device="cuda")
    x0 = torch.tensor(X.ravel(), device="cuda")
    dt_s = dt * 1e-6
    # Divisors as tensors: torch multiplies by the reciprocal of a number.
    cp, step = (torch.tensor(v, dtype=torch.float64, device="cuda") for v in (CP, dt))
    k = torch.arange(1, nt // 2 + 1, dtype=torch.float64, device="cuda")
    w = k * (2 * math.pi / nt) * (1 / dt_s)
    b = torch.log(1.0 / ((dt_s * 0.95 / math.pi) * w))
    al = case["alpha"] / 8.686e4
    spec = torch.zeros((case["points"], nt // 2 + 1), dtype=torch.complex128, device="cuda")
    for p in range(case["points"]):
        rx, ry, rz = (Ro[p, 0] - gx) - x0, Ro[p, 1] - ys, Ro[p, 2]
        r = torch.sqrt((rx * rx + ry * ry) + rz * rz).reshape(-1)
        it = torch.round(((r * 1000.0) / cp - problem["delay"][p]) / step)
        ai = (case["step"] ** 2) / (2 * math.pi * r) / dt * 1000.0
        ok = (it >= 0) & (it < nt)
        r, it, ai = r[ok] * 1e-3, it[ok], ai[ok]
        spec[p, 0] = ai.sum()
        for c0 in range(0, r.numel(), 1 << 16):
            rc, ic, ac = (v[c0:c0 + (1 << 16), None] for v in (r, it, ai))
            mag = ac * torch.exp(-rc * al * w / (2 * math.pi))
            # The delay's phase 2 pi it k / nt, reduced before it is rounded.
            arg = -w * rc * al / math.pi ** 2 * b - (ic * k % nt) * (2 * math.pi / nt)
            spec[p, 1:] += torch.complex((mag * torch.cos(arg)).sum(0),
                                         (mag * torch.sin(arg)).sum(0))
    return torch.fft.irfft(spec, n=nt)


def _leg(g, x, y, z):
    return torch.sqrt((g[0] - x) ** 2 + (g[1] - y) ** 2 + (g[2] - z) ** 2)


def _gap(p, lo, hi):
    zero = torch.zeros_like(p)
    return torch.where(p < lo, lo - p, torch.where(p > hi, p - hi, zero))


def _das_pairs(case, Ro, Gt, Gr, fs_khz, inv_cp, delay_ms):
    """Blocks of pairs: A-scans, transmit and receive elements, sample positions, travel times."""
    x, y, z = (torch.tensor(Ro[:, c].copy(), device="cuda") for c in range(3))
    method = case.get("method", "tfm")
    if method == "saft":
        for n in range(Gt.shape[0]):
            t = _leg(Gt[n], x, y, z) * inv_cp
            yield torch.tensor([n], device="cuda"), [n], None, \
                (2.0 * (t + delay_ms) * fs_khz)[None], (2.0 * t)[None]
        return
    Lt, Lr = Gt.shape[0], Gr.shape[0]
    if method == "tfm":
        tr = torch.stack([_leg(Gr[j], x, y, z) * inv_cp for j in range(Lr)])
    else:
        gx = _gap(x, Gt[0, 0], Gt[-1, 0])
        tr = torch.stack([torch.sqrt(gx ** 2 + (Gr[j, 1] - y) ** 2 + z ** 2) * inv_cp
                          for j in range(Lr)])
        gy = _gap(y, Gr[0, 1], Gr[-1, 1])
    rows = torch.arange(Lr, device="cuda")
    for i in range(Lt):
        if method == "tfm":
            t = _leg(Gt[i], x, y, z) * inv_cp
        else:
            t = torch.sqrt((Gt[i, 0] - x) ** 2 + gy ** 2 + z ** 2) * inv_cp
        a = rows * Lt + i if method == "rca_rowtx" else i * Lr + rows
        yield a, [i], rows, ((t + delay_ms) + tr) * fs_khz, t + tr


def _taps(case, u, K):
    """(sample, weight) of each tap, out-of-range ones with weight 0, and the fraction's slope."""
    if case.get("interp", "nearest") == "nearest":
        k = torch.trunc(u)
        return [(k, torch.ones_like(u), 0.0)]
    k = torch.floor(u)
    return [(k, 1.0 - (u - k), -1.0), (k + 1.0, u - k, 1.0)]


def _das_exact(case, state, Y, weights, delay=0.0, g=None):
    """Image and, with g, the gradients [weights..., data, speed] of <image, g>."""
    Gt, Gr = _arrays(case)
    Ro = _sector(case)
    Y = Y.detach().double().reshape(-1, Y.shape[-2], Y.shape[-1])
    F, n_a, K = Y.shape
    dt = 1.0 / case["fs"]
    fs_khz, inv_cp, delay_ms = (1.0 / dt) * 1000.0, 1.0 / CP, delay / 1000.0
    w = [torch.ones(G.shape[0], dtype=torch.float64, device="cuda") if q is None
         else q.detach().double() for q, G in zip(weights, (Gt, Gr)) if G is not None]
    Im = torch.zeros((F, Ro.shape[0]), dtype=torch.float64, device="cuda")
    gw = [torch.zeros_like(q) for q in w]
    gY = torch.zeros_like(Y) if g is not None else None
    gcp = torch.zeros((), dtype=torch.float64, device="cuda")
    for a, i, rows, u, travel in _das_pairs(case, Ro, Gt, Gr, fs_khz, inv_cp, delay_ms):
        wt = w[0][i[0]]
        wr = w[1][rows][:, None] if rows is not None else 1.0
        for k, c, slope in _taps(case, u, K):
            ok = (k >= 0) & (k < K)
            idx = torch.where(ok, k, 0.0).long()
            c = torch.where(ok, c, 0.0)
            for f in range(F):
                val = Y[f][a].gather(1, idx)
                Im[f] += (wt * wr * c * val).sum(0)
                if g is None:
                    continue
                gf = g[f].double()
                v = c * val * gf
                gw[0][i[0]] += (wr * v).sum()
                if rows is not None:
                    gw[1].index_add_(0, rows, (wt * v).sum(1))
                if case["grad_y"]:
                    part = torch.zeros((a.numel(), K), dtype=torch.float64, device="cuda")
                    part.scatter_add_(1, idx, wt * wr * c * gf)
                    gY[f].index_add_(0, a, part)
                if slope:
                    gcp += (wt * wr * torch.where(ok, slope, 0.0) * val * gf
                            * travel).sum() * (-fs_khz / CP)
    Im = Im[0] if case.get("frames", 1) == 1 else Im
    if g is None:
        return Im
    gY = gY[0] if case["frames"] == 1 else gY
    return [Im, *gw] + ([gY] if case["grad_y"] else []) + ([gcp] if case["grad_cp"] else [])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("sir", "att"):
        p = prepare(case, seed)["problem"]
        return [(_sir_exact if kind == "sir" else _attenuated_exact)(case, p), None, None]
    if kind == "batch":
        rng, out, left = np.random.default_rng(seed), [], EXACT_CONTRIBUTIONS
        for c in _batch_cases(case, _batch_rng(case)):
            p = _sir_problem(c, seed, rng)
            left -= _sir_contributions(c)
            out.append(_sir_exact(c, p) if left > 0 else None)
        return out
    if kind == "annular":
        return [_annular_exact(case, seed), None, None]
    if kind == "conv":
        s = prepare(case, seed)
        n = case["length"] + case["taps"] - 1
        f = torch.fft.rfft(s["A"].double(), n=n) * torch.fft.rfft(s["B"].double(), n=n)
        return torch.fft.irfft(f, n=n)
    s = prepare(case, seed)
    if kind == "tfm":
        return _das_exact(case, s, s["Y"], s["w"], case["delay"])
    if kind == "host":
        if case["precision"] == "f32":
            return None          # the float module computes its delays in float
        Y = torch.tensor(np.ascontiguousarray(s["Y"].T), device="cuda")
        return _das_exact(case, s, Y, [None, None], case["delay"])
    g = s["g"].reshape(-1, s["g"].shape[-1])
    return _das_exact(case, s, s["Y"], s["w"] + [None], 0.0, g)
