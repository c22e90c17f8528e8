"""The work that users of the engine have it do, as cases that can be timed.

Each case is a dict of plain values; ``prepare`` makes what a program holds
before the call (inputs on the GPU or the host, the handle, plan or network),
``run`` is one pass through the public entry points of ``ctas_amd`` and
``exact`` the same outputs from plain torch in 64 bits. ``listed`` names the
sizes that this repository's benchmark, tests and tools use, ``draw`` gives
others of the same ranges.
"""
import math

import numpy as np
import torch

import ctas_amd as ca

FILTERS = {"RAMP": 1, "HANN": 5}
STORES = {"fp32": ca.STORE_FP32, "fp16": ca.STORE_FP16, "bf16": ca.STORE_BF16}
INTERPS = {"ctas": ca.INTERP_CTAS, "linear": ca.INTERP_LINEAR}


def listed():
    return [
        # `ctas ct` on a scan: one GPU's share of the 256-slice absorption
        # stack that the benchmark reconstructs, in the parity mode
        {"name": "fbp-fp32-32x2048x1800", "kind": "fbp", "slices": 32, "width": 2048, "angles": 1800, "arc": 180.0,
         "store": "fp32", "interp": "ctas", "filter": "HANN", "contrast": "ABS", "center": 3.37},
        # the largest detector: 4096 px x 3000 angles with half-precision storage
        {"name": "fbp-fp16-8x4096x3000", "kind": "fbp", "slices": 8, "width": 4096, "angles": 3000, "arc": 180.0,
         "store": "fp16", "interp": "ctas", "filter": "HANN", "contrast": "ABS", "center": 3.37},
        # a cropped detector and an odd number of projections, LINEAR sampling
        {"name": "fbp-linear-9x1437x1101", "kind": "fbp", "slices": 9, "width": 1437, "angles": 1101, "arc": 180.0,
         "store": "fp32", "interp": "linear", "filter": "RAMP", "contrast": "ABS", "center": -7.25},
        # a preview of one small slice, where launches and latency count
        {"name": "fbp-fp32-1x512x360", "kind": "fbp", "slices": 1, "width": 512, "angles": 360, "arc": 180.0,
         "store": "fp32", "interp": "ctas", "filter": "RAMP", "contrast": "ABS", "center": 1.5},
        # sinograms of many detectors and angle counts queued as one batch
        {"name": "uneven-16-512..2048", "kind": "uneven", "items": 16, "width_lo": 512, "width_hi": 2048,
         "angles_lo": 360, "angles_hi": 1800, "store": "fp32", "interp": "ctas"},
        # `ctas ax`: a round of trial centres scored on one sinogram
        {"name": "axis-scores-9x2048x1800", "kind": "scores", "trials": 9, "width": 2048, "angles": 1800,
         "step": 0.5, "center": 2.5},
        # the learned front end of the axis search on one sinogram
        {"name": "axis-predict-2048x1800", "kind": "predict", "width": 2048, "angles": 1800, "center": -4.0},
        # one step's loss and gradients when that network is trained
        {"name": "axis-train-64", "kind": "train", "batch": 64},
        # ring filter of the sinograms of a batch before reconstruction
        {"name": "rings-16x1800x2048", "kind": "rings", "slices": 16, "width": 2048, "angles": 1800, "box": 15},
        # `ctas ts`: projections filtered and added into one plane
        {"name": "ts-32x2048x2048", "kind": "ts", "projections": 32, "rows": 2048, "pixels": 2048,
         "contrast": "ABS", "filter": "RAMP", "center": 1.0, "plane": 10, "keep": True},
        # `ctas ax` given the 0 and 180 degree projections of a scan
        {"name": "registration-2048x2048", "kind": "register", "rows": 2048, "pixels": 2048, "shift": 13},
        # a program of the reference's API: one slice from and to host arrays
        {"name": "host-1x1024x900", "kind": "host", "slices": 1, "width": 1024, "angles": 900, "arc": 180.0,
         "store": "fp32", "interp": "ctas", "filter": "HANN", "contrast": "ABS", "center": 3.37},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, spread over the logarithm, odd or even."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fbp", "fbp", "fbp", "fbp", "uneven", "scores", "predict", "train", "rings", "ts", "register",
                       "host"])
    if kind in ("fbp", "host"):
        w = _size(rng, 512, 4096 if kind == "fbp" else 1500)
        n = _size(rng, 360, 3000 if kind == "fbp" else 1200)
        store = rng.choice(["fp32", "fp32", "fp16", "bf16"])
        most = max(1, min(32, int(8 * 4096 * 4096 * 3000 / (w * w * n) / (1 if store != "fp32" else 2))))
        return {"kind": kind, "slices": _size(rng, 1, most if kind == "fbp" else 4), "width": w, "angles": n,
                "arc": rng.choice([180.0, 180.0, 180.0, 360.0, 150.0]), "store": store,
                "interp": rng.choice(["ctas", "ctas", "linear"]), "filter": rng.choice(["HANN", "RAMP"]),
                "contrast": rng.choice(["ABS", "ABS", "PHS"]), "center": round(rng.uniform(-20.0, 20.0), 2)}
    if kind == "uneven":
        return {"kind": kind, "items": rng.randint(3, 16), "width_lo": _size(rng, 512, 700),
                "width_hi": _size(rng, 900, 2048), "angles_lo": _size(rng, 360, 500),
                "angles_hi": _size(rng, 700, 1800), "store": rng.choice(["fp32", "fp32", "fp16"]),
                "interp": rng.choice(["ctas", "linear"])}
    if kind == "scores":
        return {"kind": kind, "trials": rng.randint(1, 12), "width": _size(rng, 512, 2048),
                "angles": _size(rng, 360, 1800), "step": rng.choice([0.25, 0.5, 8.0]),
                "center": round(rng.uniform(-10.0, 10.0), 2)}
    if kind == "predict":
        return {"kind": kind, "width": _size(rng, 512, 4096), "angles": _size(rng, 360, 1800),
                "center": round(rng.uniform(-15.0, 15.0), 2)}
    if kind == "train":
        return {"kind": kind, "batch": _size(rng, 4, 64)}
    if kind == "rings":
        return {"kind": kind, "slices": _size(rng, 1, 16), "width": _size(rng, 512, 2048),
                "angles": _size(rng, 360, 1800), "box": rng.randint(3, 30)}
    if kind == "ts":
        return {"kind": kind, "projections": _size(rng, 1, 32), "rows": _size(rng, 256, 2048),
                "pixels": rng.choice([1024, 2048, _size(rng, 600, 2300)]), "contrast": rng.choice(["ABS", "PHS"]),
                "filter": rng.choice(["RAMP", "HANN"]), "center": round(rng.uniform(-8.0, 8.0), 2),
                "plane": rng.randint(-60, 60), "keep": rng.random() < 0.5}
    return {"kind": "register", "rows": _size(rng, 64, 2048), "pixels": _size(rng, 512, 2560),
            "shift": rng.randint(-40, 40)}


# ---- inputs -----------------------------------------------------------------
def _gen(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _sinograms(S, N, w, arc, c, seed, contrast="ABS"):
    """Ellipse phantoms' projections [S][N][w]: noisy transmissions at 1e5
    photons per ray (ABS) or the line integrals with noise (PHS)."""
    g = _gen(seed)
    out = torch.zeros((S, N, w), device="cuda")
    th = torch.arange(N, device="cuda", dtype=torch.float64) * (math.radians(arc) / N)
    co, si = torch.cos(th)[None, :, None], torch.sin(th)[None, :, None]
    det = (torch.arange(w, device="cuda", dtype=torch.float32) + 0.5 - w // 2 - c)[None, None, :]
    r = torch.rand((S, 10, 6), generator=g, device="cuda", dtype=torch.float64)
    for k in range(10):
        e = [r[:, k, q].reshape(S, 1, 1) for q in range(6)]
        rad, phi = 0.3 * w * torch.sqrt(e[0]), 2 * math.pi * e[1]
        a, b = (w / 200 + w / 7 * e[2] ** 2), (w / 200 + w / 7 * e[3] ** 2)
        tilt, mu = math.pi * e[4], (2.4 * e[5] - 0.6) * 2.0 / w
        s0 = (rad * torch.cos(phi) * co + rad * torch.sin(phi) * si).float()
        r2 = (a * a * (co * torch.cos(tilt) + si * torch.sin(tilt)) ** 2
              + b * b * (si * torch.cos(tilt) - co * torch.sin(tilt)) ** 2)
        scale = (2 * mu * a * b / r2).float()
        t = det - s0
        t = r2.float() - t * t
        out += scale * t.clamp_(min=0.0).sqrt_()
        del t
    noise = torch.randn((S, N, w), generator=g, device="cuda")
    if contrast != "ABS":
        return out.add_(noise, alpha=2e-3)
    out = torch.exp_(out.neg_()).mul_(1e5)
    out += noise * out.sqrt()
    return out.clamp_(min=1.0).mul_(1e-5)


def _uneven_shapes(case):
    """Widths and angle counts of the batch, from the smallest to the largest."""
    n = case["items"]
    f = [i / max(1, n - 1) for i in range(n)]
    ws = [int(case["width_lo"] * (case["width_hi"] / case["width_lo"]) ** x) for x in f]
    ns = [int(case["angles_lo"] * (case["angles_hi"] / case["angles_lo"]) ** ((x * 3.0) % 1.0 if 0 < x < 1 else x))
          for x in f]
    return list(zip(ws, ns))


def _projections(case, seed):
    """Transmission (ABS) or line-integral projections [P][rows][pixels]."""
    g = _gen(seed)
    P, R, n = case["projections"], case["rows"], case["pixels"]
    x = torch.linspace(-1.0, 1.0, n, device="cuda")[None, None, :]
    y = torch.linspace(-1.0, 1.0, R, device="cuda")[None, :, None]
    out = torch.zeros((P, R, n), device="cuda")
    r = torch.rand((6, 5), generator=g, device="cuda")
    drift = torch.linspace(-0.1, 0.1, P, device="cuda")[:, None, None]
    for k in range(6):
        cx, cy, rx, ry, mu = (float(v) for v in r[k])
        d = 1.0 - ((x - (cx - 0.5) - drift * (cy - 0.5)) / (0.1 + 0.4 * rx)) ** 2 - ((y - (cy - 0.5)) / (0.1 + 0.4 * ry)) ** 2
        out += (0.2 + mu) * d.clamp_(min=0.0).sqrt_()
    noise = torch.randn((P, R, n), generator=g, device="cuda")
    if case["contrast"] != "ABS":
        return out.add_(noise, alpha=2e-3)
    out = torch.exp_(out.neg_()).add_(noise, alpha=3e-3)
    return out.clamp_(min=1e-3)


def _ts_angles(case):
    """Angles in radians over the limited arc of a tomosynthesis scan."""
    P = case["projections"]
    return (np.linspace(-25.0, 25.0, P) if P > 1 else np.array([7.0])).astype(np.float32) * np.float32(math.pi / 180)


def _pair(case, seed):
    """The projections at 0 and 180 degrees of one scan, as host arrays."""
    R, n, g = case["rows"], case["pixels"], _gen(seed)
    f = torch.rand((3, 5), generator=g, device="cuda").tolist()
    x = torch.linspace(-1.0, 1.0, n, device="cuda")[None, :]
    y = torch.linspace(-1.0, 1.0, R, device="cuda")[:, None]
    p = torch.zeros((R, n), device="cuda")
    for cx, cy, rx, ry, mu in f:
        d = 1.0 - ((x - 0.6 * (cx - 0.5)) / (0.1 + 0.3 * rx)) ** 2 - ((y - (cy - 0.5)) / (0.2 + 0.5 * ry)) ** 2
        p += (0.2 + 0.5 * mu) * d.clamp_(min=0.0).sqrt_()
    q = torch.roll(torch.flip(p, (1,)), case["shift"], 1)
    out = [torch.exp(-t) + 3e-3 * torch.randn((R, n), generator=g, device="cuda") for t in (p, q)]
    return [t.cpu().numpy() for t in out]


def _handle(case):
    return ca.CTrec(case["width"], case["angles"], ca.parse_contrast(case["contrast"]), case["filter"],
                    anarc=case["arc"], interp=INTERPS[case["interp"]], store=STORES[case["store"]])


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind}
    if kind in ("fbp", "host"):
        S, N, w = case["slices"], case["angles"], case["width"]
        s["sino"] = _sinograms(S, N, w, case["arc"], case["center"], seed, case["contrast"])
        s["rec"] = _handle(case)
        s["centers"] = np.full(S, case["center"], np.float32)
        if kind == "host":
            s["sino"] = s["sino"].cpu().numpy()
        else:
            s["out"] = torch.empty((S, w, w), device="cuda")
    elif kind == "uneven":
        s["items"] = []
        for i, (w, N) in enumerate(_uneven_shapes(case)):
            c = 3.0 - 0.75 * i
            s["items"].append((_sinograms(1, N, w, 180.0, c, seed + 1000 * i)[0],
                               torch.empty((w, w), device="cuda"), c))
        s["flags"] = INTERPS[case["interp"]] | STORES[case["store"]]
    elif kind == "scores":
        w, N = case["width"], case["angles"]
        s["sino"] = _sinograms(1, N, w, 180.0, case["center"], seed)
        s["rec"] = ca.CTrec(w, N, ca.ABS, "RAMP")
        k = np.arange(case["trials"]) - case["trials"] // 2
        s["axes"] = (0.5 * (w - 1) + case["center"] + case["step"] * k).astype(np.float32)
    elif kind == "predict":
        s["sino"] = _sinograms(1, case["angles"], case["width"], 180.0, case["center"], seed)[0]
        s["net"] = ca.AxisCNN(weights=ca.CNN_WEIGHTS)
    elif kind == "train":
        B = case["batch"]
        s["net"] = ca.AxisCNN(weights=ca.CNN_WEIGHTS)
        s["x"] = torch.empty((B, 2, 180, 256), dtype=torch.uint16, device="cuda")
        s["target"] = torch.empty((B, 2), device="cuda")
        ca.cnn_make_batch(seed, 0, s["x"], s["target"])
    elif kind == "rings":
        S, N, w = case["slices"], case["angles"], case["width"]
        g = _gen(seed + 1)
        s["sino"] = _sinograms(S, N, w, 180.0, 0.0, seed)
        s["sino"] *= 1.0 + 0.01 * torch.randn((S, 1, w), generator=g, device="cuda")
    elif kind == "ts":
        s["proj"] = _projections(case, seed)
        s["angles"] = _ts_angles(case)
        s["result"] = torch.zeros((case["rows"], case["pixels"]), device="cuda")
        s["filtered"] = torch.empty_like(s["proj"]) if case["keep"] else None
        s["plan"] = ca.TsPlan(case["rows"], case["pixels"], ca.parse_contrast(case["contrast"]), case["filter"])
    else:
        s["p0"], s["p180"] = _pair(case, seed)
    return s


# ---- one pass ---------------------------------------------------------------
def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "fbp":
        s["rec"].reconstruct_dev(s["sino"], s["out"], s["centers"])
        return s["out"]
    if kind == "host":
        filtered, out = s["rec"].reconstruct(s["sino"], s["centers"])
        return {"filtered": filtered, "out": out}
    if kind == "uneven":
        ca.batch_uneven(s["items"], ca.ABS, FILTERS["HANN"], flags=s["flags"])
        return [o for _, o, _ in s["items"]]
    if kind == "scores":
        s["rec"].prepare_dev(s["sino"])
        return s["rec"].axis_scores(s["axes"])
    if kind == "predict":
        return list(s["net"].predict_dev(s["sino"]))
    if kind == "train":
        loss = s["net"].gradients_dev(s["x"], s["target"])
        return {"loss": loss, "grads": s["net"].grads()}
    if kind == "rings":
        ca.ring_filter_dev(s["sino"], case["box"])
        return s["sino"]
    if kind == "ts":
        s["plan"].add_dev(s["proj"], s["angles"], s["result"], case["center"], case["plane"], s["filtered"])
        return [t for t in (s["result"], s["filtered"]) if t is not None]
    return ca.raxis_pair(s["p0"], s["p180"])


# ---- what a pass cannot do without --------------------------------------------
#: Parameters of the axis network, and multiply-adds of one sample's forward pass.
PARAMS = 245554
MACS = 9 * (2 * 32 * 180 * 256 + 32 * 32 * 90 * 128 + 32 * 64 * 45 * 64 + 64 * 64 * 22 * 32) + 11264 * 16


def _fbp_work(S, N, w):
    Z = ca.zidth(w)
    fft = 2 * 2.5 * Z * math.log2(Z)
    return {"bytes": S * (4.0 * N * w + 4.0 * w * w), "flops": S * (2.0 * N * w * w + N * fft)}


def work(case):
    kind = case["kind"]
    if kind in ("fbp", "host"):
        r = _fbp_work(case["slices"], case["angles"], case["width"])
        if kind == "host":
            r["bytes"] += 4.0 * case["slices"] * case["angles"] * case["width"]
        return r
    if kind == "uneven":
        every = [_fbp_work(1, n, w) for w, n in _uneven_shapes(case)]
        return {k: sum(r[k] for r in every) for k in ("bytes", "flops")}
    if kind == "scores":
        one = _fbp_work(1, case["angles"], case["width"])
        # the trial slices need not reach memory: one sinogram in
        return {"bytes": 4.0 * case["angles"] * case["width"],
                "flops": case["trials"] * (one["flops"] + 60.0 * case["width"] ** 2)}
    if kind == "predict":
        return {"bytes": 4.0 * case["angles"] * case["width"] + 2.0 * PARAMS, "flops": 2.0 * MACS}
    if kind == "train":
        B = case["batch"]
        return {"bytes": B * 2.0 * 2 * 180 * 256 + 6.0 * PARAMS, "flops": 3 * 2.0 * MACS * B}
    if kind == "rings":
        n = case["slices"] * case["angles"] * case["width"]
        return {"bytes": 8.0 * n, "flops": 2.0 * n}
    if kind == "ts":
        n, px = case["pixels"], float(case["rows"] * case["pixels"])
        return {"bytes": px * (case["projections"] * (8 if case["keep"] else 4) + 8),
                "flops": case["projections"] * px * (2 * 2.5 * math.log2(n) + 2)}
    px = float(case["rows"] * case["pixels"])
    trials = 1 + 2 * int(0.25 * case["pixels"] / 16)
    return {"bytes": 8.0 * px, "flops": 3.0 * trials * px}


# ---- the same outputs in 64 bits ------------------------------------------------
def _fill(name, n):
    """The frequency window of an n-point line, without a gain."""
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    m = torch.arange(1, n // 2, 2, device="cuda")
    h = torch.zeros(n, device="cuda", dtype=torch.float64)
    h[0] = 0.25
    h[m] = -1.0 / (m.double() * math.pi) ** 2
    h[n - m] = h[m]
    H = torch.fft.fft(h).real
    f = torch.where(k < n // 2, k, n - k) * (2.0 / n)
    return 0.5 * H * (0.5 * (1 + torch.cos(math.pi * f)) if name == "HANN" else torch.ones_like(f))


def _filter64(sino, name, contrast):
    """Filtered rows of [N][w]: the row and the next one's first sample,
    zero-padded to the power of two above 2 w - 2."""
    p = sino.double()
    if contrast == "ABS":
        p = -torch.log(p)
    N, w = p.shape
    Z = 1 << (2 * w - 2).bit_length()
    x = torch.zeros((N, Z), device="cuda", dtype=torch.float64)
    x[:, :w] = p
    x[:-1, w] = p[1:, 0]
    W = _fill(name, Z) * (Z / w)
    return torch.fft.ifft(torch.fft.fft(x) * W).real[:, :w].contiguous()


def _bp64(F, arc, c, linear):
    """Slices [S][w][w] of filtered sinograms [S][N][w] about one centre."""
    S, N, w = F.shape
    hp, c = w // 2, float(np.float32(c))
    j = torch.arange(w, device="cuda", dtype=torch.float64)[:, None]
    i = torch.arange(w, device="cuda", dtype=torch.float64)[None, :]
    out = torch.zeros((S, w * w), device="cuda", dtype=torch.float64)
    flat = F.reshape(S, N * w)
    for a in range(N):
        th = a * math.radians(arc) / N
        si, co = (0.0 if abs(v) < 1e-12 else v for v in (math.sin(th), math.cos(th)))
        t = (c + hp * (1.0 - si - co) + (0.5 if linear else 0.0)) + si * (j - c) + co * i
        if linear:
            k = torch.floor(t)
            f = (t - k).reshape(-1)
            k = k.long().reshape(-1)
            row = torch.zeros((S, w + 2), device="cuda", dtype=torch.float64)
            row[:, 1:-1] = F[:, a]
            q0 = row.index_select(1, k.clamp(0, w + 1))
            q1 = row.index_select(1, (k + 1).clamp(0, w + 1))
            out += q0 + f * (q1 - q0)
        else:
            k = t.long().reshape(-1) + a * w
            inside = (k >= 0) & (k < N * w)
            out += flat.index_select(1, k.clamp(0, N * w - 1)) * inside
    out = out.reshape(S, w, w) / N
    dy2, dx2 = (j - hp - c) ** 2, (i - hp) ** 2
    up, dn = hp + c, hp - c
    masked = ((i <= abs(c)) | (i >= w - abs(c) - 1) | ((j <= up) & (dy2 + dx2 >= up * up))
              | ((j >= up) & (dy2 + dx2 >= dn * dn)))
    return torch.where(masked, 0.0, out)


def _score64(sl, sigma, c):
    """The average-gradient score of one trial slice."""
    w = sl.shape[0]
    if sigma > 1.0:
        n = torch.arange(64, device="cuda", dtype=torch.float64)
        g = torch.exp(-n * n / (2 * sigma * sigma))
        for dim in (1, 0):
            sl = sum(g[k] * torch.roll(sl, k, dim) for k in range(64) if g[k] > 1e-9)
    r = math.ceil(abs(c))
    h = w - 2 * r
    p = torch.zeros((h + 2, w + 2), device="cuda", dtype=torch.float64)
    p[1:-1, 1:-1] = sl[r:w - r]
    dy = p[2:] - p[:-2]
    dH = dy[:, :-2] + 2 * dy[:, 1:-1] + dy[:, 2:]
    dx = p[:, 2:] - p[:, :-2]
    dV = dx[:-2] + 2 * dx[1:-1] + dx[2:]
    m = torch.sqrt(dH * dH + dV * dV)
    m = m[max(0, 1 - r):h - 1 - r, 1:w - 1]
    return float(m.sum() / (m.numel() if sigma > 1.0 else (m > 0).sum()))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("predict", "train"):
        return None  # bfloat16 activations: the 64-bit values are another network's
    if kind == "register":
        return None  # a search over whole shifts: its answer is one of the trials
    if kind in ("fbp", "host"):
        S, N, w = case["slices"], case["angles"], case["width"]
        sino = _sinograms(S, N, w, case["arc"], case["center"], seed, case["contrast"])
        F = torch.stack([_filter64(sino[k], case["filter"], case["contrast"]) for k in range(S)])
        out = _bp64(F, case["arc"], case["center"], case["interp"] == "linear")
        return out if kind == "fbp" else {"filtered": F, "out": out}
    if kind == "uneven":
        out = []
        for i, (w, N) in enumerate(_uneven_shapes(case)):
            c = 3.0 - 0.75 * i
            F = _filter64(_sinograms(1, N, w, 180.0, c, seed + 1000 * i)[0], "HANN", "ABS")
            out.append(_bp64(F[None], 180.0, c, case["interp"] == "linear")[0])
        return out
    if kind == "scores":
        w, N = case["width"], case["angles"]
        F = _filter64(_sinograms(1, N, w, 180.0, case["center"], seed)[0], "RAMP", "ABS")[None]
        sigma = math.radians(180.0 / (N - 1)) * w / math.pi
        k = np.arange(case["trials"]) - case["trials"] // 2
        axes = (0.5 * (w - 1) + case["center"] + case["step"] * k).astype(np.float32).astype(np.float64)
        cs = [float(np.float32(a - 0.5 * (w - 1))) for a in axes]
        return torch.tensor([_score64(_bp64(F, 180.0, c, False)[0], sigma, c) for c in cs], dtype=torch.float64)
    if kind == "rings":
        S, N, w, box = case["slices"], case["angles"], case["width"], case["box"]
        p = prepare(case, seed)["sino"].double()
        mean = p.mean(1)
        pad = torch.zeros((S, w + 2 * box), device="cuda", dtype=torch.float64)
        pad[:, box:box + w] = mean
        t = pad.unfold(1, 2 * box + 1, 1).sum(2)
        x = torch.arange(w, device="cuda")
        n = torch.full((w,), 2 * box + 1, device="cuda")
        n = torch.where(x < box, box + x + 1, torch.where(x >= w - box, box + w - x, n))
        return p + (t / n - mean)[:, None, :]
    # tomosynthesis; the choice of a column is made in 32 bits, as it is defined
    P, R, n = case["projections"], case["rows"], case["pixels"]
    proj = _projections(case, seed)
    W = _fill(case["filter"], n)
    k = torch.arange(n // 2 + 1, device="cuda")
    Wr, Wi = W[k], W[(n - k) % n]
    f32 = np.float32
    rc = f32(n * 0.5 + float(f32(case["center"])))
    x = np.arange(n, dtype=np.float32)
    result = torch.zeros((R, n), device="cuda", dtype=torch.float64)
    kept = torch.empty((P, R, n), device="cuda", dtype=torch.float64)
    for p, a in enumerate(_ts_angles(case)):
        d = proj[p].double()
        X = torch.fft.rfft(-torch.log(d) if case["contrast"] == "ABS" else d)
        kept[p] = torch.fft.irfft(torch.complex(X.real * Wr, X.imag * Wi), n)
        pc = f32(f32(case["plane"]) - f32(case["center"])) * f32(np.sin(a))
        di = (x - rc) * f32(np.cos(a)) - pc + rc
        di = np.where(di < 0, f32(0), np.where(di >= f32(n), f32(n - 1), di))
        result += kept[p][:, torch.from_numpy(di.astype(np.int64)).cuda()]
    return [result, kept] if case["keep"] else [result]
