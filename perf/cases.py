"""Timed cases of the NUFFT engine, through the package's public entry points.

listed() names fixed workloads, draw() makes more of the same ranges,
prepare() builds a plan and its device inputs, run() does one pass, work()
states the least bytes and flops of a pass, tolerance() the agreement of two
correct implementations, exact() the same transform as FP64 direct sums.

Sizes are those of the benchmark configurations (128 x 128 modes with 1e5
points, 128^3 with 1e7, 1024^2 with 5e7, 64 uneven 2D plans, radial 3D
spokes, 3D type 3 with 1e6 sources and targets) and generic odd ones between
them.
"""
import math

import numpy as np
import torch

import wgpunufft_amd as W

PREC = {"f32": W.F32, "f64": W.F64}
REAL = {"f32": torch.float32, "f64": torch.float64}
CPLX = {"f32": torch.complex64, "f64": torch.complex128}


def _single(name, kind, modes, points, eps, prec="f32", dist="uniform", step="encode",
            spread="plain", order="index", batch=1, isign=1, mode_order=0):
    """One plan: `step` "encode" bins the points and transforms, "execute"
    transforms over points that were bound once."""
    case = {"call": "plan", "kind": kind, "dim": len(modes), "points": points, "eps": eps,
            "prec": prec, "dist": dist, "step": step, "spread": spread, "order": order,
            "batch": batch, "isign": isign, "mode_order": mode_order}
    for a, n in enumerate(modes):
        case["n%d" % a] = n
    if name:
        case["name"] = name
    return case


def _many(name, kind, count, eps, table, points_lo=10_000, points_hi=2_000_000, modes_lo=64,
          modes_hi=512):
    case = {"call": "many", "kind": kind, "count": count, "eps": eps, "table": table,
            "points_lo": points_lo, "points_hi": points_hi, "modes_lo": modes_lo,
            "modes_hi": modes_hi}
    if name:
        case["name"] = name
    return case


def _type3(name, dim, sources, targets, reach, band, eps, prec="f64"):
    """Sources in [-reach, reach]^dim, targets in [-band, band]^dim."""
    case = {"call": "type3", "dim": dim, "points": sources, "targets": targets, "reach": reach,
            "band": band, "eps": eps, "prec": prec}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # one small 2D slice evaluated at a few thousand points: launch latency
        _single("t2_2d_small", 2, [91, 67], 10_007, 1e-5),
        # the 2D image-sized gridding call (benchmark configuration 1)
        _single("t1_2d_128", 1, [128, 128], 100_000, 1e-6),
        # 1D nonuniform spectra of long odd-length signals, in double
        _single("t1_1d_f64", 1, [49_999], 300_007, 1e-9, prec="f64"),
        # the 3D headline pair: gridding with the matrix-core spread, output
        # independent of the point order, and interpolation; half the points
        # in one dense cluster
        _single("t1_3d_mfma", 1, [128, 128, 128], 10_000_000, 1e-6, dist="cluster",
                spread="mfma_f16x3", order="coordinates"),
        _single("t2_3d", 2, [128, 128, 128], 10_000_000, 1e-6, dist="cluster"),
        # a default plan on a ragged 3D grid
        _single("t1_3d_plain", 1, [120, 97, 75], 2_000_003, 1e-6),
        # double precision, 3D: gridding, and repeated evaluation at points
        # bound once (the forward model of an iterative solver)
        _single("t1_3d_f64", 1, [64, 64, 64], 1_000_000, 1e-9, prec="f64"),
        _single("t2_3d_f64_bound", 2, [81, 64, 50], 1_000_003, 1e-9, prec="f64", step="execute",
                isign=-1, mode_order=1),
        # very many points on a large 2D grid (benchmark configuration 3)
        _single("t1_2d_50m", 1, [1024, 1024], 50_000_000, 1e-6),
        # 64 independent 2D problems of uneven sizes in one call
        # (benchmark configuration 4a)
        _many("t2_2d_many", 2, 64, 1e-5, 4),
        # 16 coils over one bound set of radial spokes (configuration 4b)
        _single("t1_3d_radial", 1, [256, 256, 256], 8192 * 512, 1e-6, dist="radial",
                step="execute", spread="mfma_f16x3", batch=16),
        # 3D type 3 (benchmark configuration 5)
        _type3("t3_3d", 3, 1_000_000, 1_000_000, 5.0, 200.0, 1e-10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choices(["1d", "2d", "3d", "many", "coils", "type3"], [1, 4, 6, 2, 1, 2])[0]
    prec = "f64" if rng.random() < 0.3 else "f32"
    eps = rng.choice([1e-6, 1e-9, 1e-12] if prec == "f64" else [1e-3, 1e-4, 1e-5, 1e-6])
    kind = rng.choice([1, 2])
    if what == "many":
        hi = _log(rng, 30_000, 2_000_000)
        return _many("", kind, rng.randint(8, 64), rng.choice([1e-3, 1e-5, 1e-6]),
                     rng.randint(1, 10_000), max(1_000, hi // 100), hi, 48, _log(rng, 96, 512))
    if what == "type3":
        band = float(_log(rng, 10, 150))
        return _type3("", rng.choice([2, 3, 3]), _log(rng, 10_000, 1_000_000),
                      _log(rng, 10_000, 1_000_000), round(rng.uniform(1.0, 5.0), 2), band,
                      eps, prec)
    if what == "coils":
        n = [rng.randint(40, 200) for _ in range(3)]
        return _single("", kind, n, _log(rng, 100, 4_000) * 512, rng.choice([1e-4, 1e-6]),
                       dist="radial", step="execute", batch=rng.randint(2, 8),
                       spread=rng.choice(["plain", "mfma_f16x3"]) if kind == 1 else "plain")
    if what == "1d":
        modes, points = [_log(rng, 1_000, 200_000)], _log(rng, 10_000, 10_000_000)
    elif what == "2d":
        modes = [_log(rng, 48, 1024) for _ in range(2)]
        points = _log(rng, 10_000, 50_000_000)
    else:
        modes = [_log(rng, 24, 160) for _ in range(3)]
        points = _log(rng, 10_000, 10_000_000 if prec == "f32" else 4_000_000)
    spread = order = None
    if what == "3d" and prec == "f32" and kind == 1 and rng.random() < 0.4:
        spread = "mfma_f16x3"
    if kind == 1 and rng.random() < 0.25:
        order = "coordinates"
    return _single("", kind, modes, points, eps, prec, rng.choice(["uniform", "cluster"]),
                   rng.choice(["encode", "encode", "execute"]), spread or "plain",
                   order or "index", isign=rng.choice([1, -1]), mode_order=rng.choice([0, 1]))


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _modes(case):
    return [case["n%d" % a] for a in range(case["dim"])]


def _coordinates(case, g):
    """Points in [-pi, pi)^dim, point-major: uniform; half uniform and half a
    wrapped Gaussian cluster (sigma 0.05) in shuffled order; or 512 samples
    along spokes through the origin in random directions."""
    M, d, real = case["points"], case["dim"], REAL[case["prec"]]
    if case["dist"] == "radial":
        spokes = M // 512
        v = torch.randn(spokes, d, generator=g, device="cuda", dtype=torch.float64)
        v /= v.norm(dim=1, keepdim=True)
        t = -math.pi + 2 * math.pi * torch.arange(512, device="cuda", dtype=torch.float64) / 512
        x = (v[:, None, :] * t[None, :, None]).reshape(M, d)
    else:
        x = torch.rand(M, d, generator=g, device="cuda", dtype=torch.float64)
        x = (2 * x - 1) * math.pi
        if case["dist"] == "cluster":
            half = M // 2
            centre = torch.tensor([0.3, -1.1, 2.0][:d], device="cuda", dtype=torch.float64)
            z = torch.randn(half, d, generator=g, device="cuda", dtype=torch.float64)
            x[:half] = torch.remainder(centre + 0.05 * z + math.pi, 2 * math.pi) - math.pi
            x = x[torch.randperm(M, generator=g, device="cuda")]
    top = math.nextafter(math.pi, 0) if case["prec"] == "f64" else 3.14159250
    return x.clamp(-top, top).to(real).contiguous()


def _complex(n, dtype, g):
    return torch.randn(n, generator=g, device="cuda", dtype=dtype)


def _problems(case):
    """(n0, n1, points) of each plan of a batch, log-uniform."""
    r = np.random.RandomState(case["table"])

    def pick(lo, hi):
        return int(round(math.exp(r.uniform(math.log(lo), math.log(hi)))))
    return [(pick(case["modes_lo"], case["modes_hi"]), pick(case["modes_lo"], case["modes_hi"]),
             pick(case["points_lo"], case["points_hi"])) for _ in range(case["count"])]


def _plan_inputs(case, seed):
    g = _generator(seed)
    x = _coordinates(case, g)
    per = case["points"] if case["kind"] == 1 else int(np.prod(_modes(case)))
    return x, _complex(case["batch"] * per, CPLX[case["prec"]], g)


def _many_inputs(case, seed):
    g = _generator(seed)
    xs, vs = [], []
    for n0, n1, M in _problems(case):
        x = (2 * torch.rand(M, 2, generator=g, device="cuda") - 1) * 3.1415925
        xs.append(x)
        vs.append(_complex(M if case["kind"] == 1 else n0 * n1, torch.complex64, g))
    return xs, vs


def _type3_inputs(case, seed):
    g = _generator(seed)

    def box(n, r):
        return ((2 * torch.rand(n, case["dim"], generator=g, device="cuda",
                                dtype=torch.float64) - 1) * (r * (1 - 1e-6))).to(
                                    REAL[case["prec"]])
    return (box(case["points"], case["reach"]), box(case["targets"], case["band"]),
            _complex(case["points"], CPLX[case["prec"]], g))


def prepare(case, seed):
    if case["call"] == "many":
        xs, vs = _many_inputs(case, seed)
        plans, outs = [], []
        for (n0, n1, M), x in zip(_problems(case), xs):
            plans.append(W.NufftPlan(case["kind"], W.NufftConfig([n0, n1], case["eps"])))
            outs.append(torch.empty(n0 * n1 if case["kind"] == 1 else M, dtype=torch.complex64,
                                    device="cuda"))
        return {"case": case, "plans": plans, "x": xs, "v": vs, "out": outs}
    if case["call"] == "type3":
        x, s, c = _type3_inputs(case, seed)
        d = case["dim"]
        plan = W.NufftType3Plan(d, [(-case["reach"], case["reach"])] * d,
                                [(-case["band"], case["band"])] * d, eps=case["eps"],
                                precision=PREC[case["prec"]])
        out = torch.empty(case["targets"], dtype=c.dtype, device="cuda")
        return {"case": case, "plan": plan, "x": x, "s": s, "v": c, "out": out}
    x, v = _plan_inputs(case, seed)
    cfg = (W.NufftConfig(_modes(case), case["eps"]).with_precision(PREC[case["prec"]])
           .with_isign(case["isign"]).with_mode_order(case["mode_order"])
           .with_batch(case["batch"]))
    plan = W.NufftPlan(case["kind"], cfg)
    if case["spread"] != "plain":
        plan.set_spread_method(case["spread"])
    if case["order"] != "index":
        plan.set_point_order(case["order"])
    each = cfg.mode_count() if case["kind"] == 1 else case["points"]
    out = torch.empty(case["batch"] * each, dtype=v.dtype, device="cuda")
    if case["step"] == "execute":
        plan.set_points_gpu(x)
    return {"case": case, "plan": plan, "x": x, "v": v, "out": out}


def run(state):
    case = state["case"]
    if case["call"] == "many":
        encode = W.encode_type1_many if case["kind"] == 1 else W.encode_type2_many
        return encode(state["plans"], state["x"], state["v"], state["out"])
    if case["call"] == "type3":
        return state["plan"].encode_gpu(state["x"], state["v"], state["s"], out=state["out"])
    if case["step"] == "execute":
        return state["plan"].execute_gpu(state["v"], out=state["out"])
    return state["plan"].encode_gpu(state["x"], state["v"], out=state["out"])


def _width(eps):
    """Cells per axis of the spreading kernel at upsampling factor 2."""
    return int(math.ceil(-math.log10(eps) - 1e-9)) + 1


def _fft_flops(cells):
    return 5.0 * cells * math.log2(max(cells, 2))


def work(case):
    """Inputs read once, outputs written once; 4 w^d flops for each point and
    vector and one fine-grid FFT (upsampling 2) for each vector."""
    w = _width(case["eps"])
    if case["call"] == "many":
        b = f = 0.0
        for n0, n1, M in _problems(case):
            b += M * (8 + 8) + 8.0 * n0 * n1
            f += 4.0 * w * w * M + _fft_flops(4.0 * n0 * n1)
        return {"bytes": b, "flops": f}
    d = case["dim"]
    size = 4 if case["prec"] == "f32" else 8
    if case["call"] == "type3":
        M, N = case["points"], case["targets"]
        axis = 8.0 / math.pi * case["reach"] * case["band"] + 2 * w
        return {"bytes": float((M + N) * size * (d + 2)),
                "flops": 4.0 * w ** d * (M + N) + _fft_flops(axis ** d)}
    N = float(np.prod(_modes(case)))
    M, B = case["points"], case["batch"]
    return {"bytes": M * size * (d + 2.0 * B) + 2.0 * size * N * B,
            "flops": B * (4.0 * w ** d * M + _fft_flops(2.0 ** d * N))}


def tolerance(case):
    """Two correct transforms at one requested accuracy differ by their
    kernels' truncation (eps and a few) and by the rounding of the sums."""
    rounding = 4e-14 if case.get("prec") == "f64" else 1e-6
    return {"rel": 8.0 * case["eps"] + rounding + _phase_rounding(case)}


def _phase_rounding(case):
    """Rounding of FP64 phases k x and s x, which grows with the largest
    frequency; single-precision type 3 rounds its targets' positions."""
    if case["call"] == "type3":
        return case["reach"] * case["band"] * (6e-8 if case["prec"] == "f32" else 2e-16)
    if case.get("prec") == "f64":
        return 2e-16 * max(_modes(case))
    return 0.0


# complex multiply-adds that the direct sums of one case may take
_EXACT_MOST = 6e13


def _phases(x, n, sign, order):
    """exp(sign i k x) for the n modes of one axis in the plan's order."""
    k = torch.arange(n, device=x.device, dtype=torch.float64) - n // 2
    if order == 1:
        k = torch.cat([k[n // 2:], k[:n // 2]])
    p = sign * x[:, None] * k[None, :]
    return torch.complex(torch.cos(p), torch.sin(p))


def _direct(kind, modes, x, v, sign, order, batch):
    """Type-1 or type-2 sums in FP64, the axes' phases as matrix products
    over chunks of points."""
    x, v = x.double(), v.to(torch.complex128)
    M, d = x.shape
    n0, outer = modes[0], int(np.prod(modes[1:]))
    v = v.view(batch, M) if kind == 1 else v.view(batch, outer, n0)
    if kind == 1:
        out = torch.zeros(outer, batch * n0, dtype=torch.complex128, device=x.device)
    else:
        out = torch.empty(batch, M, dtype=torch.complex128, device=x.device)
    chunk = max(256, min(1 << 20, (1 << 28) // (max(outer, n0 * batch) + n0)))
    for at in range(0, M, chunk):
        p = x[at:at + chunk]
        e = _phases(p[:, 0], n0, sign, order)
        rest = torch.ones(p.shape[0], 1, dtype=torch.complex128, device=x.device)
        for a in range(1, d):
            q = _phases(p[:, a], modes[a], sign, order)
            rest = (q[:, :, None] * rest[:, None, :]).reshape(p.shape[0], -1)
        if kind == 1:
            c = v[:, at:at + chunk].t()
            out += rest.t() @ (c[:, :, None] * e[:, None, :]).reshape(p.shape[0], -1)
        else:
            for b in range(batch):
                out[b, at:at + chunk] = ((e @ v[b].t()) * rest).sum(dim=1)
    if kind == 1:
        out = out.view(outer, batch, n0).transpose(0, 1)
    return out.reshape(-1).contiguous()


def exact(case, seed):
    if case["call"] == "many":
        xs, vs = _many_inputs(case, seed)
        return [_direct(case["kind"], [n0, n1], x, v, 1, 0, 1)
                for (n0, n1, M), x, v in zip(_problems(case), xs, vs)]
    if case["call"] == "type3":
        if case["points"] * case["targets"] > 1.5e11:
            return None
        x, s, c = _type3_inputs(case, seed)
        x, s, c = x.double(), s.double(), c.to(torch.complex128)
        out = []
        for at in range(0, s.shape[0], 256):
            p = s[at:at + 256] @ x.t()
            out.append(torch.complex(torch.cos(p), torch.sin(p)) @ c)
        return torch.cat(out)
    modes = _modes(case)
    if float(np.prod(modes)) * case["points"] * case["batch"] > _EXACT_MOST:
        return None
    x, v = _plan_inputs(case, seed)
    return _direct(case["kind"], modes, x, v, case["isign"], case["mode_order"], case["batch"])
