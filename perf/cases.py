"""The work that a user of arma_amd has it do, as cases that can be timed.

Every case goes through the package's public entry points (Context, Batch,
Server).  A case is a dict of plain values; listed() are the fixed ones,
draw() makes more of the same ranges.

kinds of case
  surface    noise, AR recurrence and post-rescale of one surface, with the
             NIT transform of the realisation where "nit" names a target law
  potential  velocity potential of a surface on nz levels (linear or
             high-amplitude solver)
  batch      many uneven surfaces in one launch sequence
  setup      Choi solve and white-noise variance of a model on the GPU
  serve      a burst of requests to the serving loop: surfaces, some with
             their potential, and chunks of a realtime stream
"""
import ctypes
import math
import random

import numpy as np
import torch

import arma_amd
from arma_amd import _abi

DEV = "cuda:0"
DELTA = (2.0 * math.pi,) * 3
DEPTH = 12.0
GRAVITY = 9.82
DTYPE = {"fp32": torch.float32, "fp64": torch.float64}

# Stationary models: (ACF, order, alpha, beta) on a 10^3 unit grid.  The
# propagating ACF's coefficients are two columns wide, (order, order, 2), the
# standing wave's are a cube.
MODELS = {
    "propagating3": ("propagating", 3, 0.06, 0.8),
    "propagating5": ("propagating", 5, 0.05, 0.6),
    "propagating7": ("propagating", 7, 0.04, 1.2),
    "standing3": ("standing", 3, 0.06, 0.8),
    "standing5": ("standing", 5, 0.06, 0.8),
    "standing7": ("standing", 7, 0.06, 0.8),
    "standing9": ("standing", 9, 0.07, 0.6),
}
# Target laws of transform = nit.
NIT = {
    "gram_charlier": dict(distribution=arma_amd.NIT_GRAM_CHARLIER, skewness=3.25, kurtosis=2.4,
                          interval=(-5.0, 5.0)),
    "skew_normal": dict(distribution=arma_amd._abi.NIT_SKEW_NORMAL, mean=0.0, stdev=1.0,
                        alpha=1.0, interval=(-5.0, 5.0)),
}
NIT_EPS, NIT_ITERATIONS = 1e-6, 100


# ---- the cases ---------------------------------------------------------------

def surface(name, shape, model, precision, noise="p521", part=(32, 48, 48), nit=""):
    return dict(name=name, kind="surface", nt=shape[0], nx=shape[1], ny=shape[2], model=model,
                precision=precision, noise=noise, pt=part[0], px=part[1], py=part[2], nit=nit)


def potential(name, shape, nto, nz, precision, solver="linear"):
    return dict(name=name, kind="potential", nt=shape[0], nx=shape[1], ny=shape[2], nto=nto,
                nz=nz, precision=precision, solver=solver)


def listed():
    return [
        # the smallest request a server sees: one noise stream, four tiles
        surface("surface-32-fp32", (32, 32, 32), "propagating3", "fp32"),
        # the plain AR configuration a first user runs: framework=none's
        # single MT19937 stream, standing wave, order 7
        surface("surface-128x64x64-fp64", (128, 64, 64), "standing7", "fp64", noise="mt19937"),
        # the headline surface, one tile per CU
        surface("surface-1024x256x256-fp64", (1024, 256, 256), "propagating7", "fp64",
                part=(16, 32, 32)),
        # the precision configuration's surface, four tiles per CU
        surface("surface-2048x512x512-fp32", (2048, 512, 512), "propagating7", "fp32",
                part=(32, 64, 64)),
        # transform = nit on ragged extents
        surface("nit-300x100x150-fp64", (300, 100, 150), "standing5", "fp64", nit="gram_charlier"),
        # a server's potential: a small surface at two levels
        potential("potential-64x64x32-fp32", (64, 64, 32), 64, 2, "fp32"),
        # the headline potential
        potential("potential-1024x256x256-fp64", (1024, 256, 256), 1024, 16, "fp64"),
        # the precision configuration's potential, a quarter of its slices
        potential("potential-512x512x512-fp32", (512, 512, 512), 512, 32, "fp32"),
        # velocity_potential_solver = high_amplitude
        potential("high-amplitude-256x128x256-fp64", (256, 128, 256), 256, 8, "fp64",
                  "high_amplitude"),
        # an ensemble of uneven surfaces of mixed orders in one launch
        dict(name="batch-12-fp32", kind="batch", count=12, precision="fp32", tmin=64, tmax=512,
             xymin=32, xymax=320, layout=42),
        # fitting a model, which precedes every surface
        dict(name="setup-order7", kind="setup", acf="standing", order=7, grid=10, count=1),
        # a burst at a server
        dict(name="serve-6", kind="serve", surfaces=4, potentials=1, chunks=2, vmin=32768,
             vmax=1048576, layout=7),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    u = rng.random()
    if u < 0.42:
        model = rng.choice(sorted(MODELS))
        precision = rng.choice(["fp32", "fp64"])
        nt, nx, ny = log_int(16, 1024), log_int(16, 512), log_int(16, 512)
        noise = "mt19937" if nt * nx * ny <= 1 << 20 and rng.random() < 0.25 else "p521"
        parts = [(16, 16, 16), (16, 32, 32), (32, 48, 48), (32, 64, 64)]
        first = rng.randrange(4)
        part = next(p for p in parts[first:] + [(64, 64, 64)] if streams((nt, nx, ny), p) <= 4096)
        nit = rng.choice(sorted(NIT)) if rng.random() < 0.2 else ""
        c = surface("", (nt, nx, ny), model, precision, noise, part, nit)
    elif u < 0.80:
        nx, ny = 1 << rng.randint(4, 10), 1 << rng.randint(4, 10)
        precision = rng.choice(["fp32", "fp64"])
        solver = "high_amplitude" if rng.random() < 0.25 else "linear"
        nt = log_int(8, 512)
        nto = nt if rng.random() < 0.7 else rng.randint(1, nt)
        nz = log_int(1, 40)
        # at most 2^30 points of potential
        nto = max(1, min(nto, (1 << 30) // (nx * ny * nz)))
        c = potential("", (nt, nx, ny), nto, nz, precision, solver)
    elif u < 0.88:
        c = dict(kind="batch", count=rng.randint(4, 16), precision=rng.choice(["fp32", "fp64"]),
                 tmin=32, tmax=log_int(64, 512), xymin=32, xymax=log_int(64, 320),
                 layout=rng.randrange(1 << 20))
    elif u < 0.95:
        # one model, or the candidates of an ensemble (not every propagating
        # ACF of these ranges has a fit; an ensemble redraws those)
        count = rng.choice([1, 1, rng.randint(2, 24)])
        c = dict(kind="setup", acf="standing" if count == 1 else
                 rng.choice(["standing", "propagating"]), order=rng.randint(3, 9),
                 grid=rng.randint(10, 12), count=count)
    else:
        c = dict(kind="serve", surfaces=rng.randint(2, 8), potentials=rng.randint(0, 2),
                 chunks=rng.randint(0, 3), vmin=32768, vmax=log_int(65536, 4194304),
                 layout=rng.randrange(1 << 20))
    c.pop("name", None)
    return c


# ---- what a program has in hand ------------------------------------------------

_ctx = None


def context():
    """A program has one context, bound to torch's current stream."""
    global _ctx
    if _ctx is None:
        _ctx = arma_amd.Context(0)
    return _ctx


def make_acf(kind, alpha, beta, grid=10):
    func = _abi.ACF_STANDING_WAVE if kind == "standing" else _abi.ACF_PROPAGATING_WAVE
    k = (beta, beta) if kind == "standing" else (-beta, 0.0)
    return _abi.acf(func, (grid,) * 3, velocity=beta, alpha=(alpha,) * 3, beta=k)


_models = {}


def fitted(model):
    """(phi, white-noise variance, gamma0) of a named model."""
    if model not in _models:
        kind, order, alpha, beta = MODELS[model]
        acf = make_acf(kind, alpha, beta)
        phi, _ = _abi.yule_walker_choi(acf, order)
        _models[model] = phi, _abi.white_noise_variance(acf, phi), float(acf[0, 0, 0])
    return _models[model]


def streams(shape, part):
    return math.prod(-(-n // p) for n, p in zip(shape, part))


_params = None


def p521(n):
    """The first n dynamic-creator records of the shipped table."""
    global _params
    if _params is None:
        _params = _abi.dcmt_p521_params(4096)
    arr = (arma_amd.MtParams * n)()
    ctypes.memmove(arr, _params, ctypes.sizeof(arr))
    return arr


def noise_seeds(seed, n):
    return np.random.default_rng(seed).integers(0, 1 << 32, n, dtype=np.uint32)


def surface_desc(shape, model, precision, noise, part, seed):
    phi, varwn, _ = fitted(model)
    prec = arma_amd.FP32 if precision == "fp32" else arma_amd.FP64
    if noise == "mt19937":
        return arma_amd.Context.ar_desc(shape, phi, varwn, [arma_amd.mt19937_params()],
                                        seeds=noise_seeds(seed, 1), precision=prec,
                                        noise_mode=arma_amd.NOISE_SEQUENTIAL,
                                        algorithm=arma_amd.AR_WAVEFRONT)
    n = streams(shape, part)
    return arma_amd.Context.ar_desc(shape, phi, varwn, p521(n), seeds=noise_seeds(seed, n),
                                    noise_mode=arma_amd.NOISE_PARTITIONED, partition=part,
                                    precision=prec, algorithm=arma_amd.AR_WAVEFRONT)


def sea(shape, precision, seed):
    """A wavy surface: 48 travelling waves of random direction, phase and
    amplitude, roughened by noise as an AR surface is."""
    nt, nx, ny = shape
    rng = np.random.default_rng(seed)
    m = 48
    amp = rng.normal(size=m) / math.sqrt(m)
    w, kx, ky = rng.uniform(0.3, 1.4, m), rng.uniform(-0.9, 0.9, m), rng.uniform(-0.9, 0.9, m)
    ph = rng.uniform(0, 2 * math.pi, m)
    t = torch.arange(nt, dtype=torch.float64, device=DEV)[:, None]
    x = torch.arange(nx, dtype=torch.float64, device=DEV)[:, None, None]
    y = torch.arange(ny, dtype=torch.float64, device=DEV)[None, :, None]
    g = [torch.from_numpy(v).to(DEV) for v in (amp, w, kx, ky, ph)]
    at = t * g[1]
    axy = (x * g[2] + y * g[3] + g[4]).reshape(nx * ny, m)
    left = torch.cat([g[0] * torch.cos(at), -g[0] * torch.sin(at)], 1)
    right = torch.cat([torch.cos(axy), torch.sin(axy)], 1)
    z = torch.matmul(left, right.t()).reshape(nt, nx, ny)
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    z += 0.2 * torch.randn(z.shape, dtype=torch.float64, device=DEV, generator=gen)
    return z.to(DTYPE[precision]).contiguous()


def pot_desc(c):
    prec = arma_amd.FP32 if c["precision"] == "fp32" else arma_amd.FP64
    return arma_amd.Context.pot_desc((c["nt"], c["nx"], c["ny"]), DELTA, DEPTH, (0.0, -10.0),
                                     (float(c["nto"] - 1), 0.0), (c["nto"], c["nz"]), prec)


def members(c):
    """The surfaces of a batch: (shape, model)."""
    rng = random.Random(c["layout"])
    names = sorted(MODELS)
    return [((rng.randint(c["tmin"], c["tmax"]), rng.randint(c["xymin"], c["xymax"]),
              rng.randint(c["xymin"], c["xymax"])), rng.choice(names)) for _ in range(c["count"])]


def requests(c):
    """The burst of a serve case: (shape, model, levels of the potential or 0)
    of every surface request, and (nx, ny) of the realtime stream."""
    rng = random.Random(c["layout"])
    out = []
    for i in range(c["surfaces"]):
        v = math.exp(rng.uniform(math.log(c["vmin"]), math.log(c["vmax"])))
        nx, ny = rng.randint(32, 96), rng.randint(32, 96)
        nz = 0
        if i < c["potentials"]:
            nx, ny, nz = 64, 32, 2
        out.append(((max(16, int(v / (nx * ny))), nx, ny), rng.choice(sorted(MODELS)), nz))
    return out, (rng.randint(32, 200), rng.randint(32, 200))


CHUNK = 16


def prepare(case, seed):
    kind = case["kind"]
    if kind == "surface":
        shape = (case["nt"], case["nx"], case["ny"])
        desc = surface_desc(shape, case["model"], case["precision"], case["noise"],
                            (case["pt"], case["px"], case["py"]), seed)
        nit = None
        if case["nit"]:
            nit = arma_amd.nit_desc(absolute_error=NIT_EPS, max_iterations=NIT_ITERATIONS,
                                    **NIT[case["nit"]])
        return dict(kind=kind, ctx=context(), desc=desc, shape=shape, nit=nit,
                    gamma0=fitted(case["model"])[2],
                    zeta=torch.empty(shape, dtype=DTYPE[case["precision"]], device=DEV))
    if kind == "potential":
        shape = (case["nt"], case["nx"], case["ny"])
        return dict(kind=kind, ctx=context(), desc=pot_desc(case), solver=case["solver"],
                    zeta=sea(shape, case["precision"], seed),
                    phi=torch.empty((case["nto"], case["nz"], case["nx"], case["ny"]),
                                    dtype=DTYPE[case["precision"]], device=DEV))
    if kind == "batch":
        mem = members(case)
        descs = [surface_desc(s, m, case["precision"], "p521", (32, 48, 48), seed + 1000 * i)
                 for i, (s, m) in enumerate(mem)]
        prec = arma_amd.FP32 if case["precision"] == "fp32" else arma_amd.FP64
        batch = context().batch(descs, [fitted(m)[2] for _, m in mem], prec)
        arena = torch.empty(batch.arena_elements, dtype=DTYPE[case["precision"]], device=DEV)
        return dict(kind=kind, batch=batch, arena=arena, count=len(mem))
    if kind == "setup":
        return dict(kind=kind, ctx=context(), acfs=setup_acfs(case, seed), order=case["order"])
    reqs, (sx, sy) = requests(case)
    descs = []
    for i, (shape, model, nz) in enumerate(reqs):
        pot = None
        if nz:
            pot = pot_desc(dict(nt=shape[0], nx=shape[1], ny=shape[2], nto=shape[0], nz=nz,
                                precision="fp32"))
        descs.append((surface_desc(shape, model, "fp32", "p521", (32, 48, 48), seed + 1000 * i),
                      fitted(model)[2], pot, shape, nz))
    stream = None
    if case["chunks"]:
        cols = streams((1, sx, sy), (1, 48, 48))
        phi, varwn, _ = fitted("propagating7")
        stream = arma_amd.Context.ar_desc(
            (1, sx, sy), phi, varwn, p521(cols), seeds=noise_seeds(seed, 1),
            noise_mode=arma_amd.NOISE_PARTITIONED, partition=(CHUNK, 48, 48),
            precision=arma_amd.FP32, algorithm=arma_amd.AR_WAVEFRONT)
    server = arma_amd.Server(0, lanes=4, budget=16 << 30, precision=arma_amd.FP32, max_batch=32)
    return dict(kind=kind, server=server, descs=descs, stream=stream, chunks=case["chunks"])


def setup_acfs(case, seed):
    rng = np.random.default_rng(seed)
    return [make_acf(case["acf"], rng.uniform(0.04, 0.1), rng.uniform(0.5, 1.2), case["grid"])
            for _ in range(case["count"])]


# ---- one pass -------------------------------------------------------------------

def run(state):
    return _RUN[state["kind"]](state)


def run_surface(s):
    ctx, zeta = s["ctx"], s["zeta"]
    ctx.ar_generate(s["desc"], zeta)
    factor = ctx.rescale(zeta, s["shape"], s["desc"].precision, s["gamma0"])
    if s["nit"] is not None:
        ctx.nit_realisation(zeta, s["shape"], s["desc"].precision, s["gamma0"], s["nit"])
    return {"zeta": zeta, "factor": factor}


def run_potential(s):
    s["ctx"].linear_potential(s["desc"], s["zeta"], s["phi"], solver=s["solver"])
    return s["phi"]


def run_batch(s):
    s["batch"].generate(s["arena"])
    return [s["batch"].surface(s["arena"], i) for i in range(s["count"])]


def run_setup(s):
    ctx = s["ctx"]
    if len(s["acfs"]) == 1:
        sols = [ctx.yule_walker_choi(s["acfs"][0], s["order"])]
    else:
        sols = ctx.yule_walker_choi_many(s["acfs"], [s["order"]] * len(s["acfs"]))
    out = []
    for acf, sol in zip(s["acfs"], sols):
        # the coefficients in a cube of the largest order, beside their shape
        phi = np.zeros((s["order"],) * 3)
        shape, var, varwn = (0, 0, 0), 0.0, 0.0
        if sol is not None:
            shape, var = sol[0].shape, sol[1]
            phi[:shape[0], :shape[1], :shape[2]] = sol[0]
            varwn = ctx.white_noise_variance(acf, sol[0])
        out.append((phi, np.array(shape, np.int32), var, varwn))
    return out


def run_serve(s):
    srv = s["server"]
    ids = {}
    for i, (desc, gamma0, pot, _, _) in enumerate(s["descs"]):
        ids[srv.submit_surface(desc, gamma0, pot)] = i
    sid = None
    if s["stream"] is not None:
        sid = srv.open_stream(s["stream"], CHUNK)
        for k in range(s["chunks"]):
            ids[srv.submit_chunk(sid)] = len(s["descs"]) + k
    out = [None] * len(ids)
    left = len(ids)
    copy = arma_amd.lib().arma_hip_server_copy
    while left:
        for c in srv.poll(64, wait_ms=-1):
            if c.status != 0:
                raise RuntimeError(f"request {c.id}: status {c.status}")
            shape = tuple(c.shape)
            zeta = torch.empty(shape, dtype=torch.float32, device=DEV)
            _abi.check(copy(srv.h, zeta.data_ptr(), c.zeta, zeta.numel() * 4))
            got = {"zeta": zeta}
            if c.phi:
                phi = torch.empty((shape[0], s["descs"][ids[c.id]][4]) + shape[1:],
                                  dtype=torch.float32, device=DEV)
                _abi.check(copy(srv.h, phi.data_ptr(), c.phi, phi.numel() * 4))
                got["phi"] = phi
            out[ids[c.id]] = got
            srv.release(c.id)
            left -= 1
    if sid is not None:
        srv.close_stream(sid)
    return out


_RUN = {"surface": run_surface, "potential": run_potential, "batch": run_batch,
        "setup": run_setup, "serve": run_serve}


# ---- what a pass cannot do without --------------------------------------------------

def work(case):
    kind = case["kind"]
    es = 4 if case.get("precision", "fp32") == "fp32" else 8
    if kind == "surface":
        n = case["nt"] * case["nx"] * case["ny"]
        w = surface_work(n, case["model"], es)
        if case["nit"]:
            w["flops"] += 25 * 40.0 * n  # bisection steps, each one CDF
        return w
    if kind == "potential":
        return potential_work(case["nto"], case["nz"], case["nx"], case["ny"], es)
    if kind == "batch":
        return total(surface_work(math.prod(s), m, es) for s, m in members(case))
    if kind == "setup":
        # dense inverses and products up to the shell 3 l^2 + 3 l + 1
        f = sum(4.0 * (3 * l * l + 3 * l + 1) ** 3 for l in range(1, case["order"]))
        b = 8.0 * (case["grid"] ** 3 + case["order"] ** 3)
        return {"bytes": b * case["count"], "flops": f * case["count"]}
    reqs, (sx, sy) = requests(case)
    parts = [surface_work(math.prod(s), m, 4) for s, m, _ in reqs]
    parts += [potential_work(s[0], nz, s[1], s[2], 4) for s, _, nz in reqs if nz]
    parts += [surface_work(CHUNK * sx * sy, "propagating7", 4)] * case["chunks"]
    return total(parts)


def surface_work(n, model, es):
    # the surface written once; the recurrence, and about 30 operations per
    # normal variate
    return {"bytes": float(n * es), "flops": n * (2.0 * fitted(model)[0].size + 30.0)}


def potential_work(nto, nz, nx, ny, es):
    # every slice read once, every level written once; one real transform
    # per slice and one per level, and the window
    n = float(nx * ny)
    fft = 2.5 * n * math.log2(n)
    return {"bytes": es * n * nto * (1 + nz), "flops": nto * (fft + nz * (fft + 6.0 * n))}


def total(parts):
    parts = list(parts)
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


# ---- the same results in 64 bits, without the package -----------------------------------

def exact(case, seed):
    kind = case["kind"]
    if kind == "surface":
        shape = (case["nt"], case["nx"], case["ny"])
        if math.prod(shape) > 1 << 27:
            return None  # the noise alone would take too long here
        desc = surface_desc(shape, case["model"], case["precision"], case["noise"],
                            (case["pt"], case["px"], case["py"]), seed)
        zeta, factor = exact_surface(desc, shape, case["model"])
        if case["nit"]:
            zeta = exact_nit(zeta, fitted(case["model"])[2], **NIT[case["nit"]])
        return {"zeta": zeta, "factor": factor}
    if kind == "potential":
        shape = (case["nt"], case["nx"], case["ny"])
        return exact_potential(sea(shape, case["precision"], seed).double(), case["nto"],
                               case["nz"], case["solver"])
    if kind == "batch":
        mem = members(case)
        if sum(math.prod(s) for s, _ in mem) > 1 << 27:
            return None
        return [exact_surface(surface_desc(s, m, case["precision"], "p521", (32, 48, 48),
                                           seed + 1000 * i), s, m)[0]
                for i, (s, m) in enumerate(mem)]
    # setup: an order-recursive fit that stops by its own rule has no plain
    # closed form; serve: its surfaces are those of the surface cases
    return None


def exact_surface(desc, shape, model):
    phi, _, gamma0 = fitted(model)
    zeta = exact_recurrence(exact_noise(desc, shape), phi)
    nt, nx, ny = shape
    start = (nt // 2 * nx + nx // 2) * ny + ny // 2
    count = -(-nt // 2) * -(-nx // 2) * -(-ny // 2)
    run_ = zeta.reshape(-1)[start:start + count]
    factor = math.sqrt(gamma0 / float(run_.var(correction=1)))
    return zeta * factor, factor


def temper(x, p):
    x = x ^ (x >> np.uint32(p.shift0))
    x = x ^ ((x << np.uint32(p.shiftB)) & np.uint32(p.maskB))
    x = x ^ ((x << np.uint32(p.shiftC)) & np.uint32(p.maskC))
    return x ^ (x >> np.uint32(p.shift1))


def mt_words(mts, seeds, count):
    """count tempered words of every stream, (streams, count); the records
    differ in aaa only."""
    p = mts[0]
    nn, mm = p.nn, p.mm
    n = len(seeds)
    aaa = np.array([mts[i].aaa for i in range(n)], np.uint32)
    st = np.empty((nn, n), np.uint32)
    s = np.array(seeds, np.uint32)
    for k in range(nn):
        st[k] = s & np.uint32(p.wmask)
        s = np.uint32(1812433253) * (s ^ (s >> np.uint32(30))) + np.uint32(k + 1)

    def twist(hi, lo, src):
        x = (hi & np.uint32(p.umask)) | (lo & np.uint32(p.lmask))
        return src ^ (x >> np.uint32(1)) ^ (aaa * (x & np.uint32(1)))

    blocks = -(-count // nn)
    out = np.empty((blocks, nn, n), np.uint32)
    for b in range(blocks):
        new = st.copy()
        for k0 in range(0, nn - 1, nn - mm):
            k1 = min(k0 + nn - mm, nn - 1)
            if k0 < nn - mm:
                src = st[k0 + mm:k1 + mm]
                if k1 + mm > nn:
                    src = np.concatenate([st[k0 + mm:], new[:k1 + mm - nn]])
            else:
                src = new[k0 + mm - nn:k1 + mm - nn]
            new[k0:k1] = twist(st[k0:k1], st[k0 + 1:k1 + 1], src)
        new[nn - 1] = twist(st[nn - 1], new[0], new[mm - 1])
        st = new
        out[b] = temper(st, p)
    return out.reshape(blocks * nn, n).T[:, :count]


def normals(words, count):
    """The first count polar normals of every stream from its words."""
    w = words[:, :words.shape[1] // 4 * 4].reshape(words.shape[0], -1, 4)
    w = torch.from_numpy(np.ascontiguousarray(w).astype(np.int64)).to(DEV).double()

    def canonical(a, b):
        v = (a + b * 4294967296.0) / 18446744073709551616.0
        return torch.where(v >= 1.0, torch.full_like(v, math.nextafter(1.0, 0.0)), v)

    x = 2.0 * canonical(w[:, :, 0], w[:, :, 1]) - 1.0
    y = 2.0 * canonical(w[:, :, 2], w[:, :, 3]) - 1.0
    r2 = x * x + y * y
    ok = (r2 <= 1.0) & (r2 != 0.0)
    mult = torch.sqrt(-2.0 * torch.log(torch.where(ok, r2, torch.ones_like(r2))) / r2)
    place = torch.cumsum(ok, 1) - 1
    half = -(-count // 2)
    out = torch.full((w.shape[0], half, 2), math.nan, dtype=torch.float64, device=DEV)
    keep = ok & (place < half)
    row = torch.arange(w.shape[0], device=DEV)[:, None].expand_as(place)[keep]
    out[row, place[keep]] = torch.stack([y * mult, x * mult], 2)[keep]
    out = out.reshape(w.shape[0], -1)[:, :count]
    if bool(torch.isnan(out).any()):
        raise RuntimeError("too few words drawn")
    return out


def exact_noise(desc, shape):
    sd = math.sqrt(desc.varwn)
    eps = torch.empty(shape, dtype=torch.float64, device=DEV)
    if desc.noise_mode == arma_amd.NOISE_SEQUENTIAL:
        part = shape
    else:
        part = tuple(desc.partition)
    np_ = [-(-n // p) for n, p in zip(shape, part)]
    count = math.prod(min(n, p) for n, p in zip(shape, part))
    n = math.prod(np_)
    need = int(4 * (count / 2 + 1) / 0.785 * 1.02) + 800
    words = mt_words(desc.mts, desc.seeds[:n], need)
    step = max(1, (1 << 27) // need)
    for p0 in range(0, n, step):
        v = normals(words[p0:p0 + step], count)
        for p in range(p0, min(n, p0 + step)):
            lo = (p // (np_[1] * np_[2]) * part[0], p // np_[2] % np_[1] * part[1],
                  p % np_[2] * part[2])
            e = [min(part[d], shape[d] - lo[d]) for d in range(3)]
            eps[lo[0]:lo[0] + e[0], lo[1]:lo[1] + e[1], lo[2]:lo[2] + e[2]] = (
                v[p - p0, :math.prod(e)].reshape(e) * sd)
    return eps


def exact_recurrence(eps, phi):
    """zeta = eps + sum phi(k, i, j) zeta(t - k, x - i, y - j), with
    phi(0, 0, 0) on eps, along the planes t + x + y = s."""
    p0, p1, p2 = phi.shape
    nt, nx, ny = eps.shape
    z = torch.zeros((nt + p0, nx + p1, ny + p2), dtype=torch.float64, device=DEV)
    z[p0:, p1:, p2:] = eps * (1.0 + float(phi[0, 0, 0]))
    w1, w2 = (nx + p1) * (ny + p2), ny + p2
    k, i, j = [torch.from_numpy(v.reshape(-1)[1:]).to(DEV) for v in np.indices(phi.shape)]
    off = k * w1 + i * w2 + j
    coef = torch.from_numpy(np.ascontiguousarray(phi.reshape(-1)[1:])).to(DEV)
    x = torch.arange(nx, device=DEV)[:, None]
    y = torch.arange(ny, device=DEV)[None, :]
    xy = (x + y).reshape(-1)
    order = torch.argsort(xy)
    base = ((x + p1) * w2 + (y + p2)).reshape(-1)[order]
    xy = xy[order]
    sums = xy.cpu().numpy()
    flat = z.reshape(-1)
    for s in range(nt + nx + ny - 2):
        a = int(np.searchsorted(sums, s - nt + 1))
        b = int(np.searchsorted(sums, s, side="right"))
        if b > a:
            at = base[a:b] + (s - xy[a:b] + p0) * w1
            flat[at] += (flat[at[:, None] - off] * coef).sum(1)
    return z[p0:, p1:, p2:].contiguous()


def exact_nit(zeta, gamma0, distribution, interval, skewness=0.0, kurtosis=3.0, mean=0.0,
              stdev=1.0, alpha=0.0):
    """Bisection for F(c) = Phi(zeta / sqrt(gamma0)); it stops once the
    interval or the residual is within the error."""
    if distribution == arma_amd.NIT_GRAM_CHARLIER:
        def cdf(x):
            poly = (kurtosis * (3 * x - x ** 3) + skewness * (4 - 4 * x * x) + 3 * x ** 3 - 9 * x)
            return (torch.exp(-0.5 * x * x) * poly / (24.0 * 2.506628274631)
                    + 0.5 * torch.erf(x / 1.4142135623731) + 0.5)
    else:
        gx, gw = np.polynomial.legendre.leggauss(20)

        def cdf(x):
            h = (x - mean) / stdev
            owen = torch.zeros_like(h)
            for u, w in zip(gx[10:], gw[10:]):
                term = 1.0 + alpha * alpha * u * u
                owen += w * torch.exp(-0.5 * h * h * term) / term
            return (0.5 * torch.erfc(-h / math.sqrt(2.0)) - 2.0 * owen * alpha / (2.0 * math.pi))

    y = 0.5 * torch.erfc(-(zeta / math.sqrt(gamma0)) / math.sqrt(2.0))
    a, b = torch.full_like(y, interval[0]), torch.full_like(y, interval[1])
    fa, fb = cdf(a) - y, cdf(b) - y
    out = torch.empty_like(y)
    live = torch.ones_like(y, dtype=torch.bool)
    for i in range(NIT_ITERATIONS):
        c = 0.5 * (a + b)
        fc = cdf(c) - y
        left = fa * fc < 0.0
        b, fb = torch.where(left, c, b), torch.where(left, fc, fb)
        right = fb * fc < 0.0
        a, fa = torch.where(right, c, a), torch.where(right, fc, fa)
        out = torch.where(live, c, out)
        live &= ((b - a) > NIT_EPS) & (fc.abs() > NIT_EPS)
        if not bool(live.any()):
            break
    return out


def derivative(z, dim, d):
    """Second-order differences along dim; the values themselves where the
    extent is below three."""
    n = z.shape[dim]
    if n < 3:
        return z.clone()

    def at(i):
        return z.narrow(dim, i, 1)

    inner = 0.5 * (z.narrow(dim, 2, n - 2) - z.narrow(dim, 0, n - 2)) / d
    first = 0.5 * (-at(2) + 4.0 * at(1) - 3.0 * at(0)) / d
    last = 0.5 * (3.0 * at(n - 1) - 4.0 * at(n - 2) + at(n - 3)) / d
    return torch.cat([first, inner, last], dim)


def largest_wave_number(lines, t, dt):
    """1 / (smallest wave number) of the waves between the local extrema of
    the lines, scanned one line after the other."""
    z0, z1, z2 = lines[:, 1:-1], lines[:, :-2], lines[:, 2:]
    dw1, dw2 = (z0 - z1).reshape(-1), (z0 - z2).reshape(-1)
    event = ((dw1 > 0.0) == (dw2 > 0.0)).nonzero()[:, 0]
    dw1, dw2, z0 = dw1[event], dw2[event], z0.reshape(-1)[event]
    a = -0.5 * (dw1 + dw2) / (dt * dt)
    b = dw1 / dt - a * dt * (2.0 * t - 1.0)
    c = z0 - t * dt * (a * t * dt + b)
    period = -0.5 * b / a
    elev = c + period * (b + a * period)
    up = elev > 0.0
    r = torch.cat([torch.zeros(1, dtype=torch.long, device=DEV),
                   torch.cumsum((up[1:] != up[:-1]).long(), 0)])
    runs = int(r[-1]) + 1
    top = torch.zeros(runs, dtype=torch.float64, device=DEV).scatter_reduce(
        0, r, elev.abs(), "amax", include_self=False)
    place = torch.arange(len(r), device=DEV)
    place = torch.where(elev.abs() == top[r], place, len(r))
    first = torch.full((runs,), len(r), device=DEV).scatter_reduce(0, r, place, "amin")
    rep = period[first][:runs - 1]  # the last run stays open
    if len(rep) < 2:
        return 1.0 / 1.7976931348623157e308
    w = 2.0 * math.pi / ((rep[1:] - rep[:-1]).abs() * 2.0)
    return 1.0 / float((w * w / GRAVITY).min())


def exact_potential(zeta, nto, nz, solver):
    nt, nx, ny = zeta.shape
    step = (float(nto - 1) - 0.0) / max(nto - 1, 1)
    times = [int(0.0 + step * i) for i in range(nto)]
    dz = 10.0 / max(nz - 1, 1)
    zt = derivative(zeta, 0, DELTA[0])
    out = torch.empty((nto, nz, nx, ny), dtype=torch.float64, device=DEV)
    px = torch.arange(nx, dtype=torch.float64, device=DEV)[:, None]
    py = torch.arange(ny, dtype=torch.float64, device=DEV)[None, :]
    levels = torch.tensor([-10.0 + dz * j for j in range(nz)], dtype=torch.float64,
                          device=DEV)[:, None, None]
    for i, it in enumerate(times):
        s = zeta[it]
        t = int(DELTA[0] * it)
        wx = largest_wave_number(s.t().contiguous(), t, DELTA[0])
        wy = largest_wave_number(s, t, DELTA[0])
        if solver == "linear":
            f = (-zt[it]).to(torch.complex128)
        else:
            zx, zy = derivative(s, 0, DELTA[1]), derivative(s, 1, DELTA[2])
            n = torch.sqrt(1.0 + zx * zx + zy * zy)
            f = zt[it] / torch.complex(-1.0 / n, (zx + zy) / n - zx - zy)
        u, v = px * (wx / max(nx - 1, 1)), py * (wy / max(ny - 1, 1))
        l = 2.0 * math.pi * torch.sqrt(u * u + v * v)
        l[0, 0] = l[1, 1]
        l = torch.roll(l, (nx // 2, ny // 2), (0, 1))
        w = (4.0 * math.pi * (torch.exp(l * levels) + torch.exp(-l * (levels + 2.0 * DEPTH)))
             / (1.0 + torch.exp(-2.0 * DEPTH * l)))
        out[i] = torch.fft.ifft2(torch.fft.fft2(f) * w).real
    # the edge points, each on the plane through three neighbours
    f = out
    corner = f[..., 1, 1] - (f[..., 2, 1] - f[..., 1, 1]) - (f[..., 1, 2] - f[..., 1, 1])
    f[..., 1:, 0] = f[..., 1:, 1] - (f[..., :-1, 2] - f[..., :-1, 1])
    f[..., 0, 0] = corner
    f[..., 0, 1] = f[..., 1, 1] - (f[..., 2, 0] - f[..., 1, 0])
    f[..., 0, 2:] = f[..., 1, 2:] - (f[..., 2, 1:-1] - f[..., 1, 1:-1])
    return out
