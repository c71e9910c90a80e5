"""Performance cases of the per-bin control-variate integrator, through its public entry points.

A case is one dict of plain values:
  path      host    integrate() on numpy bins, as a program ported from the reference calls it
            device  Context.integrate_device on GPU bins
            batch   Context.integrate_batch on GPU bins
            train   Context.refiner_train, then the trained parameters
  family    blobs2 (static blobs + step + wave), moving3 (moving blobs x occluder),
            lobes5 (5-D lobes x steps x cosine), poly (degree <= 4 in `dim` dims)
  form      crespo2021, fixed (weight 1), alpha1, importance, rr_pdf, fubini (regions over
            the first two dims, the rest by Monte Carlo)
  count     integrals per call; res0 x res1 bins, `regions` and `spp` of each (uneven: drawn
            per integral up to these)
  f64       double bins and arithmetic instead of float
  learned   refinement priority from the trained network instead of the heuristic
"""
import ctypes as C
import math

import numpy as np
import torch

import viltrum_amd as V
from viltrum_amd import integrands as I
from viltrum_amd import refiner as R

_EPOCHS = 2  # of a training case


def _case(name=None, **kw):
    c = dict(path="device", family="blobs2", form="crespo2021", dim=2, count=1, res0=64, res1=64, regions=1024, spp=16,
             f64=False, learned=False, uneven=False)
    c.update(kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one small integral from host code: a preview, an inner call of a larger program
        _case("preview_host", path="host", res0=20, res1=15, regions=192, spp=8),
        # the 2-D workload of the README and the benchmark's config 1: 64 x 64 bins
        _case("single_host", path="host", regions=1024, spp=16),
        # one ordinary image-sized integral per call, the plain path of the benchmark
        _case("single_2d", res0=512, res1=512, regions=2048, spp=55),
        # a rendered image with a time dimension (motion blur), the benchmark's config 2
        _case("motion_3d", family="moving3", dim=3, res0=512, res1=512, regions=16384, spp=64),
        # the same image with the time dimension by Monte Carlo: integrator_crespo2021_infinite<2>
        _case("motion_fubini", family="moving3", form="fubini", dim=3, res0=512, res1=512, regions=16384, spp=64),
        # a double-precision reference image on an odd grid (how truths are computed)
        _case("reference_f64", form="fixed", res0=301, res1=217, regions=20000, spp=64, f64=True),
        # a queue of unlike integrals in one call, the benchmark's config 3
        _case("uneven_batch", path="batch", family="mixed", count=256, res0=256, res1=256, regions=32768, spp=64,
              uneven=True),
        # many alike integrals with the learned priority, the benchmark's default workload
        _case("learned_batch", path="batch", count=64, res0=512, res1=512, regions=4096, spp=16, learned=True),
        # the importance-sampled residual over a batch of images
        _case("importance_batch", path="batch", form="importance", count=64, res0=256, res1=256, regions=4096, spp=16),
        # light transport in 5 dims, one integral on an odd grid with the heuristic
        _case("lobes_5d", family="lobes5", dim=5, res0=333, res1=250, regions=10000, spp=16),
        # the largest: 16 five-dimensional images, learned priority, the benchmark's config 5
        _case("learned_5d_batch", path="batch", family="lobes5", dim=5, count=16, res0=1024, res1=1024, regions=65536,
              spp=32, learned=True),
        # training of the 2-D priority network on pairs of 96 integrands
        _case("train_2d", path="train", count=96, res0=512, res1=512, regions=4096, spp=0),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["host", "host", "single", "single", "motion", "fubini", "f64", "uneven", "learned", "variant",
                       "five", "learned5", "poly", "train"])
    r0 = _log(rng, 16, 700)
    r1 = max(4, min(700, int(r0 * rng.uniform(0.5, 1.5))))
    spp = _log(rng, 2, 64)
    if kind == "host":
        return _case(path="host", res0=_log(rng, 8, 128), res1=_log(rng, 8, 128), regions=_log(rng, 32, 4096), spp=spp,
                     f64=rng.random() < 0.3)
    if kind == "single":
        return _case(res0=r0, res1=r1, regions=_log(rng, 256, 32768), spp=spp,
                     form=rng.choice(["crespo2021", "crespo2021", "fixed", "alpha1"]))
    if kind == "motion":
        return _case(family="moving3", dim=3, res0=r0, res1=r1, regions=_log(rng, 512, 32768), spp=spp)
    if kind == "fubini":
        return _case(family="moving3", form="fubini", dim=3, res0=r0, res1=r1, regions=_log(rng, 512, 32768), spp=spp)
    if kind == "f64":
        return _case(form=rng.choice(["crespo2021", "fixed"]), res0=min(r0, 400), res1=min(r1, 400),
                     regions=_log(rng, 512, 32768), spp=spp, f64=True)
    if kind == "uneven":
        return _case(path="batch", family="mixed", count=_log(rng, 8, 256), res0=256, res1=256,
                     regions=_log(rng, 4096, 32768), spp=64, uneven=True)
    if kind == "learned":
        return _case(path=rng.choice(["batch", "batch", "device"]), count=_log(rng, 2, 64), res0=min(r0, 512),
                     res1=min(r1, 512), regions=_log(rng, 512, 16384), spp=min(spp, 32), learned=True)
    if kind == "variant":
        return _case(path="batch", form=rng.choice(["importance", "rr_pdf"]), count=_log(rng, 2, 64),
                     res0=min(r0, 256), res1=min(r1, 256), regions=_log(rng, 512, 8192), spp=min(spp, 32))
    if kind == "five":
        return _case(family="lobes5", dim=5, res0=min(r0, 512), res1=min(r1, 512), regions=_log(rng, 1024, 40000),
                     spp=min(spp, 32))
    if kind == "learned5":
        return _case(path="batch", family="lobes5", dim=5, count=_log(rng, 2, 12), res0=min(r0, 512),
                     res1=min(r1, 512), regions=_log(rng, 2048, 40000), spp=min(spp, 32), learned=True)
    if kind == "poly":
        return _case(family="poly", dim=rng.choice([1, 2, 3, 4]), res0=r0, res1=r1, regions=_log(rng, 256, 8192),
                     spp=spp, f64=rng.random() < 0.3)
    return _case(path="train", count=_log(rng, 16, 128), res0=512, res1=512, regions=_log(rng, 512, 4096), spp=0)


# ---------------------------------------------------------------- inputs

def _poly(seed, dim):
    rng = I.SplitMix64(seed)
    terms = [(rng.uniform(0.5, 1.5), (0,) * dim)]
    for _ in range(5):
        terms.append((rng.uniform(-0.5, 1.0), tuple(rng.integer(0, 4) for _ in range(dim))))
    return I.poly(terms, dim)


def _items(c, seed):
    """(integrand, resolution, regions, spp) of each integral of the case."""
    base = 3_000_000 + 1009 * int(seed)
    if c["uneven"]:
        # the mix of sizes is the case's, the integrands are the seed's
        k = c["regions"] / 32768.0
        out = []
        for i, x in enumerate(I.config3_batch(seed=c["count"], count=c["count"])):
            f, nb = x["integrand"], x["integrand"].params.nblobs
            f = I.c1_family(base + i, nb) if f.dim == 2 else I.moving_blobs(base + i, nb)
            out.append((f, x["res"], max(16, int(x["regions"] * k)), x["spp"]))
        return out
    out = []
    res = (c["res0"],) if c["dim"] == 1 else (c["res0"], c["res1"])
    for i in range(c["count"]):
        if c["family"] == "blobs2":
            f = I.config4_integrand(base + i)
        elif c["family"] == "moving3":
            f = I.moving_blobs(base + i, 32)
        elif c["family"] == "lobes5":
            f = I.config5(base + i)
        else:
            f = _poly(base + i, c["dim"])
        out.append((f, res, c["regions"], c["spp"]))
    return out


def _integrator(c, regions, spp, seed):
    kw = {"refiner": V.REFINER_LEARNED} if c["learned"] else {}
    form, n = c["form"], regions - 1
    if form == "fubini":
        return V.integrator_crespo2021_infinite(2, n, 4, spp, seed=seed)
    if form == "fixed":
        return V.integrator_variance_reduction_fixed(1.0, n, spp, seed=seed, **kw)
    if form == "alpha1":
        return V.integrator_adaptive_control_variates_parallel(n, spp, seed=seed, **kw)
    if form == "importance":
        return V.integrator_variance_reduction_importance(n, spp, seed=seed, **kw)
    if form == "rr_pdf":
        return V.integrator_variance_reduction_rr_pdf(n, spp, seed=seed, **kw)
    return V.integrator_crespo2021(n, spp, seed=seed, **kw)


_train_ctx = None  # training replaces its context's network, so it has a context of its own
_networks = set()


def _trainer():
    global _train_ctx
    if _train_ctx is None:
        _train_ctx = V.Context(0)
    return _train_ctx


def _context(c):
    """The program's one context; with the learned priority its network, trained once."""
    ctx = V.default_context()
    if c["learned"] and c["dim"] not in _networks:
        if c["dim"] == 2:
            R.train(ctx, count=128, regions=4096, epochs=4, seed=0)
        else:
            R.train(ctx, count=16, regions=16384, res=(1024, 1024), epochs=3, seed=0, dim=5)
        _networks.add(c["dim"])
    return ctx


def prepare(case, seed):
    c = _case(**case)
    if c["path"] == "train":
        ps, fs = R.training_set(c["count"], c["regions"], (c["res0"], c["res1"]), seed0=5_000_000 + 1009 * int(seed))
        return {"case": c, "ctx": _trainer(), "problems": ps, "fs": fs}
    items = _items(c, seed)
    if c["path"] == "host":
        f, res, regions, spp = items[0]
        return {"case": c, "ctx": _context(c), "f": f, "res": res, "range": V.range_primary(f.dim),
                "dtype": np.float64 if c["f64"] else np.float32,
                "integrator": _integrator(c, regions, spp, int(seed) & 0xFFFF)}
    dtype = torch.float64 if c["f64"] else torch.float32
    scalar = V.F64 if c["f64"] else V.F32
    sizes = [int(np.prod(res)) for _, res, _, _ in items]
    # each integral's bins in one tensor, from a multiple of 64 bins
    starts = np.concatenate([[0], np.cumsum([(s + 63) // 64 * 64 for s in sizes])])
    bins = torch.zeros(int(starts[-1]), dtype=dtype, device="cuda")
    problems, fs, ptrs = [], [], []
    for i, (f, res, regions, spp) in enumerate(items):
        integ = _integrator(c, regions, spp, (int(seed) + i) & 0xFFFF)
        g, rng = integ.prepare(f, V.range_primary(f.dim))
        problems.append(integ.problem(g, res, rng, scalar))
        fs.append(g)
        ptrs.append(bins.data_ptr() + int(starts[i]) * bins.element_size())
    torch.cuda.synchronize()
    return {"case": c, "ctx": _context(c), "problems": problems, "fs": fs, "ptrs": ptrs, "bins": bins}


def run(state):
    c, ctx = state["case"], state["ctx"]
    if c["path"] == "train":
        ctx.refiner_train(state["problems"], state["fs"], epochs=_EPOCHS, seed=1)
        return ctx.refiner_get(2)
    if c["path"] == "host":
        bins = np.zeros(state["res"], dtype=state["dtype"])
        return V.integrate(state["integrator"], bins, state["f"], state["range"], ctx=ctx)
    stream = torch.cuda.current_stream().cuda_stream
    if c["form"] == "alpha1":  # this form adds to the bins
        state["bins"].zero_()
        torch.cuda.current_stream().synchronize()
    if c["path"] == "batch":
        ctx.integrate_batch(state["problems"], state["fs"], state["ptrs"], stream)
    else:
        for p, f, ptr in zip(state["problems"], state["fs"], state["ptrs"]):
            ctx.integrate_device(p, f, ptr, stream)
    return state["bins"]


# ---------------------------------------------------------------- the work a pass cannot do without

def work(case):
    c = _case(**case)
    if c["path"] == "train":
        # every region and every node above it is a pair: forward and backward per epoch
        kp, budgets = 32, (0.25, 0.5, 1.0, 2.0)
        pairs = sum(2 * max(2, int(c["regions"] * budgets[i % 4])) - 1 for i in range(c["count"]))
        per = 128 * (kp + 128) + 256 * kp + 49152
        # each pair's FP64 target is an 81-point quadrature of f - P
        f, _ = I.flops_per_eval(I.config4_integrand(0))
        return {"bytes": float(pairs) * (2 * kp + 4) * _EPOCHS, "flops": float(pairs) * (per * _EPOCHS + 81 * (f + 16))}
    width = 8 if c["f64"] else 4
    nbytes = flops = 0.0
    for f, res, regions, spp in _items(c, 0):
        bins = float(np.prod(res))
        rd = 2 if c["form"] == "fubini" else f.dim
        fe, _ = I.flops_per_eval(f)
        per_node = fe * (4 if c["form"] == "fubini" else 1)
        nbytes += bins * width + C.sizeof(f.params)
        # each residual sample: f and the region's polynomial; each split: two new planes of nodes
        flops += bins * spp * (fe + 2 * (3 ** rd - 1)) + (3 ** rd + (regions - 1) * 2 * 3 ** (rd - 1)) * per_node
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------- exact values in 64 bits

def _edges(n, dev):
    return torch.arange(n + 1, dtype=torch.float64, device=dev) / n


def _blobs2_exact(f, res, dev):
    """Bin averages of blobs + step + wave: products of erf differences, of sine and cosine
    integrals, and the area of each bin beyond the step's line."""
    p = f.params
    x, y = _edges(res[0], dev), _edges(res[1], dev)
    out = torch.zeros(res, dtype=torch.float64, device=dev)
    for k in range(p.nblobs):
        cx, cy, _, _, ax, ay, w = list(p.blob[k])
        ex = torch.erf(math.sqrt(ax) * (x - cx)).diff() * math.sqrt(math.pi / ax) / 2
        ey = torch.erf(math.sqrt(ay) * (y - cy)).diff() * math.sqrt(math.pi / ay) / 2
        out += w * ex[:, None] * ey[None, :]
    wa, fx, fy = list(p.wave)
    if wa:
        out += wa * (-torch.cos(fx * x).diff() / fx)[:, None] * (torch.sin(fy * y).diff() / fy)[None, :]
    if p.step_mode == 1:
        a, b, _, d, h = list(p.step)
        # d2/dxdy of max(ax + by - d, 0)^2 / (2ab) is the step
        q = (a * x[:, None] + b * y[None, :] - d).clamp(min=0.0) ** 2 / (2 * a * b)
        out += h * q.diff(dim=0).diff(dim=1)
    return out * (res[0] * res[1])


def _moving3_exact(f, res, dev):
    """Bin averages of moving blobs x occluder: the x integral in closed form between the
    occluder's line and the bin's edge, Gauss-Legendre over y (3 points a bin) and t (24
    panels of 3)."""
    p = f.params
    a, b, ct, d, _ = list(p.step)
    gx, gw = np.polynomial.legendre.leggauss(3)
    nt = 24
    ts = np.concatenate([(i + (gx + 1) / 2) / nt for i in range(nt)])
    tw = np.tile(gw / 2 / nt, nt)
    x = _edges(res[0], dev)
    lo, hi = x[:-1, None], x[1:, None]
    out = torch.zeros(res, dtype=torch.float64, device=dev)
    j = torch.arange(res[1], dtype=torch.float64, device=dev)
    for gy, wy in zip(gx, gw):
        y = (j + (gy + 1) / 2) / res[1]
        for t, wt in zip(ts, tw):
            edge = ((d - b * y - ct * t) / a)[None, :]
            l, h = (torch.minimum(torch.maximum(lo, edge), hi), hi.expand(res)) if a > 0 else (
                lo.expand(res), torch.maximum(torch.minimum(hi, edge), lo))
            acc = torch.zeros(res, dtype=torch.float64, device=dev)
            inside = (h > l).double()
            r, q = ((h > l) & ((l > lo) | (h < hi))).nonzero(as_tuple=True)  # bins that the occluder cuts
            xl, xh = l[r, q], h[r, q]
            for k in range(p.nblobs):
                cx, cy, vx, vy, ax, ay, w = list(p.blob[k])
                s, c = math.sqrt(ax), cx + vx * t
                wyk = w * math.sqrt(math.pi / ax) / 2 * torch.exp(-ay * (y - (cy + vy * t)) ** 2)
                whole = torch.erf(s * (x - c)).diff()
                acc += whole[:, None] * wyk[None, :]
                if r.numel():
                    acc[r, q] += (torch.erf(s * (xh - c)) - torch.erf(s * (xl - c)) - whole[r]) * wyk[q]
            acc *= inside
            out += acc * (wy / 2 / res[1] * wt)
    return out * (res[0] * res[1])


def _poly_exact(f, res, dev):
    p = f.params
    out = torch.zeros(res, dtype=torch.float64, device=dev)
    for m in range(p.nterms):
        t = torch.ones((), dtype=torch.float64, device=dev) * p.coef[m]
        for d in range(f.dim):
            e = p.expo[m][d]
            if d < len(res):
                v = (_edges(res[d], dev) ** (e + 1)).diff() / (e + 1) * res[d]
                t = t[..., None] * v if t.dim() else t * v
            else:
                t = t / (e + 1)
        out += t
    return out


def exact(case, seed):
    """The bin averages themselves, which every path estimates.  None for the 5-D family
    (two half-spaces through all dims: no closed form), for trained parameters, and where
    the estimate's own noise can pass a tenth of the values (the Fubini form, the heavy
    1/pdf tails of importance sampling, few samples)."""
    c = _case(**case)
    if c["path"] == "train" or c["family"] == "lobes5" or c["form"] in ("fubini", "importance"):
        return None
    if not c["uneven"] and min(c["spp"], 16) * c["regions"] < 2048:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    parts = []
    items = _items(c, seed)
    if c["uneven"] and sum(r[0] * r[1] for f, r, _, _ in items if f.dim == 3) > 1 << 19:
        return None  # minutes of quadrature for all its 3-D integrals
    for f, res, _, _ in items:
        if f.family == I.FAMILY_BLOBS:
            v = _blobs2_exact(f, res, dev) if f.dim == 2 else _moving3_exact(f, res, dev)
        else:
            v = _poly_exact(f, res, dev)
        parts.append(v)
    if c["path"] == "host":
        return parts[0].cpu().numpy()
    flat = []
    for v in parts:
        flat.append(v.reshape(-1))
        flat.append(torch.zeros(-v.numel() % 64, dtype=torch.float64, device=dev))
    return torch.cat(flat)
