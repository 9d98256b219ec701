"""Workloads whose speed this library is judged by, through its public entry
points: the drop-in batch step on host patches, uniform domains resident on
the device, a flood-scenario ensemble, a resident AMR flood and refinement
tagging, over the patch sizes, methods and problem sizes users run.

A case is a dict of plain values:

  kind "batch"     HostBatch.step over n host patches of mx x mx cells (a
                   ForestClaw rank's level), maux aux fields per cell
  kind "brick"     a domain of mi x mj patches restarted from a state kept on
                   the device, advanced by `steps` attempts and downloaded
  kind "ensemble"  `members` flood scenarios of mixed sizes in one pool, all
                   advanced by `steps` attempts, then polled and downloaded
  kind "amr"       an adaptively refined flood advanced by `steps` accepted
                   steps, regrids included, then downloaded
  kind "tag"       refinement flags of n patches

order, transverse and limiter name the method (limiter 4 is MC, 1 minmod);
wet is the share of the domain's height under the initial reservoir (1: a
radial dam break with no dry cell); tune: the program has autotuned the step
variant beforehand, as the benchmark does.
"""
from __future__ import annotations

import ctypes as ct
import math

import numpy as np
import torch

import geoflood_amd as gf
from geoflood_amd.amr import AmrRun
from geoflood_amd.pool import BrickLayout, HostBatch, Pool

GRAV, DRYTOL = 9.81, 1e-3
SECOND = dict(order=2, transverse=2, limiter=4)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a rank that owns a handful of patches: the latency of one call
        dict(name="batch16_few", kind="batch", mx=16, n=4, maux=1, **SECOND),
        # a level of a mid-size run, an odd count, bound by the host transfers
        dict(name="batch32_level", kind="batch", mx=32, n=1001, maux=1, **SECOND),
        # first-order run with capacity and friction fields beside the bathymetry
        dict(name="batch64_first_order", kind="batch", mx=64, n=90, maux=3, order=1, transverse=0, limiter=4),
        # the 256^2 radial dam break of 100 steps: every cell wet, few patches
        dict(name="brick32_radial", kind="brick", mx=32, mi=8, mj=8, steps=100, wet=1.0, tune=False, **SECOND),
        # smallest patches, wet/dry fronts
        dict(name="brick8_dam", kind="brick", mx=8, mi=61, mj=47, steps=100, wet=0.5, tune=False, **SECOND),
        # 16x16 patches with a method other than the default one
        dict(name="brick16_minmod", kind="brick", mx=16, mi=63, mj=50, steps=60, wet=0.7, tune=False, order=2,
             transverse=1, limiter=1),
        # largest patches, autotuned
        dict(name="brick64_dam", kind="brick", mx=64, mi=15, mj=17, steps=100, wet=0.6, tune=True, **SECOND),
        # the 4096^2 dam break: an eighth wet, most patches dry and still
        dict(name="brick32_4096", kind="brick", mx=32, mi=128, mj=128, steps=200, wet=0.25, tune=True, **SECOND),
        # serving: live scenarios of all sizes between two harvests
        dict(name="ensemble", kind="ensemble", members=24, steps=128),
        # the overland flood on 16x16 patches, levels 1-4, a regrid every 4 steps
        dict(name="amr16_flood", kind="amr", mx=16, maxlevel=4, steps=400),
        # the same on 32x32 patches and a shallower tree
        dict(name="amr32_flood", kind="amr", mx=32, maxlevel=3, steps=200),
        # tagging a large level
        dict(name="tag32", kind="tag", mx=32, n=4000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["batch", "batch", "brick", "brick", "brick", "ensemble", "amr", "tag"])
    method = rng.choice([SECOND, SECOND, SECOND, dict(order=2, transverse=1, limiter=1),
                         dict(order=2, transverse=2, limiter=3), dict(order=1, transverse=0, limiter=4)])
    mx = rng.choice([8, 16, 32, 64])
    if kind == "batch":
        return dict(kind=kind, mx=mx, n=_log_int(rng, 1, 2.0 ** 20 / mx ** 2), maux=rng.choice([1, 1, 2, 3]), **method)
    if kind == "brick":
        cells = math.exp(rng.uniform(math.log(96.0 ** 2), math.log(1400.0 ** 2)))
        aspect = math.exp(rng.uniform(-0.7, 0.7))
        mi = max(2, round(math.sqrt(cells * aspect) / mx))
        mj = max(2, round(math.sqrt(cells / aspect) / mx))
        return dict(kind=kind, mx=mx, mi=mi, mj=mj, steps=rng.randint(40, 160),
                    wet=rng.choice([1.0, round(rng.uniform(0.2, 0.9), 3)]), tune=rng.random() < 0.5, **method)
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(3, 30), steps=rng.randint(32, 128))
    if kind == "amr":
        mx = rng.choice([8, 16, 32])
        return dict(kind=kind, mx=mx, maxlevel=3 if mx == 32 else rng.choice([3, 4]), steps=rng.randint(60, 240))
    return dict(kind=kind, mx=mx, n=_log_int(rng, 50, 2.0 ** 22 / mx ** 2))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _fractal(ny, nx, rms, gen):
    """Terrain with power spectrum |k|^-2, zero mean, the given RMS (metres)."""
    dev = _device()
    noise = torch.randn(ny, nx, dtype=torch.float64, generator=gen).to(dev)
    ky = torch.fft.fftfreq(ny, dtype=torch.float64, device=dev)[:, None]
    kx = torch.fft.rfftfreq(nx, dtype=torch.float64, device=dev)[None, :]
    k = torch.sqrt(kx * kx + ky * ky)
    k[0, 0] = math.inf
    z = torch.fft.irfft2(torch.fft.rfft2(noise) / k, s=(ny, nx))
    z = z - z.mean()
    return z * (rms / z.std())


def _mirror(f):
    """The field with two ghost rows and columns as walls mirror them."""
    for d in (0, 1):
        n = f.shape[d]
        f = f.index_select(d, torch.tensor([1, 0, *range(n), n - 1, n - 2], device=f.device))
    return f


def _tiles(p, mx):
    """(patches, mx+4, mx+4) tiles of a padded field."""
    return p.unfold(0, mx + 4, mx).unfold(1, mx + 4, mx).reshape(-1, mx + 4, mx + 4)


def _brick_fields(case, seed):
    """h, hu, hv, b of the whole domain and the cell size."""
    gen = torch.Generator().manual_seed(seed)
    ny, nx = case["mj"] * case["mx"], case["mi"] * case["mx"]
    dev = _device()
    if case["wet"] >= 1.0:  # radial dam break on a flat bed, the dam's place drawn
        dx = 1.0 / max(nx, ny)
        c = 0.4 + 0.2 * torch.rand(2, dtype=torch.float64, generator=gen)
        x = (torch.arange(nx, dtype=torch.float64, device=dev) + 0.5) / nx - float(c[0])
        y = (torch.arange(ny, dtype=torch.float64, device=dev) + 0.5) / ny - float(c[1])
        h = torch.where(x[None, :] ** 2 + y[:, None] ** 2 < 0.04, 2.0, 1.0).to(torch.float64)
        b = torch.zeros_like(h)
    else:  # a reservoir over fractal terrain, dry elsewhere
        dx = 1.0
        x = (torch.arange(nx, dtype=torch.float64, device=dev) + 0.5) * dx
        b = _fractal(ny, nx, 3.0, gen) - x[None, :] / 500.0
        h = torch.zeros_like(b)
        h[int((1.0 - case["wet"]) * ny):, :(nx + 1) // 2] = 10.0
    z = torch.zeros_like(h)
    return h, z, z, b, dx


def _batch_patches(case, seed):
    """Patches with filled ghost cells mid-flood: pools and dry ground over
    fractal terrain, currents of a few m/s.  Returns q (n, mx+4, mx+4, 3), aux
    (n, mx+4, mx+4, maux), dx and dt as numpy."""
    gen = torch.Generator().manual_seed(seed)
    mx, n = case["mx"], case["n"]
    mi = max(1, math.isqrt(n))
    mj = -(-n // mi)
    shape = (mj * mx + 4, mi * mx + 4)
    b = _fractal(*shape, 1.5, gen)
    h = torch.clamp(0.5 - b, min=0.0)
    u, v = _fractal(*shape, 0.7, gen), _fractal(*shape, 0.7, gen)
    q = torch.stack([_tiles(f, mx)[:n] for f in (h, h * u, h * v)], -1)
    aux = _tiles(b, mx)[:n, :, :, None].repeat(1, 1, 1, case["maux"])
    if case["maux"] > 1:
        aux[..., 1:] = 1.0
    return q.contiguous().cpu().numpy(), aux.contiguous().cpu().numpy(), 2.0, 0.03


def _hills(ny, nx, ly, lx, gen, count=24):
    """A valley falling in +x with Gaussian hills, made from one matrix product."""
    r = torch.rand(4, count, dtype=torch.float64, generator=gen).numpy()
    amp, wid = 5.0 * r[0], 20.0 + 180.0 * r[1]
    x, y = (np.arange(nx) + 0.5) * lx / nx, (np.arange(ny) + 0.5) * ly / ny
    gx = np.exp(-((x[None, :] - r[2][:, None] * lx) ** 2) / (2.0 * wid[:, None] ** 2))
    gy = np.exp(-((y[None, :] - r[3][:, None] * ly) ** 2) / (2.0 * wid[:, None] ** 2))
    return (gy * amp[:, None]).T @ gx + 0.002 * (lx - x)[None, :]


def _hydrograph(peak, strip, length):
    t = np.linspace(0.0, 3600.0, 61)
    return dict(time=t, hu=peak * np.sin(np.pi * t / 3600.0) / strip, b=strip, x0=0.0, y0=0.5 * length)


def _upload(pool, layout, h, hu, hv, b):
    """One brick's fields into its slots (buffer 0)."""
    m = layout.mx
    q = torch.stack([_tiles(_mirror(f), m) for f in (h, hu, hv)], -1).contiguous().cpu().numpy()
    aux = _tiles(_mirror(b), m)[..., None].contiguous().cpu().numpy()
    pool.upload_aos(layout.first, q, aux)


def _params(case, manning):
    m = {k: case.get(k, SECOND[k]) for k in SECOND}
    gf.set_params(grav=GRAV, dry_tolerance=DRYTOL, manning_n=manning, order=m["order"], transverse=m["transverse"],
                  mthlim=(m["limiter"],) * 3)


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
_READY = []


def _init():
    if not _READY:
        gf.init(0)
        _READY.append(True)


def prepare(case, seed):
    _init()
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["kind"]](state)


def _prepare_batch(case, seed):
    _params(case, 0.03)
    q, aux, dx, dt = _batch_patches(case, seed)
    # the driver's own patch arrays, bound once as its plugin binds them
    return dict(kind="batch", q=q, batch=HostBatch(list(q), list(aux), dx, dx), dt=dt)


def _run_batch(s):
    return s["q"], s["batch"].step(0.0, s["dt"])


def _prepare_brick(case, seed):
    _params(case, 0.03)
    h, hu, hv, b, dx = _brick_fields(case, seed)
    live = BrickLayout(case["mi"], case["mj"], case["mx"], case["mx"], dx, dx)
    kept = BrickLayout(case["mi"], case["mj"], case["mx"], case["mx"], dx, dx)
    n = live.npatch
    pool = Pool(case["mx"], case["mx"], 2 * n)
    pool.set_layout([live, kept])
    _upload(pool, kept, h, hu, hv, b)
    s = dict(kind="brick", pool=pool, live=live, n=n, steps=case["steps"], dt0=0.1 * dx if case["wet"] < 1 else 0.02 * dx,
             src=np.arange(n, 2 * n, dtype=np.int32), dst=np.arange(n, dtype=np.int32), sid=None,
             out=np.zeros((n, case["mx"] + 4, case["mx"] + 4, 3)))
    if case["tune"]:
        _restart(s)
        pool.run(10)
        pool.autotune(reps=3)
    return s


def _restart(s):
    """The scenario from its kept initial state."""
    if s["sid"] is not None:
        s["pool"].remove_scenario(s["sid"])
    s["pool"].move(s["src"], s["dst"], 0)
    s["sid"] = s["pool"].add_scenario(s["live"], dt0=s["dt0"])


def _download(pool, first, out, buf):
    """Slots [first, first + len(out)) into an array the program keeps."""
    gf.check(gf.load().gf_pool_download(pool.h, first, len(out), buf, gf.dptr(out)), "gf_pool_download")


def _interior(out):
    return out[:, 2:-2, 2:-2]  # a device-resident run's ghost cells are scratch


def _run_brick(s):
    _restart(s)
    s["pool"].run(s["steps"])
    info = s["pool"].scenario(s["sid"])
    _download(s["pool"], 0, s["out"], info["cur"])
    return _interior(s["out"]), info["t"], info["dt"], info["maxcfl"], info["nsteps"], info["retakes"]


def _members(case, seed):
    """(patches a side, Manning n, peak discharge) of each scenario."""
    rng = np.random.default_rng(seed)
    sides = rng.choice([4, 8, 16, 32], p=[0.4, 0.3, 0.2, 0.1], size=case["members"])
    sides[0] = 16
    return [(int(m), float(rng.uniform(0.02, 0.06)), float(np.exp(rng.uniform(np.log(20.0), np.log(2000.0)))))
            for m in sorted(sides)]


def _prepare_ensemble(case, seed):
    _params(case, 0.035)
    mix = _members(dict(members=case["members"]), 12345 + case["members"])  # sizes by the case, terrain by the seed
    gen = torch.Generator().manual_seed(seed)
    layouts = [BrickLayout(m, m, 32, 32, 2000.0 / (32 * m), 2000.0 / (32 * m), mthbc=(0, 1, 3, 3)) for m, _, _ in mix]
    pool = Pool(32, 32, sum(lay.npatch for lay in layouts))
    pool.set_layout(layouts)
    sids = []
    for lay, (m, manning, peak) in zip(layouts, mix):
        b = torch.from_numpy(_hills(32 * m, 32 * m, 2000.0, 2000.0, gen))
        z = torch.zeros_like(b)
        _upload(pool, lay, z, z, z, b)
        sid = pool.add_scenario(lay, dt0=1.0)
        pool.set_friction(sid, manning)
        pool.set_dt_max(sid, 10.0)
        pool.set_inflow(sid, **_hydrograph(peak, 100.0, 2000.0))
        sids.append(sid)
    pool.run(400)  # under way: floods of different ages and extents
    return dict(kind="ensemble", pool=pool, layouts=layouts, count=len(sids), steps=case["steps"],
                out=np.zeros((pool.n, 36, 36, 3)))


def _run_ensemble(s):
    s["pool"].run(s["steps"])
    rec = s["pool"].scenarios(0, s["count"])
    for k, lay in enumerate(s["layouts"]):
        _download(s["pool"], lay.first, s["out"][lay.first:lay.first + lay.npatch], int(rec["cur"][k]))
    return _interior(s["out"]), rec["t"], rec["dt"], rec["maxcfl"], rec["nsteps"], rec["retakes"]


def _prepare_amr(case, seed):
    _params(case, 0.035)
    nx0 = 64 // case["mx"]

    def dem(nx, ny, level):
        return _hills(ny, nx, 2000.0, 2000.0, torch.Generator().manual_seed(seed))

    r = AmrRun(case["mx"], nx0, nx0, 2000.0, 2000.0, 1, case["maxlevel"], dem, (nx0 << case["maxlevel"]) ** 2,
               mthbc=(0, 1, 3, 3), hydro=_hydrograph(200.0, 100.0, 2000.0), eta_tol=0.01, regrid_interval=4, dt_max=10.0)
    r.start(0.0, 1.0)
    r.run(100)  # the flood under way
    return dict(kind="amr", run=r, steps=case["steps"], out=np.zeros((r.capacity, case["mx"] + 4, case["mx"] + 4, 3)),
                level=np.zeros(r.capacity, dtype=np.int32))


def _run_amr(s):
    r = s["run"]
    info = r.run(s["steps"])
    # the leaves' states in slot order, the rest of the program's arrays empty
    n = len(r.forest)
    _download(r.pool, r.half * r.capacity, s["out"][:n], info["cur"])
    s["out"][n:] = 0.0
    s["level"][:n][r.perm] = r.forest.L
    s["level"][n:] = -1
    return _interior(s["out"]), s["level"], info["t"], info["dt"], info["nsteps"], info["retakes"]


def _prepare_tag(case, seed):
    _params(case, 0.03)
    q, aux, dx, _ = _batch_patches(dict(case, maux=1), seed)
    n = len(q)
    # still water over most of the level, waves in some patches
    calm = torch.rand(n, generator=torch.Generator().manual_seed(seed + 1)).numpy() < 0.7
    q[calm, :, :, 1:] = 0.0
    pool = Pool(case["mx"], case["mx"], n)
    pool.set_patches(np.full(n, dx), np.full(n, dx), np.arange(n) * case["mx"] * dx, np.zeros(n))
    pool.upload_aos(0, q, aux)
    return dict(kind="tag", pool=pool, patches=np.arange(n, dtype=np.int32))


def _run_tag(s):
    return s["pool"].tag_refine(s["patches"], t=10.0, level=2, maxlevel=4, wave_tolerance=0.55, deep_depth=100.0,
                                max_level_deep=4, speed_tolerance=(1.0, 2.0, 3.0, 4.0), sea_level=0.5)


_PREPARE = dict(batch=_prepare_batch, brick=_prepare_brick, ensemble=_prepare_ensemble, amr=_prepare_amr,
                tag=_prepare_tag)
_RUN = dict(batch=_run_batch, brick=_run_brick, ensemble=_run_ensemble, amr=_run_amr, tag=_run_tag)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
FLOPS_PER_CELL = 900  # two Riemann problems, limiters, transverse splits and friction of a wet cell


def work(case):
    k = case["kind"]
    if k == "batch":
        cells = case["n"] * (case["mx"] + 4) ** 2
        return dict(bytes=cells * 8 * (3 + case["maux"] + 3), flops=0.6 * case["n"] * case["mx"] ** 2 * FLOPS_PER_CELL)
    if k == "tag":
        return dict(bytes=case["n"] * case["mx"] ** 2 * 32, flops=case["n"] * case["mx"] ** 2 * 12)
    if k == "brick":  # the wet part steps, the still dry part is left as it is
        wet = case["mi"] * case["mj"] * case["mx"] ** 2 * min(1.0, 0.55 * case["wet"] if case["wet"] < 1 else 1.0)
        cells = case["mi"] * case["mj"] * (case["mx"] + 4) ** 2
    elif k == "ensemble":
        cells = 36 ** 2 * sum(m * m for m, _, _ in _members(dict(members=case["members"]), 12345 + case["members"]))
        wet = 0.2 * cells
    else:
        cells = 0.9 * (64 << case["maxlevel"]) ** 2
        wet = 0.1 * cells
    return dict(bytes=case["steps"] * wet * 56 + cells * 24, flops=case["steps"] * wet * FLOPS_PER_CELL)


# ---------------------------------------------------------------------------
# the same step in plain torch, 64 bits
# ---------------------------------------------------------------------------
def _where0(c, x):
    return torch.where(c, x, torch.zeros_like(x))


def _middle(hL, hR, uL, uR):
    """Middle depth and speeds of the homogeneous Riemann problem (one Newton step)."""
    g = GRAV
    lo, hi = torch.minimum(hL, hR), torch.maximum(hL, hR)
    du, sL, sR = uR - uL, torch.sqrt(g * hL), torch.sqrt(g * hR)
    Fmin = du + 2.0 * (torch.sqrt(g * lo) - torch.sqrt(g * hi))
    Fmax = du + (hi - lo) * torch.sqrt(0.5 * g * (hi + lo) / (hi * lo))
    rr = torch.clamp(-du + 2.0 * (sL + sR), min=0.0) ** 2 / (16.0 * g)  # two rarefactions
    gL, gR = torch.sqrt(0.5 * g * (1 / hi + 1 / hL)), torch.sqrt(0.5 * g * (1 / hi + 1 / hR))
    F0 = du + (hi - hL) * gL + (hi - hR) * gR
    dF = gL - g * (hi - hL) / (4 * hi * hi * gL) + gR - g * (hi - hR) / (4 * hi * hi * gR)
    ss = (torch.sqrt(hi) - F0 / (2.0 * torch.sqrt(hi) * dF)) ** 2      # two shocks
    sr = lo - Fmin / ((Fmax - Fmin) / (hi - lo))                       # one of each
    rare, shock = Fmin > 0, Fmax <= 0
    hm = torch.where(rare, rr, torch.where(shock, ss, sr))
    c = torch.sqrt(g * hm)
    A, B = uL + 2 * sL, uR - 2 * sR
    u1 = uL - (hm - hL) * torch.sqrt(0.5 * g * (1 / hm + 1 / hL))
    u2 = uR + (hm - hR) * torch.sqrt(0.5 * g * (1 / hm + 1 / hR))
    left = hL > hR
    s1 = torch.where(rare, A - 3 * c, torch.where(shock, u1 - c, torch.where(left, A - 3 * c, B + c)))
    s2 = torch.where(rare, B + 3 * c, torch.where(shock, u2 + c, torch.where(left, A - c, B + 3 * c)))
    dry = lo <= DRYTOL
    sd = uR + uL - 2 * sR + 2 * sL
    return torch.where(dry, 0.0, hm), torch.where(dry, sd, s1), torch.where(dry, sd, s2)


def _solve(L, R):
    """Speeds (3) and f-waves (3 x (h, normal, transverse)) of the faces
    between states L and R = (h, hn, ht, b)."""
    g = GRAV
    hL, nL, tL, bL = L
    hR, nR, tR, bR = R
    wL, wR = hL > DRYTOL, hR > DRYTOL
    any_wet = wL | wR
    hL, nL, tL, hR, nR, tR = (_where0(w, x) for w, x in ((wL, hL), (wL, nL), (wL, tL), (wR, hR), (wR, nR), (wR, tR)))
    one = torch.ones_like(hL)
    dL, dR = torch.where(wL, hL, one), torch.where(wR, hR, one)
    uL, vL, uR, vR = nL / dL, tL / dL, nR / dR, tR / dR
    pL, pR = 0.5 * g * hL ** 2 + nL * nL / dL, 0.5 * g * hR ** 2 + nR * nR / dR
    # a dry side: a wall if the water cannot climb it
    hw, uw = torch.where(wR, dR, dL), torch.where(wR, -uR, uL)
    hs = torch.maximum(hw, _middle(hw, hw, uw, -uw)[0])
    rdry, ldry = wL & ~wR, wR & ~wL
    rwall, lwall = rdry & (hs + bL < bR), ldry & (hs + bR < bL)
    bR = torch.where(rdry & ~rwall & (hL + bL < bR), hL + bL, bR)
    bL = torch.where(ldry & ~lwall & (hR + bR < bL), hR + bR, bL)
    hR, nR, bR, pR, uR, vR = (torch.where(rwall, x, y) for x, y in
                              ((hL, hR), (-nL, nR), (bL, bR), (pL, pR), (-uL, uR), (vL, vR)))
    hL, nL, bL, pL, uL, vL = (torch.where(lwall, x, y) for x, y in
                              ((hR, hL), (-nR, nL), (bR, bL), (pR, pL), (-uR, uL), (vR, vL)))
    hL, hR = torch.where(any_wet, hL, one), torch.where(any_wet, hR, one)
    sgL, sgR = torch.sqrt(g * hL), torch.sqrt(g * hR)
    uh = (sgL * uL + sgR * uR) / (sgR + sgL)
    ch = torch.sqrt(0.5 * g * (hR + hL))
    hm, s1m, s2m = _middle(hL, hR, uL, uR)
    l0 = torch.minimum(torch.minimum(uL - sgL, uh - ch), s2m)
    l2 = torch.maximum(torch.maximum(uR + sgR, uh + ch), s1m)
    hll = torch.clamp((nL - nR + l2 * hR - l0 * hL) / (l2 - l0), min=0.0)
    db, hbar = bR - bL, 0.5 * (hL + hR)
    bar = 0.25 * (uL + uR) ** 2 - g * hbar
    til = torch.clamp(uL * uR, min=0.0) - g * hbar
    crit = max(DRYTOL * g, 1e-6)
    c2 = math.sqrt(crit)
    sonic = ((bar.abs() <= crit) | (bar * til <= crit ** 2) | (bar * l0 * l2 <= crit ** 2)
             | (torch.minimum(l0.abs(), l2.abs()) < c2) | ((l0 < c2) & (s1m > -c2)) | ((l2 > -c2) & (s2m < c2))
             | ((uL + sgL) * (uR + sgR) < 0) | ((uL - sgL) * (uR - sgR) < 0))
    q1, q2 = hll * (l2 - l0) / l0, hll * (l2 - l0) / l2
    dh = torch.where(sonic, -db, db * g * hbar / bar)
    dh = torch.where((l0 < -crit) & (l2 > crit), torch.maximum(torch.minimum(dh, q2), q1),
                     torch.where(l0 >= crit, torch.maximum(torch.minimum(dh, q1), -hL),
                                 torch.where(l2 <= -crit, torch.maximum(torch.minimum(dh, hR), q2), dh)))
    dp = torch.where(sonic, -g * hbar * db, -db * g * hbar * til / bar)
    dp = torch.minimum(dp, g * torch.maximum(-hL * db, -hR * db))
    dp = torch.maximum(dp, g * torch.minimum(-hL * db, -hR * db))
    d0, d1, d2 = hR - hL - dh, nR - nL, pR - pL - dp
    det = l0 - l2
    b0, b2 = (d1 - d0 * l2) / det, (d0 * l0 - d1) / det
    b1 = d2 - b0 * l0 ** 2 - b2 * l2 ** 2
    t0, t2 = b0 * l0 * vL, b2 * l2 * vR
    rest = hR * uR * vR - hL * uL * vL - t0 - t2
    up = nL + b0 * l0 <= 0
    t0, t2 = torch.where(up, t0 + rest, t0), torch.where(up, t2, t2 + rest)
    w0, w1, w2 = (_where0(any_wet & ~m, one) for m in (lwall, lwall | rwall, rwall))
    z = torch.zeros_like(hL)
    s = [_where0(any_wet, x) * w for x, w in ((l0, w0), (0.5 * (l0 + l2), w1), (l2, w2))]
    f = [[b0 * l0, b0 * l0 ** 2, t0], [z, b1, z], [b2 * l2, b2 * l2 ** 2, t2]]
    return s, [[_where0(w != 0, c) for c in fw] for fw, w in zip(f, (w0, w1, w2))]


def _limited(r, kind):
    zero, one = torch.zeros_like(r), torch.ones_like(r)
    if kind == 4:
        return torch.maximum(zero, torch.minimum(torch.minimum((1 + r) / 2, 2 * one), 2 * r))
    if kind == 3:
        return (r + r.abs()) / (1 + r.abs())
    return torch.maximum(zero, torch.minimum(one, r))


def _split(cell, a):
    """Up- and down-going parts of fluctuation a = (h, n, t) in cells (h, u, v, b, b below, b above)."""
    h, u, v, b, b1, b3 = cell
    c = torch.sqrt(GRAV * h)
    s = (v - c, v, v + c)
    beta = ((s[2] * a[0] - a[2]) / (s[2] - s[0]), -u * a[0] + a[1], (a[2] - s[0] * a[0]) / (s[2] - s[0]))
    one, z = torch.ones_like(u), torch.zeros_like(u)
    r = ((one, u, s[0]), (z, one, z), (one, u, s[2]))
    on = (h > DRYTOL) & (h + b >= torch.minimum(b1, b3))
    down = [sum(_where0(on & (s[m] < 0) & (h + b >= b1), s[m] * beta[m] * r[m][k]) for m in range(3)) for k in range(3)]
    up = [sum(_where0(on & (s[m] > 0) & (h + b >= b3), s[m] * beta[m] * r[m][k]) for m in range(3)) for k in range(3)]
    return down, up


def _sweep(q, b, dtdx, case):
    """Normal sweep along the last axis of padded states q = (h, n, t): flux
    increments of faces 1..mx+1, transverse increments of cells 1..mx (rows
    0..my+1) and the largest CFL number."""
    S = [*(x[..., 1:-1, :] for x in q), b[..., 1:-1, :]]
    s, w = _solve([x[..., :-1] for x in S], [x[..., 1:] for x in S])
    cfl = max(float((dtdx * x).abs().max()) for x in s)
    mid = slice(1, -1)
    am, ap = [], []
    for k in range(3):
        neg = sum(torch.where(s[m] < 0, w[m][k], torch.where(s[m] > 0, 0.0, 0.5 * w[m][k])) for m in range(3))
        pos = sum(torch.where(s[m] > 0, w[m][k], torch.where(s[m] < 0, 0.0, 0.5 * w[m][k])) for m in range(3))
        am.append(neg[..., mid])
        ap.append(pos[..., mid])
    fm, fp = list(am), [-x for x in ap]
    if case["order"] == 2:
        cq = [0.0, 0.0, 0.0]
        for m in range(3):
            own, sm = [x[..., mid] for x in w[m]], s[m][..., mid]
            nrm = sum(x * x for x in own)
            dl = sum(x * y[..., :-2] for x, y in zip(own, w[m]))
            dr = sum(x * y[..., 2:] for x, y in zip(own, w[m]))
            lim = _limited(torch.where(sm > 0, dl, dr) / torch.where(nrm == 0, 1.0, nrm), case["limiter"])
            c = torch.sign(sm) * (1 - sm.abs() * dtdx) * lim
            cq = [a + c * x for a, x in zip(cq, own)]
        fm, fp = [x + 0.5 * c for x, c in zip(fm, cq)], [x + 0.5 * c for x, c in zip(fp, cq)]
        if case["transverse"] == 2:
            am, ap = [x + c for x, c in zip(am, cq)], [x - c for x, c in zip(ap, cq)]
    inner = slice(2, -2)
    g1, g2 = [0.0] * 3, [0.0] * 3
    if case["transverse"]:
        h, n, t = (x[..., 1:-1, inner] for x in q)
        d = torch.where(h > DRYTOL, h, 1.0)
        cell = (torch.where(h > DRYTOL, h, DRYTOL), n / d, t / d, b[..., 1:-1, inner], b[..., :-2, inner], b[..., 2:, inner])
        for a in ([x[..., 1:] for x in am], [x[..., :-1] for x in ap]):
            dn, up = _split(cell, a)
            g1 = [g - 0.5 * dtdx * x for g, x in zip(g1, dn)]
            g2 = [g - 0.5 * dtdx * x for g, x in zip(g2, up)]
    row = slice(1, -1)
    return [x[..., row, :] for x in fm], [x[..., row, :] for x in fp], g1, g2, cfl


def _step64(q, b, dx, dt, manning, case):
    """Interior of the next state of padded fields q = (h, hu, hv), and the CFL number."""
    dry = q[0] < DRYTOL
    h, hu, hv = torch.where(dry, torch.clamp(q[0], min=0.0), q[0]), _where0(~dry, q[1]), _where0(~dry, q[2])
    r = dt / dx
    fm, fp, g1, g2, cx = _sweep((h, hu, hv), b, r, case)
    tr = [x.transpose(-1, -2) for x in (h, hv, hu)]
    gm, gp, f1, f2, cy = _sweep(tr, b.transpose(-1, -2), r, case)
    gm, gp = ([x.transpose(-1, -2) for x in (v[0], v[2], v[1])] for v in (gm, gp))
    if case["transverse"]:
        f1, f2 = ([x.transpose(-1, -2) for x in (v[0], v[2], v[1])] for v in (f1, f2))
        for k in range(3):
            gt = g2[k][..., :-1, :] + g1[k][..., 1:, :]
            ft = f2[k][..., :-1] + f1[k][..., 1:]
            gm[k], gp[k], fm[k], fp[k] = gm[k] + gt, gp[k] + gt, fm[k] + ft, fp[k] + ft
    out = [x[..., 2:-2, 2:-2] - r * (fm[k][..., 1:] - fp[k][..., :-1]) - r * (gm[k][..., 1:, :] - gp[k][..., :-1, :])
           for k, x in enumerate((h, hu, hv))]
    h = out[0]
    gam = torch.sqrt(out[1] ** 2 + out[2] ** 2) * GRAV * manning ** 2 / torch.clamp(h, min=1e-30) ** (7.0 / 3.0)
    div = torch.where(h < 1e-30, math.inf, 1.0 + dt * gam)
    return [h, out[1] / div, out[2] / div], max(cx, cy)


def exact(case, seed):
    dev = _device()
    if case["kind"] == "batch":
        q, aux, dx, dt = _batch_patches(case, seed)
        qt = torch.from_numpy(q).to(dev)
        b = torch.from_numpy(aux).to(dev)[..., 0]
        new, cfl = _step64([qt[..., k] for k in range(3)], b, dx, dt, 0.03, case)
        out = qt.clone()
        out[:, 2:-2, 2:-2] = torch.stack(new, -1)
        return out, cfl
    # chaotic fronts and long runs have no value to compare with
    if case["kind"] != "brick" or case["wet"] < 1.0 or case["mi"] * case["mj"] * case["mx"] ** 2 * case["steps"] > 3e8:
        return None
    h, hu, hv, b, dx = _brick_fields(case, seed)
    b, q = _mirror(b), [h, hu, hv]
    t, dt, cfl, done, retaken = 0.0, 0.02 * dx, 0.0, 0, 0
    for _ in range(case["steps"]):
        p = [_mirror(x) for x in q]
        for k, d in ((1, 1), (2, 0)):  # walls turn the normal momentum round
            n = p[k].shape[d]
            p[k].index_copy_(d, torch.tensor([0, 1, n - 2, n - 1], device=dev),
                             -p[k].index_select(d, torch.tensor([0, 1, n - 2, n - 1], device=dev)))
        new, cfl = _step64(p, b, dx, dt, 0.03, case)
        if cfl <= 1.0:
            t, q, done = t + dt, new, done + 1
        else:
            retaken += 1
        dt = dt * 0.9 / cfl
    m = case["mx"]
    out = torch.stack(q, -1).reshape(case["mj"], m, case["mi"], m, 3).permute(0, 2, 1, 3, 4).reshape(-1, m, m, 3)
    return out, t, dt, cfl, None, None
