"""The work that a user of this library has it do, as cases to be timed and
checked: one cycle of the VL+CT method on device-resident blocks, driven
through the Python binding (enzoe_vlct.VlctMethod, Levels, HostMethod) as a
program that keeps its own device memory would drive it.

listed() holds the cases, draw() gives more of the same ranges, prepare()
makes the blocks and the method handle a program has in hand, run() is one
pass, exact() is the same pass written in plain torch in 64 bits.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), os.pardir,
                                "enzo-e_amd"))
import enzoe_vlct as ev  # noqa: E402

SCALARS = ("density", "velocity_x", "velocity_y", "velocity_z", "total_energy")
CENTRED_B = ("bfield_x", "bfield_y", "bfield_z")
FACE_B = ("bfieldi_x", "bfieldi_y", "bfieldi_z")
PRECISION = {"fp64": ev.ENZOE_PREC_DOUBLE, "mixed": ev.ENZOE_PREC_MIXED,
             "fma": ev.ENZOE_PREC_DOUBLE_FMA}
COURANT, ETA = 0.4, 0.001


def _case(name, nx, ny=None, nz=None, **more):
    c = {"name": name, "kind": "cycle", "problem": "waves", "nbx": 1, "nby": 1, "nbz": 1,
         "nx": nx, "ny": ny or nx, "nz": nz or ny or nx, "ghost": 3, "mhd": True,
         "solver": "hlld", "recon": "plm", "theta": 2.0, "precision": "fp64", "dual": False,
         "bc": "periodic"}
    c.update(more)
    return c


def listed():
    return [
        # the smallest call: a test-sized hydro block, launches and latency count
        _case("hydro_16", 16, mhd=False, solver="hllc"),
        # the linear-wave test's block: one 32^3 MHD block, too small for the chip
        _case("waves_32", 32),
        # sub-cycled AMR levels of 32^3 blocks (1 : 3 : 6 blocks a level), one
        # coarse step with the dt on the device
        _case("amr_32", 32, kind="levels", problem="rough", nbx=32, nby=96, nbz=188),
        # decaying Mach-5 turbulence on a grid of 64^3 blocks, both precisions
        _case("turbulence_64", 64, problem="turbulence", nbx=4, nby=4, nbz=4),
        _case("turbulence_64_mixed", 64, problem="turbulence", nbx=4, nby=4, nbz=4,
              precision="mixed"),
        # the headline: one 256^3 Orszag-Tang block, both precisions
        _case("orszag_tang_256", 256, problem="orszag_tang"),
        _case("orszag_tang_256_mixed", 256, problem="orszag_tang", precision="mixed"),
        # the contracted FP64 build on a middling block
        _case("orszag_tang_128_fma", 128, problem="orszag_tang", precision="fma"),
        # hydro shear layers on 128^3 blocks
        _case("shear_128", 128, problem="shear", nbx=2, nby=2, nbz=2, mhd=False,
              solver="hllc"),
        # the dual-energy formalism on one block of odd, unequal sides
        _case("dual_odd", 93, 57, 75, problem="turbulence", dual=True, bc="outflow"),
        # the other MHD solver and limiter on small ragged blocks
        _case("hlle_ragged", 50, 37, 29, problem="rough", solver="hlle", recon="plm_athena",
              nbx=3, nby=2, nbz=2),
        # the C++ drop-in layer run stage by stage through the plugin objects,
        # driven as Cello drives it (refresh, timestep, compute)
        _case("staged_96", 96, kind="staged", problem="orszag_tang"),
    ]


#: zone-updates that no drawn case goes over (a listed one has 16.8 million)
MOST_ZONES = 6.0e6


def draw(rng):
    kind = rng.choice(["cycle"] * 8 + ["levels", "staged"])
    if kind == "levels":
        n = int(round(16 * 3 ** rng.random()))
        unit = rng.randint(1, max(1, int(MOST_ZONES / 31 / n ** 3)))
        return _drawn(rng, "levels", n, n, n, unit, rng.randint(2, 3) * unit,
                      rng.randint(4, 6) * unit, mhd=True)
    if kind == "staged":
        n = [int(round(12 * 8 ** rng.random())) for _ in range(3)]
        return _drawn(rng, "staged", *n, 1, 1, 1, mhd=rng.random() < 0.7)
    while True:
        # block sides over a factor of ten and more, blocks of a grid likewise
        n = [int(round(12 * 16 ** rng.random())) for _ in range(3)]
        nb = [int(8 ** rng.random()) for _ in range(3)] if rng.random() < 0.7 else [1, 1, 1]
        if n[0] * n[1] * n[2] * nb[0] * nb[1] * nb[2] <= MOST_ZONES:
            return _drawn(rng, "cycle", *n, *nb, mhd=rng.random() < 0.75)


def _drawn(rng, kind, nx, ny, nz, nbx, nby, nbz, mhd):
    staged = kind == "staged"
    dual = kind == "cycle" and rng.random() < 0.15
    precision = "fp64" if dual or staged else rng.choice(["fp64", "fp64", "mixed", "fma"])
    c = _case("", nx, ny, nz, kind=kind, nbx=nbx, nby=nby, nbz=nbz, mhd=mhd,
              ghost=rng.choice([3, 3, 4]), dual=dual, precision=precision,
              solver=rng.choice(["hlld", "hlld", "hlle"]) if mhd else "hllc",
              recon=rng.choice(["plm", "plm", "plm_athena", "nn"]),
              theta=rng.choice([2.0, 1.5]),
              # one block with open edges, or a periodic grid
              bc=rng.choice(["periodic", "outflow"])
              if kind == "cycle" and nbx * nby * nbz == 1 else "periodic",
              problem="rough" if kind == "levels" else
              rng.choice(["waves", "turbulence", "orszag_tang", "rough"] if mhd
                         else ["waves", "turbulence", "shear"]))
    del c["name"]
    return c


# ------------------------------------------------------------ initial states

def _gamma(c):
    return 1.4 if c["problem"] == "shear" else 5.0 / 3.0


def _count(c):
    return c["nbx"] + c["nby"] + c["nbz"] if c["kind"] == "levels" else \
        c["nbx"] * c["nby"] * c["nbz"]


def _level_of(c):
    """Refinement level of each block of a "levels" case."""
    return [0] * c["nbx"] + [1] * c["nby"] + [2] * c["nbz"]


def _widths(c):
    """Cell widths (x, y, z) of each block."""
    if c["kind"] == "levels":
        return [(1.0 / (c["nx"] << lev),) * 3 for lev in _level_of(c)]
    return [(1.0 / (c["nbx"] * c["nx"]), 1.0 / (c["nby"] * c["ny"]),
             1.0 / (c["nbz"] * c["nz"]))] * _count(c)


def _coords(c, dev):
    """Cell-centre and low-face coordinates of every block along x, y, z, in
    domain units (ghost zones wrap), as (blocks, cells + 1) tensors."""
    nb, g = _count(c), c["ghost"]
    centre, face = [], []
    for a, (n, cnt) in enumerate(zip((c["nx"], c["ny"], c["nz"]),
                                     (c["nbx"], c["nby"], c["nbz"]))):
        i = torch.arange(n + 2 * g + 1, device=dev, dtype=torch.float64) - g
        if c["kind"] == "levels":  # every block is a periodic box of its own
            i, total = i[None].expand(nb, -1), n
        else:
            b = torch.arange(nb, device=dev)
            at = (b % c["nbx"], (b // c["nbx"]) % c["nby"], b // (c["nbx"] * c["nby"]))[a]
            i, total = i[None] + n * at[:, None].to(torch.float64), n * cnt
        i = i % total
        centre.append((i + 0.5) / total)
        face.append(i / total)
    return centre, face


class _Modes:
    """Smooth periodic random fields: sums of a few cosines, one set of
    modes for a whole grid or one for each block."""

    def __init__(self, seed, sets, dev, kmax=3, count=6):
        self.rng = np.random.RandomState(seed % (1 << 32))
        self.sets, self.dev, self.kmax, self.count = sets, dev, kmax, count

    def __call__(self, x, y, z):
        f = 0.0
        for _ in range(self.count):
            k = self.rng.randint(-self.kmax, self.kmax + 1, (3, self.sets))
            k[0] += (k == 0).all(axis=0)
            kx, ky, kz, ph, amp = (
                torch.from_numpy(np.asarray(v, dtype=np.float64)).to(self.dev)[:, None]
                for v in (2 * np.pi * k[0], 2 * np.pi * k[1], 2 * np.pi * k[2],
                          self.rng.uniform(0, 2 * np.pi, self.sets),
                          self.rng.normal(size=self.sets) * math.sqrt(2.0 / self.count)))
            f = f + amp[:, :, None, None] * torch.cos(
                (kz * z)[:, :, None, None] + (ky * y)[:, None, :, None]
                + (kx * x + ph)[:, None, None, :])
        return f


def _initial(c, seed, dev):
    """The fields of every block, ghost zones included: {name: (blocks, z, y,
    x) tensor}.  The magnetic field is the curl of a vector potential on the
    cell edges, so its divergence vanishes to roundoff."""
    nb, gamma, mhd = _count(c), _gamma(c), c["mhd"]
    (xc, yc, zc), (xf, yf, zf) = _coords(c, dev)
    X, Y, Z = xc[:, :-1], yc[:, :-1], zc[:, :-1]
    own = c["kind"] == "levels"
    modes = _Modes(seed * 7919 + 17, nb if own else 1, dev)
    one = torch.ones((nb, Z.shape[1], Y.shape[1], X.shape[1]), dtype=torch.float64, device=dev)
    noise = np.random.RandomState((seed * 31 + 5) % (1 << 32)).randint(1 << 30)
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(noise))

    def rough(amp):
        return amp * (2.0 * torch.rand(one.shape, dtype=torch.float64, device=dev,
                                       generator=gen) - 1.0)

    tp, kind = 2.0 * math.pi, c["problem"]
    amp_b, mean_b = 0.0, (0.0, 0.0, 0.0)
    if kind == "orszag_tang":  # with a guide field and seeded v_z noise
        rho, p = one * (25.0 / (36.0 * math.pi)), one * (5.0 / (12.0 * math.pi))
        v = [-torch.sin(tp * Y)[:, None, :, None] * one,
             torch.sin(tp * X)[:, None, None, :] * one, rough(1e-2)]
        mean_b = (0.0, 0.0, 0.1)
    elif kind == "shear":
        inside = ((Y - 0.5).abs() < 0.25)[:, None, :, None]
        rho, p = torch.where(inside, 2.0, 1.0) * one, one * 2.5
        v = [torch.where(inside, 0.5, -0.5) * one, rough(1e-2), rough(1e-2)]
    elif kind == "turbulence":  # Mach 5, plasma beta 0.1
        rho, p = one.clone(), one / gamma
        v = [5.0 / math.sqrt(3.0) * modes(X, Y, Z) * one for _ in range(3)]
        amp_b, mean_b = 0.3, (math.sqrt(20.0 / gamma), 0.0, 0.0)
    elif kind == "rough":  # lognormal density, Mach 2, beta 1
        rho, p = torch.exp(0.5 * modes(X, Y, Z)) * one, one.clone()
        v = [2.0 * math.sqrt(gamma / 3.0) * modes(X, Y, Z) * one for _ in range(3)]
        amp_b, mean_b = 0.6, (1.0, 0.0, 0.0)
    else:  # "waves": small smooth perturbations of a uniform state
        rho, p = one * (1.0 + 1e-2 * modes(X, Y, Z)), one * (1.0 + 1e-2 * modes(X, Y, Z))
        v = [1e-2 * modes(X, Y, Z) * one for _ in range(3)]
        amp_b, mean_b = 1e-2, (1.0, math.sqrt(2.0), 0.5)
    out = dict(zip(SCALARS, [rho] + v))
    energy = p / (gamma - 1.0) + 0.5 * rho * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2])
    if mhd:
        dx, dy, dz = (torch.tensor([w[a] for w in _widths(c)], dtype=torch.float64,
                                   device=dev)[:, None, None, None] for a in range(3))
        s = amp_b / (2.0 * tp)
        Ax, Ay, Az = (s * modes(xc, yf, zf), s * modes(xf, yc, zf), s * modes(xf, yf, zc))
        if own:  # potentials in the block's own units of length
            w = [t * n for t, n in zip((dx, dy, dz), (c["nx"], c["ny"], c["nz"]))]
            Ax, Ay, Az = Ax * w[0], Ay * w[1], Az * w[2]
        if kind == "orszag_tang":
            Az = Az + ((torch.cos(2 * tp * xf) / (2 * tp))[:, None, None, :]
                       + (torch.cos(tp * yf) / tp)[:, None, :, None]) / math.sqrt(4 * math.pi)
        dj, dk, di = (lambda f: f[:, :, 1:] - f[:, :, :-1], lambda f: f[:, 1:] - f[:, :-1],
                      lambda f: f[..., 1:] - f[..., :-1])
        faces = [dj(Az)[:, :-1] / dy - dk(Ay)[:, :, :-1] / dz,
                 dk(Ax)[..., :-1] / dz - di(Az)[:, :-1] / dx,
                 di(Ay)[:, :, :-1] / dx - dj(Ax)[..., :-1] / dy]
        for name, f, m in zip(FACE_B, faces, mean_b):
            out[name] = f + m
        b = [0.5 * (out[n].narrow(d, 1, out[n].shape[d] - 1)
                    + out[n].narrow(d, 0, out[n].shape[d] - 1))
             for n, d in zip(FACE_B, (3, 2, 1))]
        out.update(zip(CENTRED_B, b))
        energy = energy + 0.5 * (b[0] * b[0] + b[1] * b[1] + b[2] * b[2])
    out["total_energy"] = energy / rho
    out["pressure"] = torch.zeros_like(one)
    if c["dual"]:
        out["internal_energy"] = p / ((gamma - 1.0) * rho)
    return out


# --------------------------------------------------------- the program's side

class _Block:
    """One block of a program that keeps its own device memory."""

    def __init__(self, desc):
        self.desc = desc


class _State:
    pass


def prepare(case, seed):
    dev = torch.device("cuda")
    fields = _initial(case, seed, dev)
    mhd, nb, g = case["mhd"], _count(case), case["ghost"]
    s = _State()
    s.case, s.out = case, {}
    # all fields of a block behind one another, each 256-byte aligned
    off, at = 0, {}
    for name, f in fields.items():
        at[name] = off
        off += (f[0].numel() + 31) // 32 * 32
    s.memory = torch.zeros((nb, off), dtype=torch.float64, device=dev)
    for name, f in fields.items():
        view = s.memory[:, at[name]:at[name] + f[0].numel()].unflatten(1, f.shape[1:])
        view.copy_(f)
        s.out[name] = view
    del fields
    s.blocks = []
    for i, w in enumerate(_widths(case)):
        b = ev.Block()
        b.mx, b.my, b.mz = (case[k] + 2 * g for k in ("nx", "ny", "nz"))
        b.ghost = g
        ptr = {name: s.out[name][i].data_ptr() for name in at}
        for a in range(3):
            b.cell_width[a] = w[a]
            b.velocity[a] = ptr[SCALARS[1 + a]]
            if mhd:
                b.bfield[a], b.bfieldi[a] = ptr[CENTRED_B[a]], ptr[FACE_B[a]]
        b.density, b.total_energy, b.pressure = (ptr["density"], ptr["total_energy"],
                                                 ptr["pressure"])
        if case["dual"]:
            b.internal_energy = ptr["internal_energy"]
        s.blocks.append(_Block(b))
    torch.cuda.synchronize()
    s.method = ev.VlctMethod(mhd=mhd, riemann=case["solver"], reconstruct=case["recon"],
                             theta=case["theta"], courant=COURANT, gamma=_gamma(case),
                             precision=PRECISION[case["precision"]],
                             dual_energy_eta=ETA if case["dual"] else None)
    if case["kind"] == "levels":
        lev = _level_of(case)
        s.levels = ev.Levels(s.method, [[b for b, l in zip(s.blocks, lev) if l == k]
                                        for k in range(3)])
    elif case["kind"] == "staged":
        s.host = ev.HostMethod(
            "mhd_choice = %s; riemann_solver = %s; reconstruct_method = %s; "
            "theta_limiter = %r; courant = %r; device_fused = false"
            % ("constrained_transport" if mhd else "no_bfield", case["solver"],
               case["recon"], case["theta"], COURANT), gamma=_gamma(case))
    else:
        s.dt = s.method.timestep(s.blocks)
    return s


def run(s):
    c = s.case
    if c["kind"] == "levels":
        # a coarse step: per-level CFL, then the sub-cycled batched steps
        s.levels.step()
        return s.out
    s.method.refresh(s.blocks, (c["nbx"], c["nby"], c["nbz"]), (c["bc"],) * 3)
    if c["kind"] == "staged":
        dt = s.host.timestep(s.blocks[0])
        s.host.compute(s.blocks, dt)
    else:
        # the step, and with it the next cycle's dt
        dt = s.dt = s.method.compute_timestep(s.blocks, s.dt)
    return {"fields": s.out, "dt": np.float64(dt)}


# ------------------------------------------------------------------ measures

def _zone_updates(c):
    n = c["nx"] * c["ny"] * c["nz"]
    return n * (c["nbx"] + 2 * c["nby"] + 4 * c["nbz"]) if c["kind"] == "levels" else \
        n * _count(c)


def work(case):
    """Every field of the state read once and written once per zone-update
    (and the pressure written); the arithmetic of the two stages' Riemann
    problems, reconstructions and updates, counted from the formulas of
    exact() (an operation each, divisions and roots too)."""
    z = _zone_updates(case)
    words = (11 if case["mhd"] else 5) + (1 if case["dual"] else 0)
    face = {"hlld": 290, "hlle": 230, "hllc": 130}[case["solver"]]
    nq = 7 if case["mhd"] else 5
    slopes = {"nn": 0, "plm": 13 * nq, "plm_athena": 9 * nq}[case["recon"]]
    flops = 2 * 3 * face + 3 * slopes + 2 * (3 * (3 * nq) + 30)
    if case["mhd"]:
        flops += 2 * (3 * 36 + 3 * 7 + 20)
    return {"bytes": 8.0 * (2 * words + 1) * z, "flops": float(flops) * z}


def tolerance(case):
    """About four times what exact() shows over these problems and some fifty
    drawn ones.  The FP64 path differs from it by roundings, now and then
    turned by a limiter or a wave fan (more so over the substeps of the
    levels); the contracted build turns more of them, on the symmetric
    Orszag-Tang flow above all; the mixed path is off by its FP32 fluxes, worst
    in the small velocity component."""
    if case["precision"] == "mixed":
        return {"rel": 8e-5, "max": 5e-2}
    if case["precision"] == "fma":
        return {"rel": 1.2e-6, "max": 1e-4}
    if case["kind"] == "levels":
        return {"rel": 2.5e-10, "max": 1e-6}
    return {"rel": 2e-13, "max": 1e-9}


# --------------------------------------------------- the step in plain torch

def _cut(f, d, lo, hi):
    """f[lo : len - hi] along axis d of (x, y, z)."""
    ax = 3 - d
    return f.narrow(ax, lo, f.shape[ax] - lo - hi)


def _inner(f, lo, hi, skip=-1):
    for d in range(3):
        if d != skip:
            f = _cut(f, d, lo, hi)
    return f


def _fast(d, p, bi, bj, bk, gamma):
    cs2, va2, ca2 = gamma * p / d, (bi * bi + (bj * bj + bk * bk)) / d, bi * bi / d
    s = cs2 + va2
    return torch.sqrt(0.5 * (s + torch.sqrt(s * s - 4 * cs2 * ca2)))


def _eint_flux(l, r, fd, gamma):
    el, er = l["p"] / ((gamma - 1) * l["d"]), r["p"] / ((gamma - 1) * r["d"])
    return torch.where(fd > 0, el, er) * fd


def _conserved(w, bi, gamma):
    """State and physical flux of a face state, as lists over d, m_i, m_j,
    m_k, e, B_j, B_k."""
    b2 = bi * bi + w["bj"] ** 2 + w["bk"] ** 2
    e = w["p"] / (gamma - 1) + 0.5 * w["d"] * (w["vi"] ** 2 + w["vj"] ** 2 + w["vk"] ** 2) \
        + 0.5 * b2
    pt = w["p"] + 0.5 * b2
    m = w["d"] * w["vi"]
    u = [w["d"], m, w["d"] * w["vj"], w["d"] * w["vk"], e, w["bj"], w["bk"]]
    f = [m, m * w["vi"] + pt - bi * bi, m * w["vj"] - bi * w["bj"], m * w["vk"] - bi * w["bk"],
         w["vi"] * (e + pt) - bi * (bi * w["vi"] + w["vj"] * w["bj"] + w["vk"] * w["bk"]),
         w["bj"] * w["vi"] - bi * w["vj"], w["bk"] * w["vi"] - bi * w["vk"]]
    return u, f, pt


def _hlld(l, r, bi, gamma):
    """Miyoshi & Kusano (2005); flux and interface normal velocity."""
    (ul, fl, ptl), (ur, fr, ptr) = _conserved(l, bi, gamma), _conserved(r, bi, gamma)
    cl = _fast(l["d"], l["p"], bi, l["bj"], l["bk"], gamma)
    cr = _fast(r["d"], r["p"], bi, r["bj"], r["bk"], gamma)
    s0 = torch.minimum(l["vi"] - cl, r["vi"] - cr)
    s4 = torch.maximum(l["vi"] + cl, r["vi"] + cr)
    sdl, sdr = s0 - l["vi"], s4 - r["vi"]
    s2 = (sdr * ur[1] - sdl * ul[1] + (ptl - ptr)) / (sdr * ur[0] - sdl * ul[0])
    ptst = 0.5 * ((ptr + ur[0] * sdr * (s2 - r["vi"])) + (ptl + ul[0] * sdl * (s2 - l["vi"])))
    bsq = bi * bi

    def star(u, w, s, sd, pt):
        sm = s - s2
        d = u[0] * sd / sm
        den = u[0] * sd * sm - bsq
        flat = den.abs() < 1e-8 * ptst
        den = torch.where(flat, 1.0, den)
        k = torch.where(flat, 0.0, bi * (sd - sm) / den)
        q = torch.where(flat, 1.0, (u[0] * sd * sd - bsq) / den)
        vj, vk, bj, bk = w["vj"] - w["bj"] * k, w["vk"] - w["bk"] * k, w["bj"] * q, w["bk"] * q
        vb = s2 * bi + vj * bj + vk * bk
        e = (sd * u[4] - pt * w["vi"] + ptst * s2
             + bi * (w["vi"] * bi + w["vj"] * w["bj"] + w["vk"] * w["bk"] - vb)) / sm
        return [d, d * s2, d * vj, d * vk, e, bj, bk], vj, vk, vb

    al, vjl, vkl, vbl = star(ul, l, s0, sdl, ptl)
    ar, vjr, vkr, vbr = star(ur, r, s4, sdr, ptr)
    rl, rr = torch.sqrt(al[0]), torch.sqrt(ar[0])
    s1, s3 = s2 - bi.abs() / rl, s2 + bi.abs() / rr
    sg, isum = torch.where(bi > 0, 1.0, -1.0), 1.0 / (rl + rr)
    vj = isum * (rl * vjl + rr * vjr + sg * (ar[5] - al[5]))
    vk = isum * (rl * vkl + rr * vkr + sg * (ar[6] - al[6]))
    bj = isum * (rl * ar[5] + rr * al[5] + sg * rl * rr * (vjr - vjl))
    bk = isum * (rl * ar[6] + rr * al[6] + sg * rl * rr * (vkr - vkl))
    vb = s2 * bi + vj * bj + vk * bk
    none = 0.5 * bsq < 1e-8 * ptst
    bl = [al[0], al[1], al[0] * vj, al[0] * vk, al[4] - rl * sg * (vbl - vb), bj, bk]
    br = [ar[0], ar[1], ar[0] * vj, ar[0] * vk, ar[4] + rr * sg * (vbr - vb), bj, bk]
    flux = []
    for q in range(7):
        x, y = torch.where(none, al[q], bl[q]), torch.where(none, ar[q], br[q])
        f = torch.where(s3 > 0, fr[q] + s4 * (ar[q] - ur[q]) + s3 * (y - ar[q]),
                        fr[q] + s4 * (ar[q] - ur[q]))
        f = torch.where(s2 >= 0, fl[q] + s0 * (al[q] - ul[q]) + s1 * (x - al[q]), f)
        f = torch.where(s1 >= 0, fl[q] + s0 * (al[q] - ul[q]), f)
        flux.append(torch.where(s0 >= 0, fl[q], torch.where(s4 <= 0, fr[q], f)))
    vbar = torch.where(s2 >= 0, s2 * (sdl / (s0 - s2)), s2 * (sdr / (s4 - s2)))
    vbar = torch.where(s0 > 0, l["vi"], torch.where(s4 < 0, r["vi"], vbar))
    return flux, vbar


def _hlle(l, r, bi, gamma):
    """HLLE with the Roe-averaged bounding speeds (Einfeldt)."""
    (ul, fl, ptl), (ur, fr, ptr) = _conserved(l, bi, gamma), _conserved(r, bi, gamma)
    cl = _fast(l["d"], l["p"], bi, l["bj"], l["bk"], gamma)
    cr = _fast(r["d"], r["p"], bi, r["bj"], r["bk"], gamma)
    rl, rr = torch.sqrt(l["d"]), torch.sqrt(r["d"])
    inv = 1.0 / (rl + rr)
    vi, vj, vk = ((rl * l[k] + rr * r[k]) * inv for k in ("vi", "vj", "vk"))
    h = (rl * ((ul[4] + ptl) / l["d"]) + rr * ((ur[4] + ptr) / r["d"])) * inv
    rho = rl * rr
    bj, bk = ((rl * r[k] + rr * l[k]) * inv for k in ("bj", "bk"))
    b2, g1 = bi * bi + bj * bj + bk * bk, gamma - 1
    x = ((l["bj"] - r["bj"]) ** 2 + (l["bk"] - r["bk"]) ** 2) * 0.5 * (g1 - 1) * inv
    y = (g1 - 1) * (l["d"] + r["d"]) * 0.5 / rho
    a2 = g1 * (h - 0.5 * (vi * vi + vj * vj + vk * vk) - b2 / rho) - x
    ca2 = bi * bi / rho
    s = a2 + (ca2 + (g1 - y) * (bj * bj + bk * bk) / rho)
    c = torch.sqrt(0.5 * (s + torch.sqrt(s * s - 4 * a2 * ca2)))
    zero = torch.zeros_like(c)
    bp = torch.maximum(torch.maximum(vi + c, r["vi"] + cr), zero)
    bm = torch.minimum(torch.minimum(vi - c, l["vi"] - cl), zero)
    inv = 1.0 / (bp - bm)
    flux = [(bp * fl[q] - bm * fr[q] + (ur[q] - ul[q]) * bp * bm) * inv for q in range(7)]
    return flux, (bp * l["vi"] - bm * r["vi"]) * inv


def _hllc(l, r, _, gamma):
    el = l["p"] / (gamma - 1) + 0.5 * l["d"] * (l["vi"] ** 2 + l["vj"] ** 2 + l["vk"] ** 2)
    er = r["p"] / (gamma - 1) + 0.5 * r["d"] * (r["vi"] ** 2 + r["vj"] ** 2 + r["vk"] ** 2)
    rl, rr = torch.sqrt(l["d"]), torch.sqrt(r["d"])
    inv = 1.0 / (rl + rr)
    vi, vj, vk = ((rl * l[k] + rr * r[k]) * inv for k in ("vi", "vj", "vk"))
    h = (rl * ((el + l["p"]) / l["d"]) + rr * ((er + r["p"]) / r["d"])) * inv
    c = torch.sqrt((gamma - 1) * (h - 0.5 * (vi * vi + vj * vj + vk * vk)).clamp(min=0.0))
    sr = torch.maximum(vi + c, r["vi"] + torch.sqrt(gamma * r["p"] / r["d"]))
    sl = torch.minimum(vi - c, l["vi"] - torch.sqrt(gamma * l["p"] / l["d"]))
    bm, bp = sl.clamp(max=0.0), sr.clamp(min=0.0)
    tl = l["p"] - (sl - l["vi"]) * l["d"] * l["vi"]
    tr = r["p"] - (sr - r["vi"]) * r["d"] * r["vi"]
    dl, dr = l["d"] * (sl - l["vi"]), -r["d"] * (sr - r["vi"])
    cw, cp = (tr - tl) / (dl + dr), ((dl * tr + dr * tl) / (dl + dr)).clamp(min=0.0)
    left = cw >= 0
    wl, wr = torch.where(left, cw / (cw - bm), 0.0), torch.where(left, 0.0, -cw / (bp - cw))
    wm = torch.where(left, -bm / (cw - bm), bp / (bp - cw))

    def outer(w, e, s):
        m = w["d"] * (w["vi"] - s)
        return [m, m * w["vi"] + w["p"], m * w["vj"], m * w["vk"],
                e * (w["vi"] - s) + w["p"] * w["vi"]]

    flux = [wl * x + wr * y for x, y in zip(outer(l, el, bm), outer(r, er, bp))]
    flux[1] = flux[1] + wm * cp
    flux[4] = flux[4] + wm * cp * cw
    return flux, wl * (l["vi"] - bm) + wr * (r["vi"] - bp)


def _slope(a, b, c, recon, theta):
    if recon == "plm_athena":
        x, y = b - a, c - b
        t = x * y
        return torch.where(t <= 0, 0.0, 2 * t / torch.where(t <= 0, 1.0, x + y))
    x, y, m = theta * (b - a), theta * (c - b), 0.5 * (c - a)
    return 0.5 * (torch.sign(x) + torch.sign(y)) * torch.minimum(
        torch.minimum(x.abs(), y.abs()), m.abs())


def _face_states(w, d, cs, recon, theta):
    """Left and right states on the faces along d between the cells of
    [cs, m - cs), from the cells' primitives."""
    names = ("d", "vi", "vj", "vk", "p", "bj", "bk")
    j, k = (d + 1) % 3, (d + 2) % 3
    keys = ("d", "v%d" % d, "v%d" % j, "v%d" % k, "p", "b%d" % j, "b%d" % k)
    l, r = {}, {}
    for name, key in zip(names, keys):
        if key not in w:
            continue
        f = _inner(w[key], cs, cs, d)
        if recon == "nn":
            f = _cut(f, d, cs, cs)
            l[name], r[name] = _cut(f, d, 0, 1), _cut(f, d, 1, 0)
        else:
            f = _cut(f, d, cs - 1, cs - 1)
            s = 0.5 * _slope(_cut(f, d, 0, 2), _cut(f, d, 1, 1), _cut(f, d, 2, 0), recon, theta)
            f = _cut(f, d, 1, 1)
            l[name], r[name] = _cut(f + s, d, 0, 1), _cut(f - s, d, 1, 0)
            if name in ("d", "p"):
                l[name], r[name] = l[name].clamp(min=1e-200), r[name].clamp(min=1e-200)
    return l, r


def _edge(ax, E, F, G):
    """Upwinded edge electric field along ax (Gardiner & Stone): E the centre
    field, F the fluxes of B, G the density fluxes, on the stage's box."""
    j, k = (ax + 1) % 3, (ax + 2) % 3

    def pick(f, oj, ok, faces):
        f = _cut(f, ax, 1, 1)
        for d, o in ((j, oj), (k, ok)):
            f = f if d in faces else _cut(f, d, o, 1 - o)
        return f

    e = {(a, b): pick(E[ax], a, b, ()) for a in (0, 1) for b in (0, 1)}
    ej = [-pick(F[j, k], 0, o, (j,)) for o in (0, 1)]  # on j faces, cells k, k + 1
    ek = [pick(F[k, j], o, 0, (k,)) for o in (0, 1)]   # on k faces, cells j, j + 1
    wj = [0.5 + 0.5 * torch.sign(pick(G[j], 0, o, (j,))) for o in (0, 1)]
    wk = [0.5 + 0.5 * torch.sign(pick(G[k], o, 0, (k,))) for o in (0, 1)]
    r_j = wk[1] * (e[1, 0] - ej[0]) + (1 - wk[1]) * (e[1, 1] - ej[1])
    l_j = wk[0] * (ej[0] - e[0, 0]) + (1 - wk[0]) * (ej[1] - e[0, 1])
    r_k = wj[1] * (e[0, 1] - ek[0]) + (1 - wj[1]) * (e[1, 1] - ek[1])
    l_k = wj[0] * (ek[0] - e[0, 0]) + (1 - wj[0]) * (ek[1] - e[1, 0])
    return 0.25 * (ej[0] + ej[1] + ek[0] + ek[1] + (l_j - r_j) + (l_k - r_k))


def _sync(rho, v, b, gamma, etot, eint):
    """Energy floor and, with a tracked internal energy, the choice between
    it and the total energy's."""
    v2 = v[0] ** 2 + v[1] ** 2 + v[2] ** 2
    b2 = b[0] ** 2 + b[1] ** 2 + b[2] ** 2 if b else torch.zeros_like(rho)
    rest, floor = 0.5 * v2 + 0.5 * b2 / rho, 1e-200 / ((gamma - 1) * rho)
    if eint is None:
        return torch.maximum(etot, floor + rest), None
    e1 = etot - rest
    good = (float(np.float32(gamma * (gamma - 1))) * e1).clamp(min=0.0) \
        > torch.maximum(ETA * v2, ETA * b2 / rho)
    eint = torch.maximum(torch.where(good & (e1 > 0.5 * eint), e1, eint), floor)
    return eint + rest, eint


def _stage(c, src, base, dt, widths, recon, cs, final):
    """One stage: the state `base` advanced by dt with the fluxes of `src`."""
    gamma, mhd = _gamma(c), c["mhd"]
    v = [src[n] for n in SCALARS[1:4]]
    b = [src[n] for n in CENTRED_B] if mhd else []
    w = {"d": src["density"], "v0": v[0], "v1": v[1], "v2": v[2]}
    if c["dual"]:
        w["p"] = (gamma - 1) * src["density"] * src["internal_energy"]
    else:
        w["p"] = (gamma - 1) * (src["density"] * (src["total_energy"] - 0.5 * (
            v[0] ** 2 + v[1] ** 2 + v[2] ** 2))
            - (0.5 * (b[0] ** 2 + b[1] ** 2 + b[2] ** 2) if mhd else 0.0))
    w.update(("b%d" % d, x) for d, x in enumerate(b))
    solve = {"hlld": _hlld, "hlle": _hlle, "hllc": _hllc}[c["solver"]]
    dU, dE, F, G = [0.0] * 5, 0.0, {}, []
    pc = _inner(w["p"], cs + 1, cs + 1).clamp(min=1e-200)
    for d in range(3):
        l, r = _face_states(w, d, cs, recon, c["theta"])
        bi = _cut(_inner(src[FACE_B[d]], cs, cs, d), d, cs + 1, cs + 1) if mhd else None
        f, vbar = solve(l, r, bi, gamma)
        for q, slot in enumerate((0, 1 + d, 1 + (d + 1) % 3, 1 + (d + 2) % 3, 4)):
            x = _inner(f[q], 1, 1, d)
            dU[slot] = dU[slot] - dt / widths[d] * (_cut(x, d, 1, 0) - _cut(x, d, 0, 1))
        if c["dual"]:
            x, y = _inner(_eint_flux(l, r, f[0], gamma), 1, 1, d), _inner(vbar, 1, 1, d)
            dE = dE - dt / widths[d] * (_cut(x, d, 1, 0) - _cut(x, d, 0, 1)) \
                - dt / widths[d] * pc * (_cut(y, d, 1, 0) - _cut(y, d, 0, 1))
        G.append(f[0])
        if mhd:
            F[d, (d + 1) % 3], F[d, (d + 2) % 3] = f[5], f[6]
        del l, r, f
    out = {n: base[n].clone() for n in base}
    bc = []
    if mhd:
        E = [_inner(-v[(d + 1) % 3] * b[(d + 2) % 3] + v[(d + 2) % 3] * b[(d + 1) % 3], cs, cs)
             for d in range(3)]
        edge = [_edge(d, E, F, G) for d in range(3)]
        for d in range(3):
            j, k = (d + 1) % 3, (d + 2) % 3
            ek, ej = edge[k], edge[j]  # cut to the faces inside along d by construction
            upd = - dt / widths[j] * (_cut(ek, j, 1, 0) - _cut(ek, j, 0, 1)) \
                + dt / widths[k] * (_cut(ej, k, 1, 0) - _cut(ej, k, 0, 1))
            x = _cut(_inner(out[FACE_B[d]], cs + 1, cs + 1, d), d, cs + 1, cs + 1)
            x += upd
        lo = cs if final else cs + 1
        for d, n in enumerate(CENTRED_B):
            f = _inner(out[FACE_B[d]], lo, lo)
            x = 0.5 * (_cut(f, d, 0, 1) + _cut(f, d, 1, 0))
            _inner(out[n], lo, lo).copy_(x)
            bc.append(_inner(out[n], cs + 1, cs + 1))
    old = {n: _inner(base[n], cs + 1, cs + 1) for n in SCALARS}
    rho = (old["density"] + dU[0]).clamp(min=1e-200)
    vel = [(old[n] * old["density"] + x) / rho for n, x in zip(SCALARS[1:4], dU[1:4])]
    etot = (old["total_energy"] * old["density"] + dU[4]) / rho
    eint = None
    if c["dual"]:
        eint = (_inner(base["internal_energy"], cs + 1, cs + 1) * old["density"] + dE) / rho
    etot, eint = _sync(rho, vel, bc, gamma, etot, eint)
    for n, x in zip(SCALARS, [rho] + vel + [etot]):
        _inner(out[n], cs + 1, cs + 1).copy_(x)
    if eint is not None:
        _inner(out["internal_energy"], cs + 1, cs + 1).copy_(eint)
    return out


def _step(c, u, dt, widths):
    half = _stage(c, u, u, 0.5 * dt, widths, "nn", 0, False)
    return _stage(c, half, u, dt, widths, c["recon"], 1 if c["recon"] == "nn" else 2, True)


def _timestep(c, u, widths):
    """The CFL term's minimum of each block (ghost zones included) times the
    Courant number; writes the pressure, and with dual energy synchronises."""
    gamma = _gamma(c)
    v = [u[n] for n in SCALARS[1:4]]
    b = [u[n] for n in CENTRED_B] if c["mhd"] else []
    b2 = b[0] ** 2 + b[1] ** 2 + b[2] ** 2 if b else 0.0
    if c["dual"]:
        e, i = _sync(u["density"], v, b, gamma, u["total_energy"], u["internal_energy"])
        u["total_energy"], u["internal_energy"] = e, i
        p = (gamma - 1) * u["density"] * i
    else:
        p = (gamma - 1) * (u["density"] * (u["total_energy"] - 0.5 * (
            v[0] ** 2 + v[1] ** 2 + v[2] ** 2)) - 0.5 * b2)
    u["pressure"] = p
    cf = torch.sqrt((gamma * p + b2) / u["density"])
    return COURANT * torch.stack([(w / (x.abs() + cf)).amin(dim=(1, 2, 3))
                                  for w, x in zip([t.expand(len(p), 1, 1, 1) for t in widths],
                                                  v)]).amin(dim=0)


def _refresh(c, u):
    """Ghost zones from the neighbouring blocks (periodic) or the nearest
    active cell or face (outflow, one block)."""
    g, nb = c["ghost"], _count(c)
    cnt, n = (c["nbx"], c["nby"], c["nbz"]), (c["nx"], c["ny"], c["nz"])
    blk = np.arange(nb)
    at = (blk % cnt[0], (blk // cnt[0]) % cnt[1], blk // (cnt[0] * cnt[1]))
    dev = u["density"].device
    for name in u:
        if name == "pressure":
            continue
        face = FACE_B.index(name) if name in FACE_B else -1
        sb, si = [], []
        for a in range(3):
            m = n[a] + 2 * g + (face == a)
            i = np.arange(m)[None] - g + n[a] * at[a][:, None]
            N, top = n[a] * cnt[a], n[a] * cnt[a] - (face != a)
            if c["bc"] == "periodic":
                i = i % N
            else:
                i = np.clip(i, 0, top)
            own = np.arange(m)[None] - g
            inside = (own >= 0) & (own < n[a] + (face == a))
            s = np.minimum(i // n[a], cnt[a] - 1)
            i = np.where(inside, own, i - s * n[a]) + g
            sb.append(torch.from_numpy(np.where(inside, at[a][:, None], s)).to(dev))
            si.append(torch.from_numpy(i).to(dev))
        f = u[name]
        src = ((sb[2][:, :, None, None] * cnt[1] + sb[1][:, None, :, None]) * cnt[0]
               + sb[0][:, None, None, :])
        u[name] = f[src, si[2][:, :, None, None], si[1][:, None, :, None],
                    si[0][:, None, None, :]]


def exact(case, seed):
    dev = torch.device("cuda")
    u = _initial(case, seed, dev)
    widths = [torch.tensor([w[a] for w in _widths(case)], dtype=torch.float64,
                           device=dev)[:, None, None, None] for a in range(3)]
    if case["kind"] == "levels":
        lev = torch.tensor(_level_of(case), device=dev)
        each = _timestep(case, u, widths)
        dt0 = min(float(each[lev == k].min()) * 2 ** k for k in range(3))
        for sub in range(4):
            on = [k for k in range(3) if sub % (1 << (2 - k)) == 0]
            at = torch.isin(lev, torch.tensor(on, device=dev))
            dt = (dt0 / (2.0 ** lev[at].to(torch.float64)))[:, None, None, None]
            part = _step(case, {n: f[at] for n, f in u.items()}, dt, [w[at] for w in widths])
            for n, f in part.items():
                u[n][at] = f
        return u
    if case["kind"] == "staged":
        _refresh(case, u)
        dt = float(_timestep(case, u, widths).min())
        return {"fields": _step(case, u, dt, widths), "dt": np.float64(dt)}
    dt = float(_timestep(case, u, widths).min())
    _refresh(case, u)
    u = _step(case, u, dt, widths)
    return {"fields": u, "dt": np.float64(float(_timestep(case, u, widths).min()))}
