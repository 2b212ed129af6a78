"""Performance cases of the Godunov step: what programs built on this framework
have it do, through the public entry points, from the shortest tube to the
largest box.

Three ways of calling appear, as in Mara2's own programs and the ones here:

  solve   upload an initial state, run it, fetch the result (a regression
          problem, a parameter study, one request of a service)
  output  a long simulation's output interval: run so many steps of the
          resident state, fetch the snapshot; the next pass goes on from there
  host    maraMainLoop with the loop on the host: the CFL time step, then one
          step, and so on
  batch   many independent solves admitted together, stepped until all are
          done, retired with their results

`P` of every result is the whole primitive state in MeshData::P layout, guard
zones included.
"""
import math
import os

import numpy as np
import torch

from mara2_amd import abi, problems
from mara2_amd.runtime import Batch, Block

FOREVER = 1e300  # a final time that no run here reaches
HERE = os.path.dirname(os.path.abspath(__file__))
SOURCES = os.path.join(os.path.dirname(HERE), "mara2_amd", "sources")
CONVECTION = (0.2, 0.01)  # gravity and heating of the thermal convection source


def _case(kind, n, steps, mode, precision="fp64", name=None, **more):
    n = tuple(n) + (1,) * (3 - len(n))
    c = dict(kind=kind, n1=n[0], n2=n[1], n3=n[2], steps=steps, mode=mode, precision=precision, **more)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: a regression-size tube stepped by the host's own
        # loop, where every step is a CFL reduction, an advance and two waits
        _case("tube", (256,), 16, "host", riemann="hllc", name="tube_256_host_loop"),
        # the Sod tube to t = 0.2 (about 1120 steps on the device)
        _case("sod", (1024,), 0, "solve", riemann="hlle", name="sod_1024"),
        # a long 1-D MHD Riemann problem of the serving stream's upper range, odd length
        _case("tube_mhd", (10007,), 300, "solve", riemann="hlle", name="tube_mhd_10007"),
        # a 2-D hydro run between outputs, ragged against the tiles
        _case("blast", (636, 477), 150, "output", riemann="hllc", name="blast2d_636x477"),
        # the ThermalConvection program: spherical mesh, source terms, outflow
        _case("convection", (384, 160), 120, "output", riemann="hllc", name="convection_384x160"),
        # 2-D MHD with flux-CT at the size of the benchmark's configuration
        _case("mhd2d", (2048, 2048), 60, "output", riemann="hlle", name="mhd2d_2048"),
        # 3-D MHD with flux-CT, a production box with unequal odd-ish sides
        _case("mhd3d", (116, 97, 108), 30, "output", riemann="hlle", name="mhd3d_116x97x108"),
        # 3-D relativistic MHD, WENO5 + HLLE + CT, RK3, short solve
        _case("rmhd3d", (128, 128, 128), 12, "solve", riemann="hlle", name="rmhd3d_128"),
        # decaying turbulence in the three forms a user picks from: the
        # reference's rounding, the fast binary64 one (the headline size), mixed
        _case("turbulence", (161, 142, 118), 40, "output", riemann="hllc", name="turbulence_161x142x118"),
        _case("turbulence", (256, 256, 256), 100, "output", "fp64_fast", riemann="hllc", name="turbulence_256_fast"),
        _case("turbulence", (192, 192, 192), 100, "output", "mixed", riemann="hllc", name="turbulence_192_mixed"),
        # the serving stream: independent 1-D and 2-D Riemann problems, hydro
        # and MHD, held together in a batch
        _case("stream", (48,), 240, "batch", "mixed", riemann="both", largest=3000, name="stream_48"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tube", "tube", "tube_mhd", "blast", "blast", "convection", "mhd2d", "mhd2d", "mhd3d", "rmhd3d",
                       "turbulence", "turbulence", "turbulence", "stream"])
    form = rng.choice(["fp64", "fp64", "mixed"])
    any_form = rng.choice(["fp64", "fp64_fast", "mixed"])
    solver = rng.choice(["hlle", "hllc"])
    if kind == "tube":
        mode = rng.choice(["host", "solve"])
        return _case(kind, (_log(rng, 100, 16384),), rng.randint(8, 24) if mode == "host" else rng.randint(100, 800),
                     mode, form, riemann=solver)
    if kind == "tube_mhd":
        return _case(kind, (_log(rng, 100, 16384),), rng.randint(100, 500), "solve", form, riemann="hlle")
    if kind == "blast":
        return _case(kind, (_log(rng, 48, 1024), _log(rng, 48, 1024)), rng.randint(60, 150), "output", any_form,
                     riemann=solver)
    if kind == "convection":
        return _case(kind, (_log(rng, 64, 512), _log(rng, 32, 256)), rng.randint(60, 120), "output", form,
                     riemann=solver)
    if kind == "mhd2d":
        return _case(kind, (_log(rng, 64, 2048), _log(rng, 64, 2048)), rng.randint(30, 60), "output", any_form,
                     riemann="hlle")
    if kind == "mhd3d":
        n = [_log(rng, 24, 128) for _ in range(3)]
        return _case(kind, n, rng.randint(15, 30), "output", form, riemann="hlle")
    if kind == "rmhd3d":
        n = [_log(rng, 24, 128) for _ in range(3)]
        return _case(kind, n, rng.randint(4, 12), "solve", form, riemann="hlle")
    if kind == "turbulence":
        n = [_log(rng, 24, 224) for _ in range(3)]
        return _case(kind, n, rng.randint(30, 60), "output", any_form, riemann=solver)
    return _case(kind, (rng.randint(12, 48),), rng.randint(60, 240), "batch", form, riemann="both",
                 largest=rng.randint(1000, 3000))


# ---------------------------------------------------------------------------
# descriptors and initial states
# ---------------------------------------------------------------------------
CFL = {"sod": 0.4, "tube": 0.4, "tube_mhd": 0.4, "blast": 0.4, "convection": 0.4, "mhd2d": 0.4, "mhd3d": 0.3,
       "rmhd3d": 0.2, "turbulence": 0.3, "stream": 0.4}


def _desc(case):
    kind, n = case["kind"], (case["n1"], case["n2"], case["n3"])
    kw = dict(cells=n, riemann=case["riemann"], precision=case["precision"])
    if kind in ("sod", "tube"):
        return abi.make_desc(law="hydro", gamma=1.4, bc="outflow", **kw)
    if kind == "tube_mhd":
        return abi.make_desc(law="mhd", gamma=1.4, bc="outflow", field_ct=0, pressure_floor=1e-6, **kw)
    # square zones: the longest side has length 1
    size = max(n)
    upper = tuple(m / size if m > 1 else 1.0 for m in n)
    if kind == "blast":
        return abi.make_desc(law="hydro", gamma=1.4, bc="reflecting", upper=upper, **kw)
    if kind == "convection":
        wedge = math.pi / 12
        return abi.make_desc(law="hydro", plm_theta=2.0, bc="outflow", geometry="spherical", log_radial=True,
                             lower=(1.0, math.pi / 2 - wedge, 0.0), upper=(10.0, math.pi / 2 + wedge, 2 * math.pi), **kw)
    if kind in ("mhd2d", "mhd3d"):
        return abi.make_desc(law="mhd", bc="periodic", upper=upper, pressure_floor=1e-6, **kw)
    if kind == "rmhd3d":
        return abi.make_desc(law="rmhd", gamma=4.0 / 3.0, recon="weno5", bc="periodic", rk_order=3, upper=upper, **kw)
    return abi.make_desc(law="hydro", bc="periodic", upper=upper, **kw)  # turbulence


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _random_field(n, rng, kmax, slope):
    """A periodic Gaussian random field with modes 1 <= |k| <= kmax, |f_k|^2 ~ k^slope, unit rms."""
    axes = [a for a in range(3) if n[a] > 1]
    shape = tuple(n[a] for a in axes)
    white = torch.randn(shape, generator=rng, dtype=torch.float64, device=rng.device)
    spec = torch.fft.fftn(white)
    ks = [torch.fft.fftfreq(m, 1.0 / m, dtype=torch.float64, device=rng.device) for m in shape]
    k2 = sum(k.reshape([-1 if a == b else 1 for b in range(len(ks))]) ** 2 for a, k in enumerate(ks))
    amp = torch.where((k2 >= 1.0) & (k2 <= kmax * kmax), k2.clamp(min=1.0) ** (slope / 4.0), torch.zeros_like(k2))
    f = torch.fft.ifftn(spec * amp).real
    return (f / f.square().mean().sqrt()).reshape(n)


def _solenoidal(n, rng, kmax, flat_z):
    """Zone-centred B = curl A of a random vector potential on the zone
    vertices: its corner divergence, the one flux-CT conserves, vanishes."""
    A = [_random_field(n, rng, kmax, 0.0) for _ in range(3)]

    def diff(f, a):
        return torch.roll(f, -1, a) - f if n[a] > 1 else torch.zeros_like(f)

    def mean(f, *axes):
        for a in axes:
            f = 0.5 * (torch.roll(f, -1, a) + f) if n[a] > 1 else f
        return f

    if flat_z:
        A[0] = A[1] = torch.zeros_like(A[2])
    B = torch.stack([mean(diff(A[2], 1), 0, 2) - mean(diff(A[1], 2), 0, 1),
                     mean(diff(A[0], 2), 0, 1) - mean(diff(A[2], 0), 1, 2),
                     mean(diff(A[1], 0), 1, 2) - mean(diff(A[0], 1), 0, 2)])
    return B / B.square().sum(0).mean().sqrt()


def _interior(case, seed):
    """Interior primitives (nq, n1, n2, n3) of a case's initial state."""
    kind, n = case["kind"], (case["n1"], case["n2"], case["n3"])
    dev = _device()
    rng = torch.Generator(device=dev)
    rng.manual_seed(int(seed))
    if kind in ("sod", "tube", "tube_mhd"):
        r = np.random.default_rng(int(seed))
        x = (torch.arange(n[0], dtype=torch.float64, device=dev) + 0.5) / n[0]
        left = x < (0.5 if kind == "sod" else r.uniform(0.4, 0.6))
        if kind == "sod":  # the published tube, each side's density and pressure varied by up to 1 %
            sides = np.array([[1.0, 0, 0, 0, 1.0], [0.125, 0, 0, 0, 0.1]])
            sides[:, [0, 4]] *= r.uniform(0.99, 1.01, (2, 2))
        else:
            sides = np.empty((2, 5))
            sides[:, 0] = np.exp(r.uniform(np.log(0.1), np.log(10), 2))
            sides[:, 1:4] = r.uniform(-1, 1, (2, 3))
            sides[:, 4] = np.exp(r.uniform(np.log(0.1), np.log(10), 2))
            if kind == "tube_mhd":
                beta = np.exp(r.uniform(0, np.log(10)))
                B = r.standard_normal(3)
                B *= np.sqrt(sides[:, 4].mean() * 2 / beta) / np.linalg.norm(B)
                jump = r.standard_normal(3) * 0.3 * np.linalg.norm(B)
                jump[0] = 0
                sides = np.concatenate([sides, np.stack([B - jump, B + jump])], 1)
        s = torch.from_numpy(sides).to(dev)
        return torch.where(left[None, :], s[0][:, None], s[1][:, None]).reshape(-1, *n)
    ones = torch.ones(n, dtype=torch.float64, device=dev)
    if kind == "blast":
        size = max(n)
        x = (torch.arange(n[0], dtype=torch.float64, device=dev) + 0.5) / size - n[0] / size * 0.5
        y = (torch.arange(n[1], dtype=torch.float64, device=dev) + 0.5) / size - n[1] / size * 0.5
        inside = (x[:, None, None] ** 2 + y[None, :, None] ** 2) < 0.01
        return torch.stack([ones + 0.1 * _random_field(n, rng, 8, 0.0).clamp(-3, 3), 0 * ones, 0 * ones, 0 * ones,
                            torch.where(inside, 10 * ones, ones)])
    if kind == "convection":
        r = 10.0 ** ((torch.arange(n[0], dtype=torch.float64, device=dev) + 0.5) / n[0])
        d = (r ** -1.5)[:, None, None] * ones
        K = CONVECTION[0] * (5 / 3 - 1) / (5 / 3)
        noise = [0.01 * _random_field(n, rng, 16, -2.0).clamp(-3, 3) for _ in range(2)]
        return torch.stack([d, noise[0] * d, noise[1] * d, 0 * ones, K * d ** (5 / 3)])
    if kind == "rmhd3d":
        u = torch.stack([_random_field(n, rng, 4, 0.0) for _ in range(3)])
        u = u / u.square().sum(0).max().sqrt() * math.sqrt(1.5 ** 2 - 1)  # Lorentz factors up to 1.5
        v = u / (1 + u.square().sum(0)).sqrt()
        return torch.cat([ones[None], v, ones[None], math.sqrt(0.1) * _solenoidal(n, rng, 4, False)])  # sigma 0.1
    if kind in ("mhd2d", "mhd3d"):
        flat = kind == "mhd2d"
        v = torch.stack([_random_field(n, rng, 8, 0.0) if a < 2 or not flat else 0 * ones for a in range(3)])
        v = 0.5 * v / v.square().sum(0).mean().sqrt()
        return torch.cat([ones[None], v, ones[None], math.sqrt(2.0) * _solenoidal(n, rng, 8, flat)])  # beta 1
    v = torch.stack([_random_field(n, rng, 16, -4.0) for _ in range(3)])
    v = v * math.sqrt(5.0 / 3.0) / v.square().sum(0).mean().sqrt()  # rms Mach 1
    return torch.cat([ones[None], v, ones[None]])


def _guarded(desc, Q):
    """Q (nq, n1, n2, n3) with the guard zones of the boundary condition."""
    for a in range(3):
        g, n = desc.guards[a], desc.cells[a]
        if g == 0:
            continue
        at = torch.arange(-g, n + g, device=Q.device)
        if desc.bc == abi.BC_PERIODIC:
            Q = Q.index_select(1 + a, at % n)
        elif desc.bc == abi.BC_OUTFLOW:
            Q = Q.index_select(1 + a, at.clamp(0, n - 1))
        else:
            low, high = at < 0, at >= n
            Q = Q.index_select(1 + a, torch.where(low, -1 - at, torch.where(high, 2 * n - 1 - at, at)))
            sign = torch.where(low | high, -1.0, 1.0).to(Q.dtype)
            Q = Q.clone()
            Q[1 + a] *= sign.reshape([-1 if a == b else 1 for b in range(3)])
    return Q


def _host_layout(desc, Q):
    """MeshData::P of interior primitives, as a host array."""
    return _guarded(desc, Q).permute(1, 2, 3, 0).contiguous().cpu().numpy()


def _stream(case, seed):
    """The solves of a batch: (descriptor, initial state) of `n1` requests of
    the serving stream.  Which meshes and laws they are depends on the case
    alone, their states on the seed."""
    mix, rng = np.random.default_rng(problems.SEED_SERVING + case["n1"]), np.random.default_rng(int(seed))
    out = []
    for _ in range(case["n1"]):
        like = problems.riemann_params(mix)
        prm = problems.riemann_params(rng)
        while (prm["dim"], prm["law"]) != (like["dim"], like["law"]):
            prm = problems.riemann_params(rng)
        prm["n"] = min(like["n"], case["largest"] if prm["dim"] == 1 else case["largest"] // 10)
        d = problems.riemann_desc(prm, precision=case["precision"])
        out.append((d, problems.riemann_problem(prm, d)))
    return out


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
class State:
    pass


def prepare(case, seed):
    s = State()
    s.case, s.cfl, s.steps = case, CFL[case["kind"]], case["steps"]
    if case["mode"] == "batch":
        s.solves = _stream(case, seed)
        room = sum(Batch.item_bytes_of(d, case["precision"]) for d, _ in s.solves)
        s.batch = Batch(room + (64 << 20), precision=case["precision"], max_solves=len(s.solves))
        return s
    s.desc = _desc(case)
    s.P = _host_layout(s.desc, _interior(case, seed))
    s.block = Block(s.desc)
    if case["kind"] == "convection":
        s.block.set_source(os.path.join(SOURCES, "thermal_convection.hsaco"), "mara_source_thermal_convection",
                           CONVECTION)
    if case["mode"] == "output":
        s.block.upload(s.P)
    return s


def run(s):
    mode = s.case["mode"]
    if mode == "batch":
        b = s.batch
        slots = [b.admit(d, P, s.cfl, 0.2, s.steps) for d, P in s.solves]
        while b.step(16):
            pass
        clocks = [b.query(i)[1:3] for i in slots]
        # every solve's result on the host, one after the other
        return {"P": np.concatenate([b.retire(i).reshape(-1) for i in slots]),
                "t": np.array([c[0] for c in clocks]), "steps": np.array([c[1] for c in clocks])}
    b = s.block
    if mode == "host":
        b.upload(s.P)
        t = 0.0
        for _ in range(s.steps):
            dt = s.cfl * b.courant_dt()
            b.advance(dt, t)
            t += dt
        return {"P": b.download(), "t": t}
    if mode == "solve":
        b.upload(s.P)
    final, most = (0.2, 100000) if s.case["kind"] == "sod" else (FOREVER, s.steps)
    t, steps, _ = b.run(s.cfl, final, most)
    return {"P": b.download(), "t": t, "steps": steps}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
ON_CHIP = 256 << 20  # a state larger than the last-level cache is read and written once per step at least


def _flops_per_zone_stage(law, recon, axes):
    """Operations of one zone in one stage: a face per axis (two
    reconstructions per field, two face states, the Riemann solver), then
    the update with the primitive recovery."""
    nq = abi.num_fields(law)
    rebuild = 2 * nq * (8 if recon == abi.RECON_PLM else 60)
    states = 2 * {abi.LAW_HYDRO: 30, abi.LAW_MHD: 75, abi.LAW_RMHD: 250}[law]
    update = {abi.LAW_HYDRO: 60, abi.LAW_MHD: 110, abi.LAW_RMHD: 500}[law]
    return axes * (rebuild + states + 9 * nq) + update


def work(case):
    if case["mode"] == "batch":
        todo = [(d, P.size, case["steps"]) for d, P in _stream(case, 0)]
    else:
        d = _desc(case)
        steps = case["steps"] or int(1.1 * case["n1"])  # the Sod tube's steps to t = 0.2
        todo = [(d, int(np.prod(abi.array_shape(d))), steps)]
    moved = flops = 0
    for d, values, steps in todo:
        zones = d.cells[0] * d.cells[1] * d.cells[2]
        axes = sum(d.cells[a] > 1 for a in range(3))
        moved += values * 8 * (2 if case["mode"] in ("solve", "host", "batch") else 1)
        if values * 8 > ON_CHIP:
            moved += 2 * values * 8 * steps
        flops += zones * steps * d.rk_order * _flops_per_zone_stage(d.law, d.recon, axes)
    return {"bytes": moved, "flops": flops}


# ---------------------------------------------------------------------------
# the same numbers in plain 64-bit torch: the scheme as its papers state it
# (PLM with the generalised minmod limiter or WENO5, HLLE or HLLC, Toth's
# flux-CT, SSP Runge-Kutta), on whole arrays
# ---------------------------------------------------------------------------
def _along(f, axis, start, count):
    return f.narrow(1 + axis, start, count)


def _minmod(theta, l, c, r):
    a, b, d = theta * (c - l), 0.5 * (r - l), theta * (r - c)
    least = torch.minimum(torch.minimum(a.abs(), b.abs()), d.abs())
    return 0.25 * (a.sign() + b.sign()).abs() * (a.sign() + d.sign()) * least


def _weno5(v, mirrored):
    """The value at the right edge (left edge if mirrored) of the middle of five zones."""
    a, b, c, d, e = reversed(v) if mirrored else v
    p = [(2 * c + 5 * d - e) / 6, (-b + 5 * c + 2 * d) / 6, (2 * a - 7 * b + 11 * c) / 6]
    s = [13 / 12 * (c - 2 * d + e) ** 2 + (3 * c - 4 * d + e) ** 2 / 4, 13 / 12 * (b - 2 * c + d) ** 2 + (b - d) ** 2 / 4,
         13 / 12 * (a - 2 * b + c) ** 2 + (a - 4 * b + 3 * c) ** 2 / 4]
    low = torch.minimum(torch.minimum(s[0], s[1]), s[2])
    high = torch.maximum(torch.maximum(s[0], s[1]), s[2])
    more = low / (high + 1e-10) * 50.0 * low
    w = [k / (1e-10 + more + x) ** 2 for k, x in zip((0.3, 0.6, 0.1), s)]
    return (w[0] * p[0] + w[1] * p[1] + w[2] * p[2]) / (w[0] + w[1] + w[2])


def _face_states(d, P, axis):
    """Primitives left and right of faces g .. N - g along `axis` (transverse extent whole)."""
    g, n = d.guards[axis], d.cells[axis]
    if d.recon == abi.RECON_WENO5:
        v = [_along(P, axis, g - 3 + m, n + 1) for m in range(6)]
        return _weno5(v[:5], False), _weno5(v[1:], True)
    l, c, r = (_along(P, axis, g - 2 + m, n + 2) for m in range(3))
    half = 0.5 * _minmod(d.plm_theta, l, c, r)
    return _along(c + half, axis, 0, n + 1), _along(c - half, axis, 1, n + 1)


def _relativistic(d, P):
    v2, B2 = (P[1:4] ** 2).sum(0), (P[5:8] ** 2).sum(0)
    Bv = (P[1:4] * P[5:8]).sum(0)
    W2 = 1 / (1 - v2)
    b0 = W2.sqrt() * Bv
    return W2, b0, (B2 + b0 * b0) / W2, P[0] + d.gamma / (d.gamma - 1) * P[4]  # W^2, b^0, b^2, rho h


def _conserved(d, P):
    v2 = (P[1:4] ** 2).sum(0)
    if d.law == abi.LAW_RMHD:
        W2, b0, bb, h = _relativistic(d, P)
        W, H, p = W2.sqrt(), h + bb, P[4] + 0.5 * bb
        b = P[5:8] / W + b0 * P[1:4]
        D = P[0] * W
        return torch.cat([D[None], H * W2 * P[1:4] - b0 * b, (H * W2 - p - b0 * b0 - D)[None], P[5:8]])
    e = 0.5 * P[0] * v2 + P[4] / (d.gamma - 1)
    if d.law == abi.LAW_MHD:
        e = e + 0.5 * (P[5:8] ** 2).sum(0)
    return torch.cat([P[:1], P[0] * P[1:4], e[None], P[5:]])


def _flux(d, P, U, a):
    vn = P[1 + a]
    F = vn * U
    if d.law == abi.LAW_HYDRO:
        F[1 + a] += P[4]
        F[4] += P[4] * vn
        return F
    Bn = P[5 + a]
    if d.law == abi.LAW_MHD:
        ps = P[4] + 0.5 * (P[5:8] ** 2).sum(0)
        F[1:4] -= Bn * P[5:8]
        F[4] += ps * vn - Bn * (P[1:4] * P[5:8]).sum(0)
    else:
        W2, b0, bb, _ = _relativistic(d, P)
        W, ps = W2.sqrt(), P[4] + 0.5 * bb
        F[1:4] -= Bn * (P[5:8] / W + b0 * P[1:4]) / W
        F[4] += ps * vn - Bn * b0 / W
    F[1 + a] += ps
    F[5:8] -= Bn * P[1:4]
    return F


def _speeds(d, P, a):
    """Slowest and fastest signal along axis a."""
    vn = P[1 + a]
    if d.law == abi.LAW_HYDRO:
        c = (d.gamma * P[4] / P[0]).sqrt()
        return vn - c, vn + c
    if d.law == abi.LAW_MHD:
        cs2, ca2, cn2 = d.gamma * P[4] / P[0], (P[5:8] ** 2).sum(0) / P[0], P[5 + a] ** 2 / P[0]
        c = (0.5 * (cs2 + ca2 + ((cs2 + ca2) ** 2 - 4 * cs2 * cn2).clamp(min=0).sqrt())).sqrt()
        return vn - c, vn + c
    # the magnetosonic quartic's outermost roots, by Newton's method from +-1,
    # beyond which it has no root (convergence from outside is monotone)
    W2, b0, bb, h = _relativistic(d, P)
    W, cs2 = W2.sqrt(), d.gamma * P[4] / h
    bn = P[5 + a] / W + b0 * vn
    K, L = W2 * W2 * h * (1 / cs2 - 1), -W2 * (h + bb / cs2)
    q = [K - L - b0 * b0, -4 * K * vn + 2 * L * vn + 2 * b0 * bn, 6 * K * vn ** 2 + L * (1 - vn ** 2) + b0 * b0 - bn * bn,
         -4 * K * vn ** 3 - 2 * L * vn - 2 * b0 * bn, K * vn ** 4 + L * vn ** 2 + bn * bn]
    ends = []
    for start in (-1.0, 1.0):
        x = torch.full_like(vn, start)
        for _ in range(60):
            f = (((q[0] * x + q[1]) * x + q[2]) * x + q[3]) * x + q[4]
            df = ((4 * q[0] * x + 3 * q[1]) * x + 2 * q[2]) * x + q[3]
            x = x - torch.where(df == 0, torch.zeros_like(f), f / df)
        ends.append(x)
    return ends[0], ends[1]


def _riemann(d, L, R, a):
    UL, UR = _conserved(d, L), _conserved(d, R)
    FL, FR = _flux(d, L, UL, a), _flux(d, R, UR, a)
    (l0, l1), (r0, r1) = _speeds(d, L, a), _speeds(d, R, a)
    ap, am = torch.maximum(l1, r1).clamp(min=0), torch.minimum(l0, r0).clamp(max=0)
    if d.riemann == abi.RIEMANN_HLLE:
        return (ap * FL - am * FR + ap * am * (UR - UL)) / (ap - am)
    vl, vr = L[1 + a], R[1 + a]
    s = ((R[4] - R[0] * vr * (ap - vr)) - (L[4] - L[0] * vl * (am - vl))) / (L[0] * (am - vl) - R[0] * (ap - vr))
    left = s >= 0
    Q, U, F = torch.where(left, L, R), torch.where(left, UL, UR), torch.where(left, FL, FR)
    c, vn = torch.where(left, am, ap), torch.where(left, vl, vr)
    f = Q[0] * (c - vn) / (c - s)
    star = f * torch.cat([torch.ones_like(f)[None], Q[1:4], (U[4] / Q[0] + (s - vn) * (s + Q[4] / (Q[0] * (c - vn))))[None]])
    star[1 + a] += f * (s - vn)
    # a supersonic face (am = 0 or ap = 0) takes the upwind flux
    return torch.where(am >= 0, FL, torch.where(ap <= 0, FR, F + c * (star - U)))


def _divergence(d, P, areas):
    """-div F on the interior, flux-CT applied where the law has it."""
    axes = [a for a in range(3) if d.cells[a] > 1]
    F = {a: _riemann(d, *_face_states(d, P, a), a) for a in axes}

    def inner(f, keep, shift=0):
        for a in axes:
            f = f if a in keep else _along(f, a, d.guards[a] + shift, d.cells[a])
        return f

    G = {a: inner(F[a], (a,)).clone() for a in axes}
    if d.law != abi.LAW_HYDRO and d.field_ct:
        for a in axes:
            for c in axes:
                if c == a:
                    G[a][5 + a] = 0
                    continue
                g, n, gc, nc = d.guards[a], d.cells[a], d.guards[c], d.cells[c]
                A, T = inner(F[a][5 + c][None], (a, c)), inner(F[c][5 + a][None], (a, c))
                own = 2 * _along(A, c, gc, nc) + _along(A, c, gc + 1, nc) + _along(A, c, gc - 1, nc)
                cross = sum(_along(_along(T, c, i, nc), a, g - j, n + 1) for i in (0, 1) for j in (0, 1))
                G[a][5 + c] = 0.125 * (own - cross)[0]
    low, high, volume = areas
    total = 0
    for a in axes:
        n = d.cells[a]
        total = total + _along(G[a], a, 1, n) * high[a] - _along(G[a], a, 0, n) * low[a]
    return -total / volume


def _mesh(d, dev):
    """(low-side areas, high-side areas, volumes), zone lengths and centres."""
    dx = [(d.upper[a] - d.lower[a]) / d.cells[a] for a in range(3)]
    if d.geometry == abi.GEOM_CARTESIAN:
        A = [dx[1] * dx[2], dx[2] * dx[0], dx[0] * dx[1]]
        return (A, A, dx[0] * dx[1] * dx[2]), min(dx), None
    at = [torch.arange(m + 1, dtype=torch.float64, device=dev) for m in d.cells]

    def radius(i):
        return d.lower[0] * (d.upper[0] / d.lower[0]) ** (i / d.cells[0])

    r, q = radius(at[0]), d.lower[1] + dx[1] * at[1]
    r0, r1, q0, q1 = r[:-1, None, None], r[1:, None, None], q[None, :-1, None], q[None, 1:, None]
    dc, dr3, dp = q0.cos() - q1.cos(), (r1 ** 3 - r0 ** 3) / 3, dx[2]
    mid = (r0 * r1).sqrt()
    length = torch.minimum(torch.minimum(r1 - r0, mid * dx[1]), mid * dp * (0.5 * (q0 + q1)).sin())
    centre = (radius(at[0][:-1] + 0.5)[:, None, None], (d.lower[1] + dx[1] * (at[1][:-1] + 0.5))[None, :, None])
    low = [r0 ** 2 * dc * dp, dr3 * q0.sin() * dp, dr3 * dc]
    return (low, [r1 ** 2 * dc * dp, dr3 * q1.sin() * dp, dr3 * dc], dr3 * dc * dp), length, centre


def _convection_source(P, centre):
    (r, q), (g0, heat) = centre, CONVECTION
    rho, vr, vq, vp, p = P
    cot = 1 / q.tan()
    g = g0 / r ** 2
    return torch.stack([0 * rho, (2 * p + rho * (vq ** 2 + vp ** 2)) / r - rho * g,
                        (p * cot + rho * (vp ** 2 * cot - vr * vq)) / r, -rho * vp * (vr + vq * cot) / r,
                        -rho * g * vr + heat * (-r).exp()])


def _primitive(d, U, guess):
    if d.law == abi.LAW_RMHD:
        # Newton's method for Z = rho h W^2 from the zone's last primitives
        W2, _, _, h = _relativistic(d, guess)
        Z, S2, B2, BS = h * W2, (U[1:4] ** 2).sum(0), (U[5:8] ** 2).sum(0), (U[1:4] * U[5:8]).sum(0)
        k = (d.gamma - 1) / d.gamma
        for _ in range(12):
            v2 = (S2 * Z * Z + BS * BS * (B2 + 2 * Z)) / ((B2 + Z) * Z) ** 2
            dv2 = -2 * (S2 + BS * BS * (3 * Z * (Z + B2) + B2 * B2) / Z ** 3) / (Z + B2) ** 3
            w = 1 - v2  # 1 / W^2
            p = k * (Z * w - U[0] * w.sqrt())
            f = Z - p + 0.5 * B2 * (1 + v2) - 0.5 * BS * BS / Z ** 2 - U[0] - U[4]
            df = 1 - k * (w - Z * dv2 + 0.5 * U[0] * dv2 / w.sqrt()) + 0.5 * B2 * dv2 + BS * BS / Z ** 3
            Z = Z - f / df
        v2 = (S2 * Z * Z + BS * BS * (B2 + 2 * Z)) / ((B2 + Z) * Z) ** 2
        w = 1 - v2
        return torch.cat([(U[0] * w.sqrt())[None], (U[1:4] + BS / Z * U[5:8]) / (Z + B2),
                          (k * (Z * w - U[0] * w.sqrt()))[None], U[5:8]])
    e = U[4] - 0.5 * (U[1:4] ** 2).sum(0) / U[0]
    if d.law == abi.LAW_MHD:
        e = e - 0.5 * (U[5:8] ** 2).sum(0)
    p = e * (d.gamma - 1)
    if d.law == abi.LAW_MHD and d.pressure_floor > 0:
        p = torch.where(p < 0, d.pressure_floor * U[0], p)
    return torch.cat([U[:1], U[1:4] / U[0], p[None], U[5:]])


def _time_step(d, Q, length):
    fastest = 0
    for a in range(3):
        low, high = _speeds(d, Q, a)
        here = torch.maximum(low.abs(), high.abs())
        fastest = here if a == 0 else torch.maximum(fastest, here)
    return float((length / fastest).min())


def exact(case, seed):
    if case["mode"] == "batch":
        return None  # tens of solves, each of hundreds of steps of their own: minutes in plain torch
    d = _desc(case)
    zones = case["n1"] * case["n2"] * case["n3"]
    if _device() == "cpu" and zones * max(case["steps"], case["n1"] if case["kind"] == "sod" else 0) > 2e6:
        return None  # over 20 seconds without a GPU
    Q = _interior(case, seed)
    areas, length, centre = _mesh(d, Q.device)
    weights = {2: (1.0, 0.5), 3: (1.0, 0.25, 2.0 / 3.0)}[d.rk_order]
    final = 0.2 if case["kind"] == "sod" else FOREVER
    t, steps = 0.0, 0
    while t < final and (not case["steps"] or steps < case["steps"]):
        dt = min(CFL[case["kind"]] * _time_step(d, Q, length), final - t)
        U0 = U = _conserved(d, Q)
        for b in weights:
            rate = _divergence(d, _guarded(d, Q), areas)
            if case["kind"] == "convection":
                rate = rate + _convection_source(Q, centre)
            U = U0 * (1 - b) + (U + dt * rate) * b
            Q = _primitive(d, U, Q)
        t += dt
        steps += 1
    out = {"P": _host_layout(d, Q), "t": t}
    if case["mode"] != "host":
        out["steps"] = steps
    return out
