"""What a user of this framework has it do, as cases that can be timed.

A case is a dict of plain values.  `kind` says which program it stands for:

  run       a simulation: Zel'dovich initial conditions on the GPU, then the
            step loop (timestep, update_x, buffer_grid, buffer_x,
            ext_pp_force when PP is on, particle_mesh, buffer_v), then the
            state that a checkpoint writes; `z_end` = 0 runs to the end of
            the clock, else `steps` steps.  `cells` returns the cell arrays
            alone, as a large run's in-loop check reads them
  resume    the same loop restarted from a checkpoint of a clustered state,
            and the checkpoint written again: where a long run spends nearly
            all of its steps
  forward   one pass of the differentiable particle-mesh model
  grad      forward, mean squared error against a target, and the gradient
            with respect to the initial white noise
  ensemble  forward, loss and gradient of several boxes of uneven sizes in
            one graph replay
  power     P(k) of a particle state, the in-loop analysis

The sizes are those of the configurations, tests and benchmark of this
repository (meshes that its FFTs are built for), from the smallest box, where
calls and launches count, to the 512^3-particle step of the benchmark.
"""
import math

import numpy as np
import torch

from cafproject_amd import dpm, ics
from cafproject_amd.cube import Cube
from cafproject_amd.timestep import Clock

OMEGA_M = 0.31
COSMO = ics.Cosmology()


def _run(name, nc, nnt, np_nc, izipx, izipv, pid, pp, layout, spacing, z_i, z_end, steps, cells):
    c = dict(kind="run", nc=nc, nnt=nnt, np_nc=np_nc, izipx=izipx, izipv=izipv, pid=pid, pp=pp, layout=layout,
             spacing=spacing, z_i=z_i, z_end=z_end, steps=steps, cells=cells)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest box: a test or a parameter scan; calls and launches
        _run("run_32_pp", 16, 2, 2, 2, 2, True, True, 0, 0.78, 49.0, 0.0, 12, False),
        # the 128^3 particle-mesh run, z = 49 to 0 with the reference's time
        # steps, one tile, 1-byte positions
        _run("run_128_pm_to_z0", 64, 1, 2, 1, 2, True, False, 0, 1.5625, 49.0, 0.0, 0, False),
        # a mesh that is no power of two (96^3 particles, 192^3 fine mesh, 3^3 tiles)
        _run("run_96_pp", 48, 3, 2, 2, 2, False, True, 0, 0.78, 9.0, 0.0, 10, False),
        # the large box's layout (compact fine mesh, 4^3 tiles, 2-byte positions) at 256^3
        _run("run_256_compact_pp", 128, 4, 2, 2, 2, False, True, 2, 0.78, 3.0, 0.0, 8, True),
        # the benchmark's 512^3 PM+PP step
        _run("run_512_pp", 256, 2, 2, 1, 2, False, True, 0, 0.78125, 49.0, 0.0, 6, True),
        # late in a run: halos, crowded cells, many pairs
        dict(kind="resume", name="resume_128_pp", nc=64, nnt=2, izipx=1, izipv=2, pid=True, spacing=0.78, z=0.5,
             steps=8),
        # density of one box, on a mesh that is no power of two
        dict(kind="forward", name="forward_96", ng=96, ratio=2, steps=10, keep=True, box=100.0),
        # gradients: the smallest and the full-size box, and recompute instead of checkpoints
        dict(kind="grad", name="grad_32", ng=32, ratio=2, steps=10, keep=True, box=80.0),
        dict(kind="grad", name="grad_64_recompute", ng=64, ratio=2, steps=4, keep=False, box=100.0),
        dict(kind="grad", name="grad_128", ng=128, ratio=2, steps=10, keep=True, box=128.0),
        # a quarter of the 48-box ensemble (16/16/8/8 of 32/64/96/128)
        dict(kind="ensemble", name="ensemble_12", n32=4, n64=4, n96=2, n128=2, steps=10),
        # P(k) on the fine mesh, with no allocation in the call
        dict(kind="power", name="power_256", nc=64, nnt=2, izipx=2, mesh=256, noalloc=True),
    ]


def draw(rng):
    kind = rng.choice(["run", "run", "resume", "forward", "grad", "grad", "ensemble", "power"])
    if kind == "run":
        # nc whose coarse (nc), fine (4 nc) and particle (np_nc nc) meshes have FFTs
        nc, np_nc = rng.choice([(16, 2), (18, 1), (20, 1), (24, 2), (32, 2), (48, 2), (64, 1), (64, 2),
                                (128, 1), (128, 2), (144, 1)])
        nnt = rng.choice([t for t in (1, 2, 3, 4, 6) if nc % t == 0 and nc // t >= 8])
        return _run(None, nc, nnt, np_nc, rng.choice([1, 2]), rng.choice([1, 2, 2]), rng.random() < 0.5,
                    rng.random() < 0.7, rng.choice([0, 0, 1, 2]), round(math.exp(rng.uniform(math.log(0.5), math.log(1.6))), 3),
                    rng.choice([49.0, 20.0, 9.0, 5.0]), 0.0, rng.randint(3, 9), rng.random() < 0.3)
    if kind == "resume":
        nc = rng.choice([24, 32, 48, 64])
        nnt = rng.choice([t for t in (1, 2, 3, 4) if nc % t == 0 and nc // t >= 12])
        return dict(kind="resume", nc=nc, nnt=nnt, izipx=rng.choice([1, 2]), izipv=2, pid=rng.random() < 0.5,
                    spacing=round(rng.uniform(0.6, 1.2), 3), z=round(rng.uniform(0.3, 3.0), 2), steps=rng.randint(3, 10))
    if kind in ("forward", "grad"):
        ng, ratio = rng.choice([(16, 2), (24, 2), (32, 1), (32, 2), (32, 4), (48, 2), (48, 4), (64, 1), (64, 2),
                                (72, 2), (96, 2), (96, 1), (128, 1), (128, 2)])
        keep = kind == "forward" or ng * ratio > 128 or rng.random() < 0.7
        return dict(kind=kind, ng=ng, ratio=ratio, steps=rng.randint(1, 10 if keep else 4), keep=keep,
                    box=round(rng.uniform(50.0, 200.0), 1))
    if kind == "ensemble":
        return dict(kind="ensemble", n32=rng.randint(1, 8), n64=rng.randint(0, 6), n96=rng.randint(0, 2),
                    n128=rng.randint(0, 1), steps=rng.randint(3, 10))
    nc = rng.choice([16, 24, 32, 48, 64])
    return dict(kind="power", nc=nc, nnt=rng.choice([1, 2]), izipx=rng.choice([1, 2]),
                mesh=rng.choice([4 * nc, 2 * nc, nc]), noalloc=rng.random() < 0.5)


# ------------------------------------------------------------ the step loop
class Loop:
    """The step loop of a simulation from the state that the Cube holds."""

    def __init__(self, g, a, z_end, sigma, vz_max, dt_vmax, mass):
        self.g, self.mass, self.sigma, self.vz_max = g, mass, sigma, vz_max
        self.clock = Clock(a, [z_end], OMEGA_M, 1 - OMEGA_M)
        self.dtc = dict(dt_fine=1000.0, dt_coarse=1000.0, dt_pp=1000.0, dt_vmax=dt_vmax)

    def step(self):
        g, c = self.g, self.clock
        c.timestep(**self.dtc)
        a_mid, dt = float(c.a_mid), float(c.dt)
        vs = g.update_x(float(c.dt_old), dt, self.vz_max, self.sigma)
        g.buffer_grid()
        g.buffer_x()
        if g.pp_on:
            f2 = g.ext_pp_force(a_mid, dt, self.sigma, self.mass)
            gg = np.float32(1.0) / np.float32(6.0) / np.float32(np.pi)
            f2 = max(np.float32(f2), np.float32(1e-20))
            self.dtc["dt_pp"] = float(np.float32(1.0) / (np.sqrt(f2) * np.float32(a_mid) * gg))
        pm = g.particle_mesh(a_mid, dt, self.sigma, vs["sigma_vi_new"], self.mass)
        g.buffer_v()
        self.sigma, self.vz_max = vs["sigma_vi_new"], pm["vz_max"]
        self.dtc.update(dt_fine=pm["dt_fine"], dt_coarse=pm["dt_coarse"], dt_vmax=pm["dt_vmax"])
        return vs, pm


def _limits(vfield, sigma):
    """vz_max and the first dt constraint, from the cell velocities and the residuals' spread."""
    vz = float(np.abs(vfield[:, 2]).max()) + 7.5 * sigma
    vm = float(np.abs(vfield).max()) + 7.5 * sigma
    return vz, float(np.float32(18.0) / np.float32(vm))


def _cube(c, **more):
    g = Cube(c["nc"], c["nnt"], izipx=c["izipx"], izipv=c["izipv"], has_pid=c.get("pid", False), **more)
    g.init_kernels()
    return g


# ------------------------------------------------------------ prepare, run
def prepare(case, seed):
    c = dict(case)
    kind = c["kind"]
    if kind == "run":
        g = _cube(c, np_nc=c["np_nc"], pp_on=c["pp"], mem_layout=c["layout"])
        n = (c["nc"] * c["np_nc"]) ** 3
        box = c["spacing"] * c["nc"] * c["np_nc"]
        a, sigma = g.make_ics(box, c["z_i"], seed, cosmo=COSMO)
        vz, dt_vmax = _limits(g.get_state(particles=False)["vfield"], sigma)
        return dict(c=c, g=g, box=box, seed=seed, vz=vz, dt_vmax=dt_vmax, mass=float(np.float32((4 * c["nc"]) ** 3 / n)))
    if kind == "resume":
        # the checkpoint: a particle-mesh run from z = 49 to z, written to the host
        n = (2 * c["nc"]) ** 3
        mass = float(np.float32((4 * c["nc"]) ** 3 / n))
        g = _cube(c)
        a, sigma = g.make_ics(2 * c["nc"] * c["spacing"], 49.0, seed, cosmo=COSMO)
        vz, dt_vmax = _limits(g.get_state(particles=False)["vfield"], sigma)
        loop = Loop(g, a, c["z"], sigma, vz, dt_vmax, mass)
        while not loop.clock.final_step:
            loop.step()
        ck = g.get_state()
        g.close()
        dtc = dict(loop.dtc, dt_pp=0.005)
        return dict(c=c, g=_cube(c, pp_on=True, image_buffer=3.0, tile_buffer=6.0), ck=ck, a=float(loop.clock.a), sigma=loop.sigma,
                    vz=loop.vz_max, dtc=dtc, mass=mass)
    if kind in ("forward", "grad"):
        ng, nf = c["ng"], c["ng"] * c["ratio"]
        box = dpm.DPM(ng, nf, c["steps"], checkpoint=c["keep"])
        box.set_amplitude(dpm.amplitude(ng, c["box"], COSMO))
        box.set_schedule(*dpm.schedule(0.1, 1.0, c["steps"]))
        noise, target = _noise(c, seed)
        s = dict(c=c, box=box, noise=noise, target=target, delta=torch.empty(nf ** 3, device="cuda"),
                 dbar=torch.empty(nf ** 3, device="cuda"), noise_bar=torch.empty(ng ** 3, device="cuda"))
        torch.cuda.synchronize()
        return s
    if kind == "ensemble":
        classes = tuple((n, c["n%d" % n]) for n in (32, 64, 96, 128) if c["n%d" % n])
        b, t = dpm.make_ensemble(classes, nsteps=c["steps"], seed0=1000 * (seed % 1000000))
        return dict(c=c, batch=b, t=t)
    x, v = _particles(c, seed)
    g = Cube(c["nc"], c["nnt"], izipx=c["izipx"], has_pid=False)
    g.set_state_xv(x, v)
    return dict(c=c, g=g)


def run(s):
    c = s["c"]
    kind = c["kind"]
    if kind == "run":
        g = s["g"]
        a, sigma = g.make_ics(s["box"], c["z_i"], s["seed"], cosmo=COSMO)
        loop = Loop(g, a, c["z_end"], sigma, s["vz"], s["dt_vmax"], s["mass"])
        done = 0
        while not loop.clock.final_step and (c["steps"] == 0 or done < c["steps"]):
            vs, pm = loop.step()
            done += 1
        return dict(state=g.get_state(particles=not c["cells"]), vs=vs, pm=pm, done=done)
    if kind == "resume":
        g, ck = s["g"], s["ck"]
        g.set_state(ck["xp"], ck["vp"], ck["pid"], ck["rhoc"], ck["vfield"])
        loop = Loop(g, s["a"], 0.0, s["sigma"], s["vz"], 1000.0, s["mass"])
        loop.dtc = dict(s["dtc"])
        for _ in range(c["steps"]):
            vs, pm = loop.step()
        return dict(state=g.get_state(), vs=vs, pm=pm)
    if kind in ("forward", "grad"):
        box, delta = s["box"], s["delta"]
        box.forward(s["noise"].data_ptr(), delta.data_ptr())
        if kind == "forward":
            return dict(delta=delta)
        # the loss is the caller's own: torch reads delta once the box's
        # stream is done, and the box reads dbar once torch's is
        box.sync()
        torch.sub(delta, s["target"], out=s["dbar"]).mul_(2.0 / delta.numel())
        torch.cuda.current_stream().synchronize()
        box.adjoint(s["dbar"].data_ptr(), s["noise_bar"].data_ptr())
        return dict(delta=delta, noise_bar=s["noise_bar"])
    if kind == "ensemble":
        s["batch"].run(graph=True)
        return [dict(delta=t["delta"], noise_bar=t["noise_bar"], loss=t["loss"]) for t in s["t"]]
    k, p, n = s["g"].power(c["mesh"], 100.0, noalloc=c["noalloc"])
    return dict(k=k, power=p, modes=n)


# ------------------------------------------------------------ inputs
def _noise(c, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    noise = torch.randn(c["ng"] ** 3, device="cuda", generator=gen)
    target = 0.5 * torch.randn((c["ng"] * c["ratio"]) ** 3, device="cuda", generator=gen)
    return noise, target


def _particles(c, seed):
    """Half of the particles spread evenly, half in halos of several sizes."""
    rng = np.random.default_rng(seed)
    nc = c["nc"]
    n = (2 * nc) ** 3
    x = rng.random((n, 3)) * nc
    halo = rng.integers(0, max(8, nc ** 2), n // 2)
    x[: n // 2] = (rng.random((max(8, nc ** 2), 3)) * nc)[halo] + rng.standard_normal((n // 2, 3)) * (0.2 + (halo % 7)[:, None] * 0.3)
    return np.mod(x, nc), (0.1 * rng.standard_normal((n, 3))).astype(np.float32)


# ------------------------------------------------------------ work
def _step_work(n, nf3, nc3, bx, bv, pp):
    """One step: every stage reads its inputs once and writes its outputs once
    (drift, PP, two deposits, two kicks over the particles; density, spectra
    and forces over the meshes)."""
    beta = 7 * bx + 8 * bv if pp else 6 * bx + 6 * bv
    fft = 4 * 2.5 * (nf3 * math.log2(nf3) + nc3 * math.log2(nc3))
    return n * beta + nf3 * 54 + nc3 * 86, fft + n * (400 + (33 * 27 if pp else 0))


def _dpm_work(c_ng, nf, steps, grad, keep):
    n, m = c_ng ** 3, nf ** 3
    fft = 2.5 * m * math.log2(m)
    force = (12 * n + 4 * m) + 8 * m + 30 * m          # deposit, forward, three inverse
    one = force + (36 * n + 12 * m) + 36 * n           # and the gather with the kick, and the drift
    b, f = steps * one + 16 * n + 8 * m, (steps + 1) * (4 * fft + 200 * n)
    if grad:
        # per step the transpose: scatter, three forward, one inverse, weight
        # gradients; without checkpoints the forward again up to each step
        b += steps * ((24 * n + 12 * m) + 24 * m + 16 * m + (48 * n + 16 * m)) + 12 * m + 8 * n
        f += steps * (4 * fft + 600 * n)
        if not keep:
            b, f = b + steps * (steps + 1) / 2 * one, f + steps * (steps + 1) / 2 * 4 * fft
    return b, f


def work(case):
    c, kind = case, case["kind"]
    if kind in ("run", "resume"):
        np_nc, pp = c.get("np_nc", 2), c.get("pp", True)
        b, f = _step_work((c["nc"] * np_nc) ** 3, (4 * c["nc"]) ** 3, c["nc"] ** 3, 3 * c["izipx"], 3 * c["izipv"], pp)
        steps = c["steps"] or 30
        return dict(bytes=b * steps, flops=f * steps)
    if kind in ("forward", "grad"):
        b, f = _dpm_work(c["ng"], c["ng"] * c["ratio"], c["steps"], kind == "grad", c["keep"])
        return dict(bytes=b, flops=f)
    if kind == "ensemble":
        w = [(c["n%d" % n], _dpm_work(n, 2 * n, c["steps"], True, True)) for n in (32, 64, 96, 128)]
        return dict(bytes=sum(k * x[0] for k, x in w), flops=sum(k * x[1] for k, x in w))
    n, m = (2 * c["nc"]) ** 3, c["mesh"] ** 3
    return dict(bytes=n * 3 * c["izipx"] + 16 * m, flops=2.5 * m * math.log2(m) + 40 * n)


# ------------------------------------------------------------ 64-bit values
def _kfac(n, d):
    m = torch.fft.fftfreq(n, dtype=torch.float64, device="cuda") * n
    mx = torch.arange(n // 2 + 1, dtype=torch.float64, device="cuda")
    ax = [mx.view(1, 1, -1), m.view(1, -1, 1), m.view(-1, 1, 1)]
    k2 = (2 * math.pi / n) ** 2 * (ax[0] ** 2 + ax[1] ** 2 + ax[2] ** 2)
    k2[0, 0, 0] = 1.0
    k = torch.where(ax[d].abs() * 2 == n, torch.zeros_like(ax[d]), 2 * math.pi / n * ax[d])
    return k / k2


def _cic(x, n):
    fl = torch.floor(x.detach())
    f = x - fl
    i0 = torch.remainder(fl.long(), n)
    i1 = torch.remainder(i0 + 1, n)
    for q in range(8):
        b = (q & 1, (q >> 1) & 1, q >> 2)
        i = [i1[:, a] if b[a] else i0[:, a] for a in range(3)]
        w = [f[:, a] if b[a] else 1 - f[:, a] for a in range(3)]
        yield (i[2] * n + i[1]) * n + i[0], w[0] * w[1] * w[2]


def _exact_model(ng, nf, steps, amp, noise):
    """The model in 64 bits: density contrast of the white noise `noise`."""
    ic, st = dpm_schedule(steps)
    r = nf // ng
    wk = torch.fft.rfftn(noise.view(ng, ng, ng))
    psi = torch.stack([torch.fft.irfftn(1j * _kfac(ng, d) * amp * wk, s=(ng, ng, ng)).reshape(-1) for d in range(3)], 1) * r
    q = torch.arange(ng, dtype=torch.float64, device="cuda") * r
    lat = torch.stack([t.reshape(-1) for t in reversed(torch.meshgrid(q, q, q, indexing="ij"))], 1)
    x, p = lat + ic[0] * psi, ic[1] * psi
    K = [_kfac(nf, d) for d in range(3)]

    def deposit(x):
        rho = torch.zeros(nf ** 3, dtype=torch.float64, device="cuda")
        for m, w in _cic(x, nf):
            rho = rho.index_add(0, m, w)
        return rho

    def force(x):
        rk = torch.fft.rfftn(deposit(x).view(nf, nf, nf))
        F = [torch.fft.irfftn(1j * K[d] * rk, s=(nf, nf, nf)).reshape(-1) for d in range(3)]
        out = [0.0, 0.0, 0.0]
        for m, w in _cic(x, nf):
            out = [out[d] + w * F[d].index_select(0, m) for d in range(3)]
        return torch.stack(out, 1)

    F = force(x)
    for ka, dr, kb in st:
        p = p + ka * F
        x = x + dr * p
        F = force(x)
        p = p + kb * F
    return deposit(x) * (nf ** 3 / ng ** 3) - 1.0


def dpm_schedule(steps, a0=0.1, a1=1.0):
    """Growth of the initial conditions and the kick and drift coefficients, by quadrature."""
    om = OMEGA_M

    def e(a):
        return np.sqrt(om / a ** 3 + 1 - om)

    def growth(a):
        hsq = om / a ** 3 + 1 - om
        oma, ola = om / (a ** 3 * hsq), (1 - om) / hsq
        return a * 2.5 * oma / (oma ** (4.0 / 7) - ola + (1 + oma / 2) * (1 + ola / 70))

    def integral(f, lo, hi):
        x, w = np.polynomial.legendre.leggauss(40)
        return 0.5 * (hi - lo) * float(np.sum(w * f(0.5 * (hi - lo) * x + 0.5 * (hi + lo))))

    h = 1e-5 * a0
    f = (math.log(growth(a0 + h)) - math.log(growth(a0 - h))) / (math.log(a0 + h) - math.log(a0 - h))
    d0 = growth(a0) / growth(1.0)
    at = np.linspace(a0, a1, steps + 1)
    out = []
    for lo, hi in zip(at[:-1], at[1:]):
        mid = 0.5 * (lo + hi)
        out.append((1.5 * om * integral(lambda a: 1 / (a * a * e(a)), lo, mid), integral(lambda a: 1 / (a ** 3 * e(a)), lo, hi),
                    1.5 * om * integral(lambda a: 1 / (a * a * e(a)), mid, hi)))
    return (d0, a0 ** 2 * d0 * f * e(a0)), out


def _exact_power(c, seed):
    x, _ = _particles(c, seed)
    x = torch.from_numpy(x).cuda()
    nc, ng, res = c["nc"], c["mesh"], 256.0 if c["izipx"] == 1 else 65536.0
    pos = (torch.floor(x * res) + 0.5) / res * (ng / nc) - 0.5
    rho = torch.zeros(ng ** 3, dtype=torch.float64, device="cuda")
    for m, w in _cic(pos, ng):
        rho = rho.index_add(0, m, w)
    ck = torch.fft.rfftn((rho / rho.mean() - 1.0).view(ng, ng, ng)) / ng ** 3
    ny = ng // 2
    f = torch.fft.fftfreq(ng, dtype=torch.float64, device="cuda") * ng
    fx = torch.arange(ny + 1, dtype=torch.float64, device="cuda")
    kx, ky, kz = fx.view(1, 1, -1), f.view(1, -1, 1), f.view(-1, 1, 1)
    kr = torch.sqrt(kx ** 2 + ky ** 2 + kz ** 2)
    s = torch.sinc(kx / ng) * torch.sinc(ky / ng) * torch.sinc(kz / ng)
    amp = ck.abs() ** 2 / s ** 4 * (4 * math.pi) * kr ** 3
    ix, i = torch.arange(ny + 1, device="cuda").view(1, 1, -1), torch.arange(ng, device="cuda")
    iy, iz = i.view(1, -1, 1), i.view(-1, 1, 1)
    edge = (ix == 0) | (ix == ny)
    skip = ((ix == 0) & (iy == 0) & (iz == 0)) | (edge & (iy > ny)) | (edge & ((iy == 0) | (iy == ny)) & (iz > ny))
    b = torch.where(skip, torch.zeros((), dtype=torch.long, device="cuda"), torch.round(kr).long()).reshape(-1)
    nbin = int(round(ny * math.sqrt(3.0)))
    cnt, ks, ps = (torch.zeros(nbin + 2, dtype=torch.float64, device="cuda").index_add(0, b, v.expand(ng, ng, ny + 1).reshape(-1))[1: nbin + 1]
                   for v in (torch.ones_like(kr), kr, amp))
    return dict(k=(ks / cnt * 2 * math.pi / 100.0).cpu(), power=(ps / cnt).cpu(), modes=None)


def exact(case, seed):
    c, kind = dict(case), case["kind"]
    if kind == "power":
        return _exact_power(c, seed)
    if kind not in ("forward", "grad"):
        return None
    ng, nf = c["ng"], c["ng"] * c["ratio"]
    m = np.fft.fftfreq(ng) * ng
    kz, ky, kx = np.meshgrid(m, m, np.arange(ng // 2 + 1), indexing="ij")
    k = 2 * np.pi / c["box"] * np.sqrt(kx ** 2 + ky ** 2 + kz ** 2)
    # the linear spectrum as the program hands it over, in 32 bits: an input
    amp = np.sqrt(np.where(k > 0, COSMO.pk(np.where(k > 0, k, 1.0)), 0.0) / (c["box"] / ng) ** 3).astype(np.float32)
    amp = torch.from_numpy(amp.astype(np.float64)).cuda()
    noise, target = _noise(c, seed)
    if kind == "forward":
        with torch.no_grad():
            return dict(delta=_exact_model(ng, nf, c["steps"], amp, noise.double()))
    w = noise.double().requires_grad_(True)
    delta = _exact_model(ng, nf, c["steps"], amp, w)
    (grad,) = torch.autograd.grad(delta, w, 2.0 / nf ** 3 * (delta.detach() - target.double()))
    return dict(delta=delta.detach(), noise_bar=grad)
