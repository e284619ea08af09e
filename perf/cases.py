"""Performance cases: the work that users of this framework have it do, each
through its public entry points, with FP64 references in plain torch.

Inputs are made on the GPU from the seed alone: porosity masks by thresholding
Gaussian-smoothed noise (a fixed share of pores), divergence-free pore
velocities as the curl of a vector potential that vanishes on every edge that
touches a solid, initial magnetization 1 in the pores.  These are the
distributions of `initializator_amd.generators`, which makes them on the host.

Every simulation pass is one run of a prepared solver with the signal of each
step, and the download of the state it ends in: a pass continues from the state
that the pass before it left, as a program does that saves its state every few
hundred or thousand steps.
"""
import math

import numpy as np
import torch

from initializator_amd.generators import G_REF, gradient_for_b, pgse_schedule, stable_dt
from initializator_amd.solver import BatchSolver, Corrector, HipSolver

DX, DIFF = 1e-6, 2.3e-9  # voxel size (m), pore diffusivity (m^2/s)
DT = stable_dt(DX, DIFF)
VMAX = 1e-3  # largest face velocity (m/s)
DELTA, BIG_DELTA = 2e-3, 20e-3  # lobes of the pulsed-gradient pair (s)
T2_BULK = 2.0

# Each domain case: grid nx, ny, nz, components nc, porosity phi, surface
# relaxivity rho (m/s), steps per pass; grad: pulsed gradient (T/m); scheme,
# bc (one code per axis: 0 zero derivative, 1 periodic, 2 zero value).
_DOMAIN = dict(kind="domain", nc=2, phi=0.2, rho=10e-6, grad=0.0, flow=True, exact_phase=False, mak=False,
               bcx=0, bcy=0, bcz=0, tilt=False, trim=0, field=False, mixture=False)


def _domain(name=None, **kw):
    d = dict(_DOMAIN, **kw)
    return dict(name=name, **d) if name else d


def listed():
    return [
        # A Carr-Purcell train on a small sample: RF pulses between runs of a few dozen
        # steps, all three components, the shortest calls of a pulse sequence.
        dict(name="cpmg_48", kind="cpmg", nx=48, ny=48, nz=48, phi=0.3, rho=10e-6, echoes=20, half=25, grad=0.02),
        # The plain decay configuration (64^3, one real component, no flow, no gradient).
        _domain("decay_64", nx=64, ny=64, nz=64, nc=1, phi=0.3, flow=False, steps=2000),
        # The flagship configuration: 256^3, flow, both lobes of the pulsed gradient and the decay after.
        _domain("flow_256", nx=256, ny=256, nz=256, grad=0.3, steps=2000),
        # A slab of a large sample (one eighth of 512 x 512 x 1024 with its ghost planes).
        _domain("flow_slab_512", nx=512, ny=512, nz=130, grad=0.3, rho=5e-6, steps=1000),
        # A ragged crop of a scan: odd sizes, three components, tilted main field, gradient on
        # three axes, a trimmed signal window.
        _domain("crop_203x97x151", nx=203, ny=97, nz=151, nc=3, phi=0.3, grad=0.1, tilt=True, trim=3, steps=1000),
        # The second-order scheme at the flagship size.
        _domain("maccormack_256", nx=256, ny=256, nz=256, grad=0.3, mak=True, steps=1000),
        # A periodic sample in an inhomogeneous field (per-voxel field map).
        _domain("periodic_field_160", nx=160, ny=160, nz=160, phi=0.25, bcx=1, bcy=1, bcz=1, field=True, steps=1000),
        # Two fluids: per-voxel diffusivity and relaxation, two weighted signals per step.
        _domain("mixture_128", nx=128, ny=128, nz=128, phi=0.3, grad=0.1, mixture=True, steps=1000),
        # Many uneven samples at once, each with its own gradient (replayed graph
        # chunks and a rest).
        dict(name="batch_24", kind="batch", count=24, lo=32, hi=128, steps=500, exact_phase=False),
        # The learned solve: coarse steps of eight plain ones, corrected by the net, checked, and
        # redone as plain steps where the check fails.
        dict(name="learned_128", kind="learned", nx=128, ny=128, nz=128, phi=0.2, rho=10e-6, grad=0.3, coarse=60,
             factor=8),
        # Training the net on what the batch generates.
        dict(name="train_8", kind="train", count=8, lo=32, hi=96, rounds=2, factor=8, stride=8),
        # The net alone on given features: outputs, and the parameter gradients.
        dict(name="net_96x80x64", kind="net", nx=96, ny=80, nz=64),
    ]


def draw(rng):
    def size(lo, hi):  # log-uniform, any parity
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["domain"] * 7 + ["cpmg", "batch", "learned", "train", "net"])
    phi = round(rng.uniform(0.15, 0.4), 3)
    if kind == "domain":
        nx, ny, nz = size(40, 288), size(40, 288), size(40, 200)
        special = rng.choice(["plain", "plain", "plain", "exact", "mak", "general", "mixture"])
        nc = rng.choice([1, 2, 2, 3]) if special != "exact" else 2
        kw = dict(nx=nx, ny=ny, nz=nz, nc=nc, phi=phi, rho=rng.choice([1e-6, 5e-6, 10e-6, 30e-6]),
                  flow=rng.random() < 0.8, grad=rng.choice([0.0, 0.05, 0.3]) if nc > 1 else 0.0,
                  steps=rng.randint(300, 1500), exact_phase=special == "exact", mak=special == "mak",
                  mixture=special == "mixture", tilt=nc == 3 and special != "general" and rng.random() < 0.5,
                  trim=rng.choice([0, 0, 2, 5]))
        if special in ("general", "mak", "mixture"):
            kw.update(bcx=rng.randint(0, 2), bcy=rng.randint(0, 2), bcz=rng.randint(0, 2))
            kw["field"] = special == "general" and nc > 1
        return _domain(**kw)
    if kind == "cpmg":
        return dict(kind="cpmg", nx=size(20, 96), ny=size(20, 96), nz=size(20, 96), phi=phi, rho=10e-6,
                    echoes=rng.randint(5, 30), half=rng.randint(5, 50), grad=0.02)
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(4, 28), lo=rng.randint(24, 48), hi=rng.randint(64, 128),
                    steps=rng.randint(65, 600), exact_phase=rng.random() < 0.5)
    if kind == "learned":
        return dict(kind="learned", nx=size(60, 160), ny=size(60, 160), nz=size(60, 160), phi=phi, rho=10e-6,
                    grad=rng.choice([0.05, 0.3]), coarse=rng.randint(20, 80), factor=8)
    if kind == "train":
        return dict(kind="train", count=rng.randint(2, 8), lo=rng.randint(20, 40), hi=rng.randint(48, 96),
                    rounds=rng.randint(1, 2), factor=8, stride=rng.randint(0, 12))
    return dict(kind="net", nx=size(20, 128), ny=size(20, 128), nz=size(20, 96))


# ---------------------------------------------------------------------------
# inputs

def _generator(seed, stream):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + stream) % (1 << 62))


def _smooth(shape, seed, stream, sigma):
    """Gaussian-smoothed white noise (reflecting edges, 4 sigma)."""
    a = torch.randn(shape, generator=_generator(seed, stream), device="cuda")
    r = int(4 * sigma + 0.5)
    t = torch.arange(-r, r + 1, dtype=torch.float64)
    w = torch.exp(-0.5 * (t / sigma) ** 2)
    w = (w / w.sum()).tolist()
    for ax in range(3):
        n = shape[ax]
        out = torch.zeros_like(a)
        at = torch.arange(n, device="cuda")
        for k in range(-r, r + 1):
            i = (at + k) % (2 * n)
            i = torch.where(i < n, i, 2 * n - 1 - i)
            out += a.index_select(ax, i) * w[k + r]
        a = out
    return a


def _porosity(shape, phi, seed, sigma=3.0):
    """Pore mask with the round(phi*N) largest smoothed values."""
    s = _smooth(shape, seed, 0, sigma).flatten()
    keep = s.argsort(stable=True)[s.numel() - int(round(phi * s.numel())):]
    mask = torch.zeros(s.numel(), dtype=torch.bool, device="cuda")
    mask[keep] = True
    return mask.view(shape)


def _velocity(mask, seed, sigma=4.0):
    """Divergence-free face velocities (FP64) that vanish on pore-solid faces."""
    nz, ny, nx = mask.shape
    p = torch.zeros((nz + 2, ny + 2, nx + 2), dtype=torch.bool, device="cuda")
    p[1:-1, 1:-1, 1:-1] = mask
    ax = p[:-1, :-1, 1:-1] & p[:-1, 1:, 1:-1] & p[1:, :-1, 1:-1] & p[1:, 1:, 1:-1]
    ay = p[:-1, 1:-1, :-1] & p[:-1, 1:-1, 1:] & p[1:, 1:-1, :-1] & p[1:, 1:-1, 1:]
    az = p[1:-1, :-1, :-1] & p[1:-1, :-1, 1:] & p[1:-1, 1:, :-1] & p[1:-1, 1:, 1:]
    ax = _smooth(tuple(ax.shape), seed, 1, sigma).double() * ax
    ay = _smooth(tuple(ay.shape), seed, 2, sigma).double() * ay
    az = _smooth(tuple(az.shape), seed, 3, sigma).double() * az
    vx = (az[:, 1:] - az[:, :-1]) - (ay[1:] - ay[:-1])
    vy = (ax[1:] - ax[:-1]) - (az[:, :, 1:] - az[:, :, :-1])
    vz = (ay[:, :, 1:] - ay[:, :, :-1]) - (ax[:, 1:] - ax[:, :-1])
    peak = max(float(v.abs().max()) for v in (vx, vy, vz))
    return [v * (VMAX / peak if peak > 0 else 1.0) for v in (vx, vy, vz)]


def _host(t):
    return t.double().cpu().numpy()


def _domain_inputs(case, seed):
    """What a program has before it makes its solver, as CUDA tensors."""
    shape = (case["nz"], case["ny"], case["nx"])
    mask = _porosity(shape, case["phi"], seed)
    d = dict(shape=shape, mask=mask, vel=_velocity(mask, seed) if case.get("flow", True) else None)
    if case.get("field"):  # susceptibility-like field map, tens of microtesla
        d["field"] = _smooth(shape, seed, 7, 5.0).double() * 1e-3
    if case.get("mixture"):  # two fluids with a smooth saturation, rates and weights by volume
        s = torch.sigmoid(20.0 * _smooth(shape, seed, 8, 4.0).double() * 4.0)
        d["D"] = mask * (DIFF * s + 0.4e-9 * (1 - s))
        d["r2"] = mask * (s / T2_BULK + (1 - s) / 0.3 + 2.0)
        d["r1"] = d["r2"] / 1.5
        d["w"] = (mask * s, mask * (1 - s))
    return d


def _axis(case):
    return (0.6, 0.0, 0.8) if case.get("tilt") else (0.0, 0.0, 1.0)


def _schedule(case):
    """[steps, 3] pulsed gradients, or None without any."""
    if not case["grad"] or case["nc"] == 1:
        return None
    s = pgse_schedule(case["steps"], DT, case["grad"], DELTA, BIG_DELTA)
    if case["nc"] == 3:
        s[:, 0], s[:, 1] = 0.5 * s[:, 2], -0.25 * s[:, 2]
    return s


def _initial(case, mask):
    """Magnetization after a 90 degree pulse (or its one real component)."""
    m = mask.double()
    z = torch.zeros_like(m)
    return [m, z, 0.25 * m][: case["nc"]]


def _solver(case, d):
    s = HipSolver(d["shape"], case["nc"], DX, DT, DIFF, 1.0 / T2_BULK, r1_bulk=1.0 / 2.5, rho1=0.5 * case["rho"],
                  rho2=case["rho"], p_eq=1.0 if case["nc"] == 3 else 0.0, b0_dir=_axis(case),
                  velocity=d["vel"] is not None, precession=case["nc"] > 1 and bool(case["grad"] or case["field"]),
                  phase_exact=case["exact_phase"], buffer=(case["trim"],) * 3, scheme=int(case["mak"]),
                  bc=(case["bcx"], case["bcy"], case["bcz"]))
    s.upload_mask(d["mask"].cpu().numpy().astype(np.uint8))
    if d["vel"] is not None:
        s.upload_velocity(*[_host(v) for v in d["vel"]])
    if "field" in d:
        s.upload_field(_host(d["field"]))
    if "D" in d:
        s.upload_coefficients(_host(d["D"]), _host(d["r2"]), _host(d["r1"]))
        s.upload_phase_weights(_host(d["w"][0]), _host(d["w"][1]))
    s.upload_magnetization(*[_host(m) for m in _initial(case, d["mask"])])
    return s


def _cpmg_case(case):
    return _domain(nx=case["nx"], ny=case["ny"], nz=case["nz"], nc=3, phi=case["phi"], rho=case["rho"],
                   grad=case["grad"], flow=False, steps=1)


def _cpmg_solver(case, d):
    c = _cpmg_case(case)
    s = HipSolver(d["shape"], 3, DX, DT, DIFF, 1.0 / T2_BULK, r1_bulk=1.0 / 2.5, rho1=0.5 * c["rho"], rho2=c["rho"],
                  p_eq=1.0, grad=(0.0, 0.0, case["grad"]), precession=True)
    s.upload_mask(d["mask"].cpu().numpy().astype(np.uint8))
    m = d["mask"].double()
    z = _host(torch.zeros_like(m))
    s.upload_magnetization(z, z, _host(m))
    return s


def _batch_specs(case, seed):
    """Uneven instances as the batched workload draws them (edges lo..hi, all three their own; the
    grids belong to the case, what fills them to the seed)."""
    r = np.random.default_rng([int(seed), 17])
    grids = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    specs = []
    for i in range(case["count"]):
        shape = tuple(int(v) for v in grids.integers(case["lo"], case["hi"] + 1, 3))
        phi, rho, b = float(r.uniform(0.15, 0.4)), float(r.uniform(1e-6, 50e-6)), float(10.0 ** r.uniform(7.0, 9.0))
        mask = _porosity(shape, phi, int(seed) * 64 + i)
        specs.append(dict(shape=shape, rho1=rho, rho2=rho, grad_amp=gradient_for_b(b, DELTA, BIG_DELTA), delta=DELTA,
                          big_delta=BIG_DELTA, mask=mask, vel=_velocity(mask, int(seed) * 64 + i)))
    return specs


def _batch_solver(specs, exact_phase):
    b = BatchSolver(specs, 2, DX, DT, DIFF, 1.0 / T2_BULK, r1_bulk=1.0 / 2.5, velocity=True, precession=True,
                    phase_exact=exact_phase)
    for i, s in enumerate(specs):
        m = s["mask"].double()
        b.upload(i, s["mask"].cpu().numpy().astype(np.uint8), [_host(m), _host(torch.zeros_like(m))],
                 [_host(v) for v in s["vel"]])
    return b


def _trained_net(seed):
    """A corrector after a short training on four small samples."""
    specs = _batch_specs(dict(count=4, lo=32, hi=48), int(seed) + 5)
    b = _batch_solver(specs, True)
    net = Corrector(int(seed) % 1000)
    net.train(b, factor=8, rounds=60, stride=4, lr=2e-3)
    b.close()
    return net


def _net_inputs(case, seed):
    shape = (case["nz"], case["ny"], case["nx"])
    mask = _porosity(shape, 0.25, seed).double()
    f = torch.stack([_smooth(shape, seed, 20 + k, 3.0).double() * 8.0 for k in range(6)], -1) * mask[..., None]
    f[..., 2] = mask
    g = torch.randn(shape + (2,), generator=_generator(seed, 30), device="cuda").double() * mask[..., None]
    r = np.random.default_rng([int(seed), 31])
    w = np.concatenate([r.normal(0, math.sqrt(2 / 162), 2592), r.normal(0, 0.05, 16),
                        r.normal(0, math.sqrt(2 / 432), 6912), r.normal(0, 0.05, 16),
                        r.normal(0, math.sqrt(2 / 432), 864), r.normal(0, 0.05, 2)]).astype(np.float32)
    return f.float().cpu().numpy(), g.float().cpu().numpy(), w


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "domain":
        st["solver"] = _solver(case, _domain_inputs(case, seed))
        st["sched"] = _schedule(case)
    elif kind == "cpmg":
        st["solver"] = _cpmg_solver(case, _domain_inputs(_cpmg_case(case), seed))
    elif kind == "batch":
        st["batch"] = _batch_solver(_batch_specs(case, seed), case["exact_phase"])
        st["batch"].autotune(3)
    elif kind == "learned":
        c = _domain(nx=case["nx"], ny=case["ny"], nz=case["nz"], phi=case["phi"], rho=case["rho"], grad=case["grad"],
                    exact_phase=True, steps=case["coarse"] * case["factor"])
        st["solver"] = _solver(c, _domain_inputs(c, seed))
        st["sched"] = _schedule(c)
        st["net"] = _trained_net(seed)
    elif kind == "train":
        st["batch"] = _batch_solver(_batch_specs(case, seed), True)
        st["net"] = Corrector(int(seed) % 1000)
    else:
        st["net"] = Corrector(0)
        st["features"], st["grad_out"], st["net"].params = _net_inputs(case, seed)
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "domain":
        sig = state["solver"].run(case["steps"], state["sched"])
        return dict(signal=sig, m=state["solver"].download_magnetization())
    if kind == "cpmg":
        s, h = state["solver"], case["half"]
        s.pulse(2, math.pi / 2, (1.0, 0.0, 0.0))
        sig = [s.run(h)]
        for k in range(case["echoes"]):
            s.pulse(2, math.pi, (0.0, 1.0, 0.0))
            sig.append(s.run(2 * h))
        return dict(signal=np.concatenate(sig), m=s.download_magnetization())
    if kind == "batch":
        sig = state["batch"].run(case["steps"])
        return dict(signal=sig, m=[state["batch"].download(i) for i in range(case["count"])])
    if kind == "learned":
        sig, _ = state["net"].run_learned(state["solver"], case["coarse"], case["factor"], state["sched"])
        return dict(signal=sig, m=state["solver"].download_magnetization())
    if kind == "train":
        losses = state["net"].train(state["batch"], factor=case["factor"], rounds=case["rounds"],
                                    stride=case["stride"])
        return dict(losses=losses, params=state["net"].params)
    return dict(out=state["net"].forward(state["features"]),
                grad=state["net"].backward(state["features"], state["grad_out"]))


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _solve_work(vox, phi, nc, steps, extra=0):
    """A step reads and writes the state of the pores and reads their three velocity sums (extra: further
    per-pore words); the pore map is one bit a voxel.  Solids never change.  About 24 + 24 nc FP32
    operations a pore and step (six face weights, six differences a component, relaxation, precession)."""
    pores = phi * vox
    return steps * (pores * (8.0 * nc + 12.0 + 4.0 * extra) + vox / 8.0), steps * pores * (24.0 + 24.0 * nc)


def work(case):
    kind = case["kind"]
    if kind in ("domain", "cpmg", "learned"):
        vox = case["nx"] * case["ny"] * case["nz"]
        if kind == "domain":
            # the second-order scheme passes over the pores twice
            steps, nc = case["steps"] * (2 if case["mak"] else 1), case["nc"]
            extra = (0 if case["flow"] else -3) + (1 if case["field"] else 0) + (4 if case["mixture"] else 0)
        elif kind == "cpmg":
            steps, nc, extra = case["half"] * (1 + 2 * case["echoes"]), 3, -3
        else:
            steps, nc, extra = case["coarse"], 2, 0
        by, fl = _solve_work(vox, case["phi"], nc, steps, extra)
        if kind == "learned":  # the net's multiply-adds on the pores, its features and outputs once
            fl += 2.0 * 10368 * case["phi"] * vox * case["coarse"]
            by += 24.0 * case["phi"] * vox * case["coarse"]
        return dict(bytes=by + 8.0 * nc * vox, flops=fl)
    if kind in ("batch", "train"):
        vox = case["count"] * ((case["lo"] + case["hi"]) / 2.0) ** 3
        if kind == "batch":
            by, fl = _solve_work(vox, 0.275, 2, case["steps"])
            return dict(bytes=by + 16.0 * vox, flops=fl)
        by, fl = _solve_work(vox, 0.275, 2, case["rounds"] * (case["stride"] + case["factor"] + 1))
        # forward and both backward products of the net
        return dict(bytes=by + case["rounds"] * vox * 32.0, flops=fl + case["rounds"] * vox * 2.0 * 3 * 10368)
    vox = case["nx"] * case["ny"] * case["nz"]
    return dict(bytes=vox * 4.0 * (6 + 2 + 6 + 2), flops=vox * 2.0 * 4 * 10368)


# ---------------------------------------------------------------------------
# the same in 64 bits, without this repository's kernels

class _Pores:
    """One or several domains as lists of pores: neighbour positions and face weights in FP64."""

    def __init__(self, case, d, rho1, rho2):
        mask = d["mask"]
        nz, ny, nx = mask.shape
        n = int(mask.sum())
        pid = torch.full(mask.shape, -1, dtype=torch.int64, device="cuda")
        pid[mask] = torch.arange(n, device="cuda")
        self.mask, self.n = mask, n
        zyx = mask.nonzero()
        self.z, self.y, self.x = (zyx[:, k].double() for k in range(3))
        own = torch.arange(n, device="cuda")
        bc = (case["bcx"], case["bcy"], case["bcz"])
        mak = case["mak"]
        rates = [torch.full((n,), r, dtype=torch.float64, device="cuda") for r in (1.0 / 2.5, 1.0 / T2_BULK)]
        D = d["D"][mask] if "D" in d else None
        cd = DT * DIFF / DX ** 2
        self.nb, self.w = [], []
        for ax, size, vel in ((0, nx, 0), (1, ny, 1), (2, nz, 2)):
            dim = 2 - ax
            pos = zyx[:, dim]
            sums = None
            if d["vel"] is not None:
                v = d["vel"][vel].float().double()  # the solver holds FP32 velocities
                lo, hi = v.narrow(dim, 0, size)[mask], v.narrow(dim, 1, size)[mask]
                sums = lo + hi
            for side in (-1, 1):
                edge = pos == (0 if side < 0 else size - 1)
                j = pid.roll(-side, dim)[mask]
                solid = (j < 0) & ~edge
                if bc[ax] == 0:
                    j = torch.where(edge, own, j)
                elif bc[ax] == 2:
                    j = torch.where(edge, torch.full_like(j, n), j)
                else:  # a solid opposite cell holds 0
                    j = torch.where(edge & (j < 0), torch.full_like(j, n), j)
                j = torch.where(solid, own, j)
                kn = (~solid).double()
                if D is None:
                    w = cd * kn
                else:
                    other = torch.where(edge | solid | (j >= n), D, D[j.clamp(max=n - 1)])
                    w = DT / DX ** 2 * kn * 2 * D * other / (D + other)
                adv = torch.zeros_like(w)
                if sums is not None:
                    h = 0.5 * DT / DX
                    face = lo if side < 0 else hi
                    if not mak:
                        adv = torch.where(face != 0, h * (-side * sums).clamp(min=0.0), adv)
                    else:
                        adv = -side * kn * h * sums
                self.nb.append(j.int())
                self.w.append((w, adv, side))
                for q, rho in enumerate((rho1, rho2)):
                    rates[q] += solid * rho / DX
        if "r2" in d:
            rates = [d["r1"][mask], d["r2"][mask]]
        self.r1, self.r2 = (DT * r for r in rates)

    def weights(self, stage):
        """(neighbour, weight) of the faces, upwind or of one of the two second-order stages; the first
        is the pore itself."""
        faces = [(j, (w + (a if stage == "up" or side == (-1 if stage == "predict" else 1) else 0.0))[:, None])
                 for j, (w, a, side) in zip(self.nb, self.w)]
        return [(None, -sum(w for _, w in faces))] + faces


def _rate(faces, m):
    """sum of w (m[neighbour] - m) over the faces; neighbour n reads 0."""
    p = torch.cat([m, torch.zeros_like(m[:1])])
    d = faces[0][1] * m
    for j, w in faces[1:]:
        d.addcmul_(w, p.index_select(0, j))
    return d


def _rotate(v, axis, angle):
    """Rotation by angle about a unit axis (right-handed with M x B precession reversed)."""
    a = torch.tensor(axis, dtype=torch.float64, device="cuda")
    c, s = math.cos(angle), math.sin(angle)
    return v * c + torch.linalg.cross(a.expand_as(v), v) * s + a * (v * a).sum(1, keepdim=True) * (1 - c)


def _full(pores, m):
    out = []
    for q in range(m.shape[1]):
        f = torch.zeros(pores.mask.shape, dtype=torch.float64, device="cuda")
        f[pores.mask] = m[:, q]
        out.append(f.cpu().numpy())
    return out


def _exact_domain(case, seed):
    d = _domain_inputs(case, seed)
    nc, mak = case["nc"], case["mak"]
    p = _Pores(case, d, 0.5 * case["rho"], case["rho"])
    sched = _schedule(case)
    m = torch.stack([f[d["mask"]] for f in _initial(case, d["mask"])], 1)
    t = case["trim"]
    inside = torch.ones(p.n, dtype=torch.bool, device="cuda")
    for pos, size in ((p.x, case["nx"]), (p.y, case["ny"]), (p.z, case["nz"])):
        inside &= (pos >= t) & (pos < size - t)
    weights = [inside * w[d["mask"]] for w in d["w"]] if "w" in d else [inside.double()]
    axis = torch.tensor(_axis(case), dtype=torch.float64, device="cuda")
    field = d["field"][d["mask"]] if "field" in d else None
    stages = [p.weights(s) for s in (("predict", "correct") if mak else ("up",))]

    def change(faces, v, g):
        out = _rate(faces, v)
        if nc == 3:
            par = (v * axis).sum(1, keepdim=True) * axis
            out += p.r1[:, None] * (axis - par) + p.r2[:, None] * (par - v)
        else:
            out -= p.r2[:, None] * v
        angle = [DT * G_REF * g[k] * DX * (pos + 0.5) for k, pos in enumerate((p.x, p.y, p.z))] if g is not None else None
        if field is not None:
            b = DT * G_REF * field
            angle = [torch.zeros_like(b), torch.zeros_like(b), b] if angle is None else [angle[0], angle[1], b]
        if nc == 2 and angle is not None:
            if case["exact_phase"]:
                s, c1 = torch.sin(angle[2]), torch.cos(angle[2]) - 1
                out += torch.stack([v[:, 1] * s + v[:, 0] * c1, v[:, 1] * c1 - v[:, 0] * s], 1)
            else:
                out += torch.stack([angle[2] * v[:, 1], -angle[2] * v[:, 0]], 1)
        elif nc == 3 and angle is not None:
            out += torch.linalg.cross(v, torch.stack(angle, 1))
        return out

    def sums(m):
        return torch.cat([(w[:, None] * m).sum(0) for w in weights])

    signal = [sums(m)]
    for k in range(case["steps"]):
        g = sched[k] if sched is not None and sched[k].any() else None
        n = m + change(stages[0], m, g)
        if mak:
            n = 0.5 * (m + n + change(stages[1], n, g))
        m = n
        signal.append(sums(m))
    return dict(signal=torch.stack(signal).cpu().numpy(), m=_full(p, m))


def _exact_cpmg(case, seed):
    c = _cpmg_case(case)
    d = _domain_inputs(c, seed)
    p = _Pores(c, d, 0.5 * c["rho"], c["rho"])
    faces = p.weights("up")
    m = torch.zeros((p.n, 3), dtype=torch.float64, device="cuda")
    m[:, 2] = 1.0
    axis = torch.tensor((0.0, 0.0, 1.0), dtype=torch.float64, device="cuda")
    angle = DT * G_REF * case["grad"] * DX * (p.z + 0.5)
    signal = []

    def steps(m, n):
        signal.append(m.sum(0))
        for _ in range(n):
            par = m[:, 2:] * axis
            dm = _rate(faces, m) + p.r1[:, None] * (axis - par) + p.r2[:, None] * (par - m)
            dm[:, 0] += angle * m[:, 1]
            dm[:, 1] -= angle * m[:, 0]
            m = m + dm
            signal.append(m.sum(0))
        return m

    m = steps(_rotate(m, (1.0, 0.0, 0.0), math.pi / 2), case["half"])
    for _ in range(case["echoes"]):
        m = steps(_rotate(m, (0.0, 1.0, 0.0), math.pi), 2 * case["half"])
    return dict(signal=torch.stack(signal).cpu().numpy(), m=_full(p, m))


def _exact_batch(case, seed):
    specs = _batch_specs(case, seed)
    base = _domain(nx=1, ny=1, nz=1, steps=1)
    parts = [_Pores(base, s, s["rho1"], s["rho2"]) for s in specs]
    first = np.cumsum([0] + [p.n for p in parts])
    lists = [p.weights("up") for p in parts]
    faces = [(None if k == 0 else torch.cat([f[k][0] + int(first[i]) for i, f in enumerate(lists)]).int(),
              torch.cat([f[k][1] for f in lists])) for k in range(7)]
    r2 = torch.cat([p.r2 for p in parts])
    unit = torch.cat([DT * G_REF * s["grad_amp"] * DX * (p.z + 0.5) for s, p in zip(specs, parts)])
    m = torch.zeros((int(first[-1]), 2), dtype=torch.float64, device="cuda")
    m[:, 0] = 1.0
    nd, nD = round(DELTA / DT), round(BIG_DELTA / DT)

    def sums(m):
        return torch.stack([v.sum(0) for v in m.split(np.diff(first).tolist())])

    signal = [sums(m)]
    for k in range(case["steps"]):
        d = _rate(faces, m) - r2[:, None] * m
        sign = -1.0 if nD <= k < nD + nd else 1.0 if k < nd else 0.0
        if sign:
            a = sign * unit
            if case["exact_phase"]:
                s, c1 = torch.sin(a), torch.cos(a) - 1
                d += torch.stack([m[:, 1] * s + m[:, 0] * c1, m[:, 1] * c1 - m[:, 0] * s], 1)
            else:
                d += torch.stack([a * m[:, 1], -a * m[:, 0]], 1)
        m = m + d
        signal.append(sums(m))
    return dict(signal=torch.stack(signal, 1).cpu().numpy(),
                m=[_full(p, m[int(first[i]):int(first[i + 1])]) for i, p in enumerate(parts)])


def _conv(x, w, b):
    """3x3x3 zero-padded convolution, channels last: w [out][in][27]."""
    nz, ny, nx, _ = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = b.expand(nz * ny * nx, -1)
    for k in range(27):
        z, y, c = k // 9, k // 3 % 3, k % 3
        out = out + p[z:z + nz, y:y + ny, c:c + nx].reshape(-1, x.shape[3]) @ w[:, :, k].T.contiguous()
    return out.view(nz, ny, nx, -1)


def _exact_net(case, seed):
    f, g, w = _net_inputs(case, seed)
    p = torch.tensor(w, dtype=torch.float64, device="cuda", requires_grad=True)
    x = torch.tensor(f, dtype=torch.float64, device="cuda")
    x = torch.relu(_conv(x, p[:2592].view(16, 6, 27), p[2592:2608]))
    x = torch.relu(_conv(x, p[2608:9520].view(16, 16, 27), p[9520:9536]))
    out = _conv(x, p[9536:10400].view(2, 16, 27), p[10400:])
    (out * torch.tensor(g, dtype=torch.float64, device="cuda")).sum().backward()
    return dict(out=out.detach().cpu().numpy(), grad=p.grad.cpu().numpy())


def exact(case, seed):
    kind = case["kind"]
    if kind == "domain":
        return _exact_domain(case, seed)
    if kind == "cpmg":
        return _exact_cpmg(case, seed)
    if kind == "batch":
        return _exact_batch(case, seed)
    if kind == "net":
        return _exact_net(case, seed)
    return None  # bfloat16 training and the accept-or-redo decisions of the learned solve have no such value
