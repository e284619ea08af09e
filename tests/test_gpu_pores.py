"""The sweeps over the list of the pores (the automatic choice) against the
row layout: the same operations on the same values, so the fields agree bit
for bit and the signal to the order of its FP64 sums (rtol 1e-12, as between
the other layouts).  Masks sit on the edges of the list: groups of exactly 64
pores and one more or less, planes without a pore, a grid of pores only, one
pore, planes whose neighbours lie further apart than a 16-bit offset (the
tile sweeps take over), and solids that pores read."""
import numpy as np
import pytest

from initializator_amd import generators
from initializator_amd.solver import BatchSolver, HipSolver

pytestmark = pytest.mark.gpu

DX, D = 1e-6, 2.3e-9
DT = generators.stable_dt(DX, D)


def _mask(kind):
    if kind in (63, 64, 65, 128, 129):  # pores of each plane
        shape = (5, 13, 21)
        m = np.zeros(shape, np.uint8)
        for z in range(shape[0]):
            m[z].flat[np.random.default_rng([kind, z]).permutation(13 * 21)[:kind]] = 1
        return m
    if kind == "gaps":  # planes and rows without pores
        m = generators.porosity((9, 14, 30), 0.4, seed=3, sigma=1.0)
        m[0] = m[4] = m[8] = 0
        m[:, 5] = 0
        return m
    if kind == "full":
        return np.ones((4, 11, 18), np.uint8)
    if kind == "one":
        m = np.zeros((3, 4, 5), np.uint8)
        m[1, 2, 3] = 1
        return m
    if kind == "none":
        return np.zeros((3, 4, 5), np.uint8)
    assert kind == "far"  # 64 pores over a plane, all pores in the next one
    m = np.zeros((3, 300, 300), np.uint8)
    m[1] = 1
    for z in (0, 2):
        m[z].flat[np.random.default_rng(z).permutation(90000)[:64]] = 1
    return m


def _run(mask, m0, vel, rows, nc, sched, steps=11, **kw):
    prec = sched is not None
    with HipSolver(mask.shape, nc, DX, DT, D, 0.5, r1_bulk=0.4, rho1=4e-6, rho2=9e-6, velocity=vel is not None,
                   precession=prec, p_eq=0.1 if nc == 3 else 0.0, **kw) as s:
        s.set_layout(not rows)
        s.upload_mask(mask)
        if vel is not None:
            s.upload_velocity(*vel)
        s.upload_magnetization(*m0[:nc])
        out = []
        for k in range(2):  # the second run continues from a downloaded state
            out.append((s.run(steps, sched), s.download_magnetization()))
            if nc == 3:
                s.pulse(2, 0.3, (0.1, 0.9, 0.2))
            elif nc == 2:
                s.pulse(1, 2e-9, (0.0, 0.0, 1.0))
            out.append((s.signal(), s.download_magnetization()))
    return out


def _same(a, b):
    for (sa, fa), (sb, fb) in zip(a, b):
        for x, y in zip(fa, fb):
            assert np.array_equal(x, y, equal_nan=True)
        np.testing.assert_allclose(sa, sb, rtol=1e-12, atol=1e-300)


@pytest.mark.parametrize("kind", [63, 64, 65, 128, 129, "gaps", "full", "one", "none", "far"])
@pytest.mark.parametrize("scheme,bc,solid_flow", [(0, (0, 0, 0), False), (0, (0, 0, 0), True), (0, (1, 2, 1), True),
                                                  (1, (0, 0, 0), True), (1, (2, 1, 1), False)])
def test_list_equals_rows(kind, scheme, bc, solid_flow):
    mask = _mask(kind)
    rng = np.random.default_rng(7)
    nz, ny, nx = mask.shape
    if solid_flow:  # velocity on every face, some of them 0
        vel = [rng.uniform(-1e-3, 1e-3, s) * (rng.random(s) > 0.2)
               for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx))]
    else:
        vel = generators.velocity(mask, seed=2, sigma=1.0)
    m0 = [rng.random(mask.shape) - 0.3 for _ in range(3)]  # solids hold values too
    nc = 1 + (nx + scheme) % 3
    sched = None if nc == 1 else np.tile([0.0 if nc == 2 else 0.05, 0.0, 0.2], (11, 1))
    kw = dict(scheme=scheme, bc=bc, buffer=(1, 0, 1))
    if nc == 3:
        kw["b0_dir"] = (0.2, -0.3, 0.9)
    _same(_run(mask, m0, vel, False, nc, sched, **kw), _run(mask, m0, vel, True, nc, sched, **kw))


def test_solids_that_are_not_finite_leave_it_to_the_tiles():
    """A solid's NaN spreads as the tile sweeps on bricks spread it (their zero weight times NaN)."""
    mask = _mask("gaps")
    m0 = [mask.astype(float), np.zeros(mask.shape)]
    z, y, x = np.argwhere((mask[1:-1, 1:-1, 1:-1] == 0))[17] + 1
    m0[0][z, y, x] = np.nan
    outs = []
    for variant in (-1, 4):  # 4: 64 x 16 bricks
        with HipSolver(mask.shape, 2, DX, DT, D, 0.5) as s:
            s.set_tile(variant, 0)
            s.upload_mask(mask)
            s.upload_magnetization(*m0)
            outs.append((s.run(5), s.download_magnetization()))
    _same([outs[0]], [outs[1]])


@pytest.mark.parametrize("exact,graph", [(False, 0), (True, 4)])
def test_batch_list_equals_tiles(exact, graph):
    """The batch on the list of the pores (the automatic choice) against a tile of the batch: uneven
    instances, one of them without pores, one with velocity on pore-solid faces, solids that hold values;
    runs, a download between them, and an instance uploaded again."""
    kinds = [63, "gaps", "none", "full", "one", 129]
    rng = np.random.default_rng(11)
    specs = []
    for i, k in enumerate(kinds):
        m = _mask(k)
        nz, ny, nx = m.shape
        vel = generators.velocity(m, seed=i, sigma=1.0)
        if k == "gaps":
            vel = [rng.uniform(-1e-3, 1e-3, s) for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx))]
        specs.append(dict(shape=m.shape, mask=m, vel=vel, m0=[rng.random(m.shape), rng.random(m.shape) - 0.4],
                          rho1=(i + 1) * 1e-6, rho2=(i + 2) * 1e-6, grad_amp=0.1 * (i + 1), delta=3 * DT,
                          big_delta=(4 + i) * DT))
    again = [rng.random(specs[1]["shape"]) for _ in range(2)]
    outs = []
    for variant in (-1, 4):
        b = BatchSolver(specs, 2, DX, DT, D, 0.5, velocity=True, precession=True, phase_exact=exact, buffer=(0, 1, 0))
        b.set_tile(variant, 0, graph, True)
        for i, s in enumerate(specs):
            b.upload(i, s["mask"], s["m0"], s["vel"])
        out = [(b.run(9), b.download(1))]
        out.append((b.run(5), b.download(3)))
        b.upload(1, specs[1]["mask"], again, specs[1]["vel"])
        out.append((b.run(8), sum((b.download(i) for i in range(len(specs))), [])))
        outs.append(out)
        b.close()
    for (sa, fa), (sb, fb) in zip(*outs):
        for x, y in zip(fa, fb):
            assert np.array_equal(x, y)
        np.testing.assert_allclose(sa, sb, rtol=1e-11, atol=1e-13)


@pytest.mark.parametrize("shape,phi", [((8, 8, 8), 1.0), ((9, 17, 7), 0.5), ((16, 24, 8), 0.3), ((1, 1, 1), 1.0),
                                       ((3, 2, 100), 0.6), ((24, 24, 24), 1.0), ((64, 64, 64), 0.25),
                                       ((64, 64, 65), 0.25)])
@pytest.mark.parametrize("nc,vel,exact", [(1, False, False), (1, True, False), (2, False, False), (2, True, True),
                                          (2, False, True), (2, True, False), (3, False, False), (3, True, False)])
def test_several_steps_a_launch_equal_single_steps(shape, phi, nc, vel, exact):
    """Small grids take up to four steps a launch, box by box (64 x 64 x 65: one layer of boxes too many,
    single steps); against the row layout.  Boxes full of pores, off the grid's edge, without a pore; runs of
    1 to 11 steps, so of every remainder; a gradient that changes from step to step; a trimmed window; a field
    map that takes the problem to the general kernels and back."""
    mask = (np.ones(shape, np.uint8) if phi == 1.0 else generators.porosity(shape, phi, 3, sigma=2.0 if shape[0] > 8 else 0.7))
    if shape == (64, 64, 64):
        mask[:24, :24, :24] = 0
    rng = np.random.default_rng(4)
    v = generators.velocity(mask, 5, sigma=1.5, vmax=1e-3, d=(DX, DX, DX)) if vel else None
    m0 = [rng.random(shape) - 0.3 for _ in range(nc)]
    kw = dict(buffer=tuple(1 if n > 4 else 0 for n in shape[::-1]), phase_exact=exact)
    if nc == 3:
        kw.update(p_eq=0.1, **(dict(b0_dir=(0.2, -0.3, 0.9)) if vel else {}))
    field = rng.standard_normal(shape) * 1e-5
    outs = []
    for rows in (False, True):
        with HipSolver(shape, nc, DX, DT, D, 0.5, r1_bulk=0.4, rho1=4e-6, rho2=9e-6, velocity=vel, precession=nc > 1,
                       **kw) as s:
            s.set_layout(not rows)
            s.upload_mask(mask)
            if vel:
                s.upload_velocity(*v)
            s.upload_magnetization(*m0)
            out = []
            for steps in (1, 2, 3, 4, 11):
                g = None
                if nc > 1:
                    g = np.zeros((steps, 3))
                    g[:, 2] = np.arange(steps) % 3 * 0.1
                    g[:, :2] = 0.0 if nc == 2 else 0.03
                out.append((s.run(steps, g), s.download_magnetization()))
            if nc == 3 and not vel:
                for b in (field, None):
                    s.upload_field(b)
                    out.append((s.run(6), s.download_magnetization()))
            outs.append(out)
    _same(*outs)
