"""Calls that change which sweep the next run takes while the state lives in the
list of the pores: what they return equals a solver that never leaves the rows."""
import ctypes
import time

import numpy as np
import pytest

from initializator_amd import generators
from initializator_amd.solver import BatchSolver, HipSolver, check

pytestmark = pytest.mark.gpu

DX, D = 1e-6, 2.3e-9
DT = generators.stable_dt(DX, D)


def _solver(shape, mask, m0, nc, rows=False, **kw):
    s = HipSolver(shape, nc, DX, DT, D, 0.5, r1_bulk=0.4, rho1=4e-6, rho2=9e-6, **kw)
    s.set_layout(not rows)
    s.upload_mask(mask)
    s.upload_magnetization(*m0[:nc])
    return s


@pytest.mark.parametrize("leave", ["layout", "tile", "per voxel"])
@pytest.mark.parametrize("before", [False, True])
def test_signal_after_weights_that_come_while_another_sweep_is_set(leave, before):
    """A run leaves the state in the list only; then another sweep is set and
    phase weights are uploaded (the first ones, or others in place of them):
    the signal is that of the new weights, here and in row 0 of the next run."""
    shape, nc = (14, 11, 37), 2
    mask = generators.porosity(shape, 0.3, 5, sigma=1.0)
    rng = np.random.default_rng(6)
    m0 = [rng.random(shape) - 0.3 for _ in range(nc)]
    w = [rng.random(shape) for _ in range(4)]
    outs = []
    for rows in (False, True):
        with _solver(shape, mask, m0, nc, rows) as s:
            if before:
                s.upload_phase_weights(w[0], w[1])
            s.run(5)
            if not rows:
                s.set_layout(False) if leave == "layout" else s.set_tile(4 if leave == "tile" else -2)
            s.upload_phase_weights(w[2], w[3])
            outs.append([s.signal(), s.run(4), *s.download_magnetization()])
    for a, b in zip(*outs):
        np.testing.assert_allclose(a, b, rtol=1e-12, atol=1e-14)
    for a, b in zip(outs[0][2:], outs[1][2:]):
        np.testing.assert_array_equal(a, b)
    f = outs[0][2:]
    assert np.isfinite(f[0]).all() and outs[0][0].shape == (2 * nc,)


def test_a_grid_of_more_rows_than_a_launch_has_wavefronts_for():
    """2^26 rows of one voxel and some more: a wavefront each would pass the
    2^32 threads of a launch.  The steps equal those over the rows."""
    shape = (8193, 8192, 1)
    rng = np.random.default_rng(8)
    mask = (rng.random(shape, dtype=np.float32) < 0.3).astype(np.uint8)
    m0 = rng.random(shape)
    outs = []
    for rows in (False, True):
        with _solver(shape, mask, [m0], 1, rows) as s:
            sig = s.run(3)
            outs.append((sig, s.download_magnetization()[0]))
        print(f"[rows] {shape} rows={rows}", flush=True)
    np.testing.assert_allclose(outs[0][0], outs[1][0], rtol=1e-12)
    assert np.array_equal(outs[0][1], outs[1][1])


def _us(s, steps):
    """Device time of a step, the least of three runs."""
    ms, n, best = ctypes.c_double(), ctypes.c_int64(), 1e30
    s.run(steps)
    for _ in range(3):
        s.run(steps)
        check(s.lib.nmr_hip_last_run_ms(s.ctx, ctypes.byref(ms), ctypes.byref(n)), "nmr_hip_last_run_ms")
        best = min(best, ms.value / steps * 1e3)
    return best


# Measured, tiles over list: 0.58, 0.71, 0.71, 1.85 and 1.88.
@pytest.mark.parametrize("n,phi,nc,bc,scheme,data,at_most", [
    (200, 1.0, 1, (2, 2, 2), 0, False, 1.15), (200, 1.0, 1, (1, 1, 1), 0, False, 1.15),
    (160, 1.0, 2, (1, 1, 1), 1, True, 1.15), (160, 0.4, 2, (1, 1, 1), 0, False, 0.75),
    (160, 0.4, 1, (0, 0, 0), 0, False, 0.75)])
def test_the_automatic_sweep_is_the_faster_one(n, phi, nc, bc, scheme, data, at_most):
    """The automatic choice against the tiles: no slower where ghosts and
    per-voxel data (uploaded last) make the list dearer, and the list where it
    is faster by far."""
    shape = (n, n, n)
    mask = generators.porosity(shape, phi, 3, sigma=2.0) if phi < 1 else np.ones(shape, np.uint8)
    with _solver(shape, mask, [mask.astype(float)] * 3, nc, bc=bc, scheme=scheme) as s:
        if data:
            s.upload_coefficients(np.full(shape, D), np.full(shape, 0.5), np.full(shape, 0.4))
            s.upload_phase_weights(0.5 * mask, 0.5 * mask)
        auto = _us(s, 40)
        s.set_tile(4)
        tile = _us(s, 40)
    print(f"[choice] {n} {phi} nc {nc} bc {bc}: automatic {auto:.1f}, tiles {tile:.1f} us a step", flush=True)
    assert auto <= at_most * tile


def test_another_velocity_on_the_same_mask():
    """The list and its state stay where only the velocity changes; where that
    makes pores read solids, or none, the list is built again.  Runs between
    the uploads equal those over the rows."""
    shape, nc = (11, 13, 29), 2
    mask = generators.porosity(shape, 0.35, 9, sigma=1.0)
    rng = np.random.default_rng(10)
    nz, ny, nx = shape
    inert = [generators.velocity(mask, seed, sigma=1.0, vmax=1e-3, d=(DX,) * 3) for seed in (1, 2)]
    solid = [[rng.uniform(-1e-3, 1e-3, s) for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx))]
             for _ in range(2)]
    m0 = [rng.random(shape) - 0.3 for _ in range(nc)]  # solids hold values too
    for scheme in (0, 1):
        outs = []
        for rows in (False, True):
            with _solver(shape, mask, m0, nc, rows, velocity=True, scheme=scheme) as s:
                out = []
                for v in (inert[0], inert[1], solid[0], solid[1], inert[0]):
                    s.upload_velocity(*v)
                    out.append((s.run(6), s.download_magnetization()))
                    s.upload_velocity(*inert[1])
                    s.upload_velocity(*v)
                    out.append((s.run(5), s.signal()))
                out.append((s.run(1), s.download_magnetization()))
            outs.append(out)
        for a, b in zip(*outs):
            np.testing.assert_allclose(a[0], b[0], rtol=1e-12, atol=1e-14)
            np.testing.assert_allclose(a[1], b[1], rtol=1e-12, atol=1e-14)
        for a, b in zip(outs[0][-1][1], outs[1][-1][1]):
            np.testing.assert_array_equal(a, b)


def test_a_velocity_uploaded_again_costs_what_it_does_for_the_tiles():
    """The list stays where only the velocity changes (64^3; building it again
    took 0.56 ms, the upload for the tiles 0.32)."""
    shape = (64, 64, 64)
    mask = generators.porosity(shape, 0.3, 3, sigma=2.0)
    vel = generators.velocity(mask, 5, sigma=2.0, vmax=1e-3, d=(DX,) * 3)
    least = {-1: 1e9, 4: 1e9}
    with _solver(shape, mask, [mask.astype(float)] * 2, 2, velocity=True) as s:
        for _ in range(12):
            for tile in least:
                s.set_tile(tile)
                s.upload_velocity(*vel)
                s.run(1)
                t = time.perf_counter()
                s.upload_velocity(*vel)
                least[tile] = min(least[tile], (time.perf_counter() - t) * 1e3)
                s.run(1)
    print(f"[uploads] velocity again: list {least[-1]:.3f}, tiles {least[4]:.3f} ms", flush=True)
    assert least[-1] <= 1.3 * least[4]


class _Filled:
    """Takes the device's free memory but for `leave` bytes."""

    def __init__(self, leave):
        self.hip, self.blocks = ctypes.CDLL("libamdhip64.so"), []
        for size in (16 << 30, 1 << 30, 64 << 20, 8 << 20):
            while self.free() - leave >= size:
                p = ctypes.c_void_p()
                if self.hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) != 0:
                    self.hip.hipGetLastError()
                    break
                self.blocks.append(p)

    def free(self):
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert self.hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for p in self.blocks:
            self.hip.hipFree(p)


def test_no_memory_for_the_list_or_beside_it():
    """384^3, one component, a list of 0.45 GB with 0.23 GB to build it, tiles of
    0.45 GB.  With 0.6 GB left the upload takes the tiles, as it did before there
    was a list; with 0.25 GB beside a list, setting a tile gives the list back."""
    shape = (384, 384, 384)
    rng = np.random.default_rng(12)
    mask = (rng.random(shape, dtype=np.float32) < 0.3).astype(np.uint8)
    m0 = rng.random(shape)
    with _solver(shape, mask, [m0], 1, True) as s:
        want = s.run(2), s.download_magnetization()[0]
    with _solver(shape, mask, [m0], 1) as s:  # (every kernel of either way is loaded)
        s.run(2)
        s.set_tile(4)
        s.run(2)
    with HipSolver(shape, 1, DX, DT, D, 0.5, r1_bulk=0.4, rho1=4e-6, rho2=9e-6) as s:
        s.upload_mask(mask)
        with _Filled(600 << 20) as full:
            print(f"[memory] {full.free() >> 20} MiB left before the upload", flush=True)
            s.upload_magnetization(m0)
            got = s.run(2), s.download_magnetization()[0]
            print(f"[memory] {full.free() >> 20} MiB left", flush=True)
    np.testing.assert_allclose(got[0], want[0], rtol=1e-12)
    assert np.array_equal(got[1], want[1])
    with _solver(shape, mask, [m0], 1) as s:
        held = s.device_bytes()
        first = s.run(1)
        with _Filled(250 << 20) as full:
            print(f"[memory] {full.free() >> 20} MiB left beside the list", flush=True)
            s.set_tile(4)
            got = np.concatenate([first, s.run(1)[1:]]), s.download_magnetization()[0]
            s.set_tile(-1)  # and back: no memory to build the list again, or what the tiles leave
            s.run(1)
        assert s.device_bytes() < 1.5 * held
    np.testing.assert_allclose(got[0], want[0], rtol=1e-12)
    assert np.array_equal(got[1], want[1])


def test_the_autotuner_does_not_take_another_batchs_choice_of_the_list():
    """Three 96^3 instances whose list cannot be had (a solid that is not
    finite) are tuned first; then others of the same shapes, a fifth of them
    pores, for which the list takes less than half the tile's time.  Which of
    them a run takes shows in the order of the signal's FP64 sums (of values over
    16 decades: those of FP32 values of one size are exact in any order)."""
    shape = (96, 96, 96)
    size = 10.0 ** -(np.arange(96) / 6.0)[:, None, None]
    masks = [generators.porosity(shape, 0.2, seed, sigma=2.0) for seed in range(3)]

    def batch(bad=False):
        b = BatchSolver([dict(shape=shape)] * 3, 2, DX, DT, D, 0.5, r1_bulk=0.4)
        for i, m in enumerate(masks):
            rng = np.random.default_rng(i)
            m0 = [rng.random(shape) * size, (rng.random(shape) - 0.5) * size]
            if bad and i == 1:
                m0[0][tuple(np.argwhere(m == 0)[5])] = np.nan
            b.upload(i, m, m0)
        return b

    def run(b):
        out = b.run(20)
        b.close()
        return out

    first = batch(True)
    first.autotune(3)
    first.close()
    tuned = batch()
    variant, lz, persistent = tuned.autotune(3)
    tuned = run(tuned)
    on_list = run(batch())
    on_tile = batch()
    on_tile.set_tile(variant, lz, persistent=persistent)
    on_tile = run(on_tile)
    assert not np.array_equal(on_list, on_tile)  # (else the next line shows nothing)
    np.testing.assert_array_equal(tuned, on_list)


@pytest.mark.parametrize("scheme", ["fits", "grows", "empty", "solid flow", "not finite"])
def test_an_instance_uploaded_again_keeps_the_others_in_the_list(scheme):
    """Between runs one instance gets another state, mask and velocity: one that
    fits its place in the list, one that does not, one without pores, one whose
    pores read solids, one with a solid that is not finite; then the first again.
    The fields equal those of a batch on a tile, bit for bit."""
    rng = np.random.default_rng(13)
    shapes = [(9, 14, 30), (12, 7, 41), (6, 6, 6)]
    masks = [generators.porosity(s, 0.3, k, sigma=1.0) for k, s in enumerate(shapes)]

    def state(k, mask):
        return [rng.random(shapes[k]), rng.random(shapes[k]) - 0.5]

    def flow(k, mask, everywhere=False):
        nz, ny, nx = shapes[k]
        if everywhere:
            return [rng.uniform(-1e-3, 1e-3, s) for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx))]
        return generators.velocity(mask, 3 + k, sigma=1.0, vmax=1e-3, d=(DX,) * 3)

    first = [(m, state(k, m), flow(k, m)) for k, m in enumerate(masks)]
    other = generators.porosity(shapes[1], {"fits": 0.29, "grows": 0.6}.get(scheme, 0.3), 7, sigma=1.0)
    if scheme == "empty":
        other[:] = 0
    again = (other, state(1, other), flow(1, other, scheme == "solid flow"))
    if scheme == "not finite":
        again[1][0][tuple(np.argwhere(other == 0)[3])] = np.nan
    outs = []
    for variant in (-1, 4):
        b = BatchSolver([dict(shape=s, grad_amp=0.1, delta=3 * DT, big_delta=6 * DT) for s in shapes], 2, DX, DT, D, 0.5,
                        r1_bulk=0.4, velocity=True, precession=True)
        b.set_tile(variant)
        out = []
        for k, (m, m0, v) in enumerate(first):
            b.upload(k, m, m0, v)
        out.append([b.run(5)])
        for m, m0, v in (again, first[1], again):
            b.upload(1, m, m0, v)
            out.append([b.run(4)] + (b.download(1) if scheme == "grows" else []))
            out.append([b.run(3)] + sum((b.download(k) for k in range(3)), []))
        outs.append(out)
        b.close()
    for x, y in zip(*outs):
        np.testing.assert_allclose(x[0], y[0], rtol=1e-11, atol=1e-12)
        for p, q in zip(x[1:], y[1:]):
            np.testing.assert_array_equal(p, q)


def test_an_instance_uploaded_again_costs_little_more_than_for_the_tiles():
    """24 instances of edge 32-128; one is uploaded again and the batch steps
    twice: 2.0 ms on the tiles (measured before: 3.3 on the list, which was built
    again from all instances)."""
    g = np.random.default_rng(1)
    specs = []
    for i in range(24):
        shape = tuple(int(v) for v in g.integers(32, 129, 3))
        m = generators.porosity(shape, 0.25, i, sigma=2.0)
        specs.append(dict(shape=shape, mask=m, m0=[m.astype(float), np.zeros(shape)],
                          vel=generators.velocity(m, i, sigma=2.0, vmax=1e-3, d=(DX,) * 3)))
    least = {}
    for tile in (-1, 4):
        b = BatchSolver(specs, 2, DX, DT, D, 0.5, velocity=True)
        b.set_tile(tile)
        for i, s in enumerate(specs):
            b.upload(i, s["mask"], s["m0"], s["vel"])
        b.run(2)
        for _ in range(8):
            t = time.perf_counter()
            b.upload(3, specs[3]["mask"], specs[3]["m0"], specs[3]["vel"])
            b.run(2)
            least[tile] = min(least.get(tile, 1e9), (time.perf_counter() - t) * 1e3)
        b.close()
    print(f"[uploads] an instance again and two steps: list {least[-1]:.2f}, tiles {least[4]:.2f} ms", flush=True)
    assert least[-1] <= 1.3 * least[4]


@pytest.mark.parametrize("bc", [(0, 0, 0), (1, 1, 1), (2, 2, 2), (0, 1, 2), (2, 0, 1), (1, 2, 0)])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 5, 2), (4, 1, 9), (7, 6, 64)])
def test_padded_download_is_the_interior_with_its_ghosts(shape, bc):
    """After a step the padded layout holds the compact one and, a cell further,
    what each axis's rule puts there: the cell beside, the opposite one, 0."""
    rng = np.random.default_rng(14)
    mask = (rng.random(shape) < 0.6).astype(np.uint8)
    mask.flat[0] = 1
    m0 = [rng.random(shape) for _ in range(3)]
    with _solver(shape, mask, m0, 3, bc=bc) as s:
        s.run(1)
        inside, padded = s.download_magnetization(), s.download_magnetization(layout=1)
    for a, b in zip(inside, padded):
        want = a
        for axis in (2, 1, 0):
            width = [(0, 0)] * 3
            width[axis] = (1, 1)
            want = np.pad(want, width, mode={0: "edge", 1: "wrap", 2: "constant"}[bc[2 - axis]])
        np.testing.assert_array_equal(b, want)
