"""The learned corrector on the GPU: the BF16 MFMA convolution kernels
(forward, input gradient, weight gradient) against the FP64 restatement
with BF16 rounding emulated (oracle/corrector.py) and against the torch
fixture; training on batched-solver samples (loss decreases, bitwise
repeatable); the learned solve's residual check and plain fallback; and
what the trained net gains over the coarse step without it."""
import os

import numpy as np
import pytest

from oracle import corrector as oc
from initializator_amd import generators
from initializator_amd.solver import BatchSolver, Corrector, HipSolver

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


def rel_l2(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


@pytest.fixture(scope="module")
def fix():
    return dict(np.load(os.path.join(HERE, "golden", "corrector_fixture.npz")))


@pytest.mark.parametrize("shape,seed", [((7, 9, 10), 0), ((13, 11, 37), 1), ((3, 4, 5), 2), ((6, 2, 70), 3)])
def test_forward_against_emulating_oracle(shape, seed):
    rng = np.random.default_rng(seed)
    params = oc.random_params(seed)
    feats = rng.normal(0.0, 1.0, shape + (6,))
    with Corrector() as net:
        net.params = params.astype(np.float32)
        got = net.forward(feats)
    want = oc.forward(params.astype(np.float32), feats.astype(np.float32), emulate=True)
    e = rel_l2(got, want)
    print(f"[corrector] forward {shape}: relL2 vs emulating oracle {e:.2e}", flush=True)
    assert e < 1e-3


def test_forward_and_backward_against_torch_fixture(fix):
    with Corrector() as net:
        net.params = fix["params"].astype(np.float32)
        out = net.forward(fix["features"])
        g = net.backward(fix["features"], fix["grad_out"])
    e_out, e_g = rel_l2(out, fix["out"]), rel_l2(g, fix["grad_params"])
    p32 = fix["params"].astype(np.float32)
    g_emul = oc.backward(p32, fix["features"].astype(np.float32), fix["grad_out"].astype(np.float32))
    e_emul = rel_l2(g, g_emul)
    print(f"[corrector] vs torch FP64: output relL2 {e_out:.2e}, gradient relL2 {e_g:.2e}; "
          f"gradient vs BF16-emulating oracle {e_emul:.2e}", flush=True)
    # BF16 storage of weights, activations and propagated gradients moves the
    # result off exact FP64 by the amount the emulating oracle shows (~5e-2
    # for this fixture's gradient); against that oracle the kernels agree closely
    assert e_out < 2e-2 and e_g < 0.1 and e_emul < 1e-3


@pytest.mark.parametrize("shape,seed", [((7, 9, 10), 4), ((9, 6, 41), 5)])
def test_backward_against_emulating_oracle(shape, seed):
    rng = np.random.default_rng(seed)
    params = oc.random_params(seed).astype(np.float32)
    feats = rng.normal(0.0, 1.0, shape + (6,)).astype(np.float32)
    gout = rng.normal(0.0, 1.0, shape + (2,)).astype(np.float32)
    with Corrector() as net:
        net.params = params
        got = net.backward(feats, gout)
    want = oc.backward(params, feats, gout, emulate=True)
    for name, lo, hi in [("W1", 0, 2592), ("b1", 2592, 2608), ("W2", 2608, 9520), ("b2", 9520, 9536),
                         ("W3", 9536, 10400), ("b3", 10400, 10402)]:
        e = rel_l2(got[lo:hi], want[lo:hi])
        print(f"[corrector] backward {shape} {name}: relL2 {e:.2e}", flush=True)
        assert e < 5e-3, name


@pytest.mark.parametrize("shape,seed", [((7, 9, 10), 10), ((13, 11, 37), 11), ((3, 4, 5), 12), ((6, 2, 70), 13),
                                        ((35, 19, 17), 14), ((20, 33, 48), 15)])
def test_convolution_kernels_give_the_same_bits(shape, seed):
    """z-marching columns (several column heights, including one plane and
    more planes than the grid), staged tiles and row gathers feed the same
    MFMA operands in the same order: forward outputs and parameter gradients
    agree bit for bit."""
    rng = np.random.default_rng(seed)
    params = oc.random_params(seed).astype(np.float32)
    feats = rng.normal(0.0, 1.0, shape + (6,)).astype(np.float32)
    gout = rng.normal(0.0, 1.0, shape + (2,)).astype(np.float32)
    res = {}
    with Corrector() as net:
        net.params = params
        for kind, zc in [(0, 0), (0, 1), (0, 3), (0, 64), (1, 0), (2, 0), (3, 5)]:
            net.set_conv(kind, zc)
            res[(kind, zc)] = (net.forward(feats), net.backward(feats, gout))
    ref_out, ref_g = res[(2, 0)]
    assert np.all(np.isfinite(ref_out)) and np.all(np.isfinite(ref_g))
    for k, (o, g) in res.items():
        np.testing.assert_array_equal(o, ref_out, err_msg=str(k))
        np.testing.assert_array_equal(g, ref_g, err_msg=str(k))


def test_convolution_kernel_choice_is_checked():
    from initializator_amd._lib import NmrError
    with Corrector() as net:
        for kind, zc in [(4, 0), (-1, 0), (0, -1), (0, 5000)]:
            with pytest.raises(NmrError):
                net.set_conv(kind, zc)
        net.set_conv(0, 0)


DX, D = 1e-6, 2.3e-9
DT = generators.stable_dt(DX, D)


def _instances(n, seed0=100):
    out = []
    for i in range(n):
        r = np.random.default_rng(seed0 + i)
        shp = tuple(int(v) for v in r.integers(18, 34, 3))
        phi = float(r.uniform(0.2, 0.4))
        mask = generators.porosity(shp, phi, seed0 + i, sigma=2.0)
        vel = generators.velocity(mask, seed0 + i, sigma=2.0, vmax=1e-3, d=(DX, DX, DX))
        out.append(dict(shape=shp, mask=mask, vel=vel, rho1=float(r.uniform(1e-6, 50e-6)),
                        grad_amp=float(r.uniform(0.0, 0.3)), delta=2e-3, big_delta=4e-3))
    for s in out:
        s["rho2"] = s["rho1"]
    return out


def _batch(specs):
    b = BatchSolver(specs, 2, DX, DT, D, 0.5, r1_bulk=1 / 2.5e10, velocity=True, precession=True, phase_exact=True)
    for i, s in enumerate(specs):
        b.upload(i, s["mask"], [s["mask"].astype(np.float64), np.zeros(s["shape"])], s["vel"])
    return b


def _train(seed=7, rounds=24, ninst=6):
    specs = _instances(ninst)
    with _batch(specs) as b:
        net = Corrector(seed)
        losses = net.train(b, factor=8, rounds=rounds, stride=8, lr=2e-3)
    return net, losses


def test_training_reduces_loss_and_repeats_bitwise():
    net, losses = _train()
    first, last = losses[:4].mean(), losses[-4:].mean()
    print(f"[corrector] training loss {first:.3e} -> {last:.3e}", flush=True)
    assert np.all(np.isfinite(losses)) and last < 0.5 * first
    net2, losses2 = _train()
    assert np.array_equal(net.params, net2.params)
    assert np.array_equal(losses, losses2)
    net.close()
    net2.close()


def _solver(case_seed=900, shape=(30, 28, 32)):
    mask = generators.porosity(shape, 0.3, case_seed, sigma=2.0)
    vel = generators.velocity(mask, case_seed, sigma=2.0, vmax=1e-3, d=(DX, DX, DX))
    s = HipSolver(shape, 2, DX, DT, D, 0.5, r1_bulk=1 / 2.5e10, rho1=20e-6, rho2=20e-6, velocity=True,
                  precession=True, phase_exact=True)
    s.upload_mask(mask)
    s.upload_velocity(*vel)
    s.upload_magnetization(mask.astype(np.float64), np.zeros(shape))
    return s, mask, vel


def _plain_signal(nsteps, sched, factor):
    s, _, _ = _solver()
    sig = s.run(nsteps, sched)
    f = s.download_magnetization()
    s.close()
    return sig[::factor], f


def test_fallback_reproduces_the_plain_solve():
    """A corrector whose output is NaN fails every residual check; every
    coarse step is redone as plain steps and the result is the plain
    solve's (fields bit for bit)."""
    ncoarse, factor = 6, 8
    sched = generators.pgse_schedule(ncoarse * factor, DT, 0.2, 2e-4, 6e-4)
    want_sig, want_f = _plain_signal(ncoarse * factor, sched, factor)
    with Corrector(1) as net:
        p = net.params
        p[-1] = np.nan
        net.params = p
        net.set_scales(1e-3, 1e-3)
        s, _, _ = _solver()
        sig, nf = net.run_learned(s, ncoarse, factor, sched, tol=1e-3, reasons=True)
        f = s.download_magnetization()
        s.close()
    assert nf == (ncoarse, ncoarse, 0, 0)
    # fields bit for bit; the signal sums are the same values summed in another order
    for a, b in zip(f, want_f):
        np.testing.assert_array_equal(a, b)
    np.testing.assert_allclose(sig, want_sig, rtol=1e-12, atol=1e-12 * np.abs(want_sig).max())


def test_learned_solve_same_bits_for_every_convolution_kernel():
    """The learned solve with the last layer on every row (z-marching) or on
    the rows that hold a pore only (tiles, z-marching sparse): corrections
    are read at pores only, so fields and signals are the same bits."""
    ncoarse, factor = 4, 8
    sched = generators.pgse_schedule(ncoarse * factor, DT, 0.2, 2e-4, 6e-4)
    out = {}
    with Corrector(5) as net:
        net.set_scales(1e-3, 1e-4)
        for kind in (0, 1, 3):
            net.set_conv(kind)
            s, _, _ = _solver()
            sig, nf = net.run_learned(s, ncoarse, factor, sched, tol=1e30, reasons=True)
            out[kind] = (sig, nf, s.download_magnetization())
            s.close()
    sig0, nf0, f0 = out[0]
    assert nf0[0] < ncoarse and np.all(np.isfinite(sig0))
    for kind, (sig, nf, f) in out.items():
        assert nf == nf0, kind
        np.testing.assert_array_equal(sig, sig0, err_msg=str(kind))
        for a, b in zip(f, f0):
            np.testing.assert_array_equal(a, b, err_msg=str(kind))


def test_oversized_corrections_fall_back():
    """A correction larger than tol times the field (output bias 1000 in
    units of out_scale 1) fails the size check on every step."""
    ncoarse, factor = 3, 8
    with Corrector(2) as net:
        p = net.params
        p[10400:] = 1000.0
        net.params = p
        net.set_scales(1e-3, 1.0)
        s, _, _ = _solver()
        _, why = net.run_learned(s, ncoarse, factor, None, tol=1e-3, reasons=True)
        s.close()
    assert why == (ncoarse, 0, 0, ncoarse)


def test_trained_corrector_gains_over_the_coarse_step_alone():
    """On a held-out porous case: the trained net keeps the learned solve's
    signal close to the plain solve; the coarse step alone (a net whose
    output is zero, every step accepted) drifts far more or blows up."""
    net, _ = _train(rounds=32)
    ncoarse, factor = 24, 8
    sched = generators.pgse_schedule(ncoarse * factor, DT, 0.2, 1e-3, 3e-3)
    want, _ = _plain_signal(ncoarse * factor, sched, factor)
    s, _, _ = _solver()
    sig, nf = net.run_learned(s, ncoarse, factor, sched, tol=1e-2)
    s.close()
    e_learn = rel_l2(sig, want)
    zero = Corrector(3)
    p = zero.params
    p[9536:] = 0.0
    zero.params = p
    zero.set_scales(*net.scales())
    s, _, _ = _solver()
    sig0, nf0 = zero.run_learned(s, ncoarse, factor, sched, tol=1e30)
    s.close()
    e_coarse = rel_l2(sig0, want) if np.all(np.isfinite(sig0)) else np.inf
    print(f"[corrector] held-out 30x28x32, {ncoarse} coarse steps of 8: learned relL2 {e_learn:.2e} "
          f"({nf} fallbacks), coarse step alone relL2 {e_coarse:.2e} ({nf0} fallbacks)", flush=True)
    assert e_learn < 1e-2
    assert e_coarse > 3 * e_learn
    net.close()
    zero.close()


def test_matrix_core_rate_is_measured():
    """nmr_hip_mfma_rate times the convolutions' MFMA instruction on
    register operands: a positive rate no higher than the dense BF16 peak
    (2.5 PFLOP/s, with 10 % for clock boost)."""
    import ctypes

    from initializator_amd import _lib

    lib = _lib.load()
    tf = ctypes.c_double()
    assert lib.nmr_hip_mfma_rate(256, 2, ctypes.byref(tf)) == 0, lib.nmr_hip_last_error().decode()
    print(f"[mfma] {tf.value:.0f} TFLOP/s dense BF16 (v_mfma_f32_16x16x32_bf16)", flush=True)
    assert 0.0 < tf.value <= 2750.0


@pytest.mark.parametrize("kind", ["smooth", "ragged", "one", "none", "read solids", "trim"])
def test_learned_solve_on_the_list_of_pores_equals_the_rows(kind):
    """The learned solve steps on the list of the pores where a run would, on
    the row buffers otherwise: the same operations on the same values, so the
    fields agree bit for bit and the signal to the order of its FP64 sums.
    Some steps are accepted and some redone (a bound on the corrections that
    splits them), on grids off every tile's edge, with one pore and none, with
    solids that pores read, and with a trimmed signal window."""
    shape = {"ragged": (7, 19, 37), "one": (3, 4, 5), "none": (3, 4, 5)}.get(kind, (20, 18, 33))
    if kind in ("one", "none"):
        mask = np.zeros(shape, np.uint8)
        mask[1, 2, 3] = kind == "one"
    else:
        mask = generators.porosity(shape, 0.3, 31, sigma=1.5)
    vel = generators.velocity(mask, 32, sigma=1.5, vmax=1e-3, d=(DX, DX, DX))
    if kind == "read solids":
        vel = generators.velocity(np.ones(shape, np.uint8), 33, sigma=1.5, vmax=1e-3, d=(DX, DX, DX))
    rng = np.random.default_rng(34)
    m0 = [rng.normal(0.5, 0.2, shape), rng.normal(0.0, 0.2, shape)]
    if kind != "read solids":
        m0 = [m * mask for m in m0]
    ncoarse, factor = 6, 4
    sched = generators.pgse_schedule(ncoarse * factor, DT, 0.2, 2e-4, 4e-4)
    out = {}
    with Corrector(8) as net:
        net.set_scales(1e-3, 1e-3)
        for rows in (False, True):
            for tol in (1e30, 4e-4):
                with HipSolver(shape, 2, DX, DT, D, 0.5, r1_bulk=1 / 2.5e10, rho1=20e-6, rho2=20e-6, velocity=True,
                               precession=True, phase_exact=True, buffer=(1, 2, 0) if kind == "trim" else (0, 0, 0)) as s:
                    s.set_layout(not rows)
                    s.upload_mask(mask)
                    s.upload_velocity(*vel)
                    s.upload_magnetization(*m0)
                    a, na = net.run_learned(s, ncoarse, factor, sched, tol=tol, reasons=True)
                    b = s.run(3)  # a run continues from where the learned solve left off
                    c, nb = net.run_learned(s, 2, factor, None, tol=tol, reasons=True)
                    out[rows, tol] = (np.concatenate([a, b, c]), na + nb, s.download_magnetization())
    for tol in (1e30, 4e-4):
        (sig, nf, f), (sig_r, nf_r, f_r) = out[False, tol], out[True, tol]
        print(f"[learned] {kind} tol {tol:g}: {nf}", flush=True)
        assert nf == nf_r
        for a, b in zip(f, f_r):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_allclose(sig, sig_r, rtol=1e-12, atol=1e-12 * max(1e-30, np.abs(sig_r).max()))


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 31), (3, 2, 32), (2, 2, 33), (5, 4, 63), (1, 7, 65), (9, 40, 96),
                                   (33, 17, 34)])
def test_weight_gradient_at_the_edges_of_segments(shape):
    """The weight gradient runs over x segments of 32 voxels, 512 partials of
    them: rows that end on a segment's edge and next to it, fewer segments than
    partials and more, against the convolution gradients in FP64 of the BF16
    tensors (exact inputs, positive weights and activations, so that only the
    FP32 sums round).  Then another grid on the same net and back: what one
    leaves in the halo is not seen by the other."""
    rng = np.random.default_rng(list(shape))
    p = np.zeros(10402, np.float32)
    for c in range(6):  # layer 1: channel c hands on feature c; layer 2: the same; layer 3: sums of them
        p[(c * 6 + c) * 27 + 13] = 1.0
        p[2608 + (c * 16 + c) * 27 + 13] = 1.0
        p[9536 + c * 27 + 13], p[9536 + (16 + c) * 27 + 13] = 1.0, 0.5
    f = rng.integers(1, 64, shape + (6,)).astype(np.float32)
    g = rng.integers(-8, 9, shape + (2,)).astype(np.float32)

    def taps(x, y):  # dW[t] = sum_v x[v + off(t)] y[v]
        q = np.pad(x.astype(np.float64), 1)
        nz, ny, nx = y.shape
        return np.array([(q[k // 9:k // 9 + nz, k // 3 % 3:k // 3 % 3 + ny, k % 3:k % 3 + nx] * y).sum() for k in range(27)])

    with Corrector() as net:
        net.params = p
        got = net.backward(f, g)
        net.backward(rng.random((4, 5, 6, 6)).astype(np.float32), np.ones((4, 5, 6, 2), np.float32))
        again = net.backward(f, g)
    np.testing.assert_array_equal(got, again)
    back = g[..., 0].astype(np.float64) + 0.5 * g[..., 1]  # exact in BF16: the gradient at channels 0..5 of layers 2 and 1
    scale = 64.0 * 12.0 * np.prod(shape)
    for c in range(6):
        for o in range(2):
            e = np.abs(got[9536 + (16 * o + c) * 27:][:27] - taps(f[..., c], g[..., o].astype(np.float64)))
            assert e.max() <= 2.0 ** -22 * scale, (c, o)
        e = np.abs(got[2608 + (16 * 2 + c) * 27:][:27] - taps(f[..., c], back))
        assert e.max() <= 2.0 ** -22 * scale, c
        e = np.abs(got[(6 * 3 + c) * 27:][:27] - taps(f[..., c], back))
        assert e.max() <= 2.0 ** -22 * scale, c
    np.testing.assert_allclose(got[10400:], g.reshape(-1, 2).sum(0), atol=2.0 ** -22 * scale)


def test_training_gives_the_same_net_whatever_the_batch_steps_on():
    """The batch steps on the list of the pores, on a tile in bricks or in rows
    while it trains: the same samples, so the same losses and parameters, and
    the same state left behind."""
    specs, out = _instances(4), []
    for layout, variant in ((True, -1), (True, 4), (False, -1)):
        with _batch(specs) as b, Corrector(3) as net:
            b.set_layout(layout)
            b.set_tile(variant)
            losses = net.train(b, factor=4, rounds=3, stride=3)
            out.append([losses, net.params] + sum((b.download(i) for i in range(4)), []) + [b.run(2)])
    for o in out[1:]:
        for x, y in zip(o[:-1], out[0][:-1]):
            np.testing.assert_array_equal(x, y)
        np.testing.assert_allclose(o[-1], out[0][-1], rtol=1e-11, atol=1e-12)
