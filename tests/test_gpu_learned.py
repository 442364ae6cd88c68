"""GPU checks of the learned correction: BF16 MFMA forward and gradients
against the CPU oracle (same bf16 rounding points, FP64 sums), the band ->
tile gather bit for bit, training on a learnable task, and the true-residual
fallback of the correction inside the solve."""
import numpy as np
import pytest

from solve_helpers import band_problem
from test_oracle_net import random_params

pytestmark = pytest.mark.gpu


def bf16_bits(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def bits_f32(u):
    return (np.asarray(u, np.uint16).astype(np.uint32) << 16).view(np.float32)


def net_for(pkg, hip, params, out_scale=1.0):
    return pkg.CorrectorNet(hip, params, out_scale)


@pytest.mark.parametrize("n", [1, 5])
def test_forward_matches_oracle(pkg, orc, hip, n):
    rng = np.random.default_rng(n)
    p = random_params(rng)
    bits = bf16_bits(rng.normal(size=(n, 20, 20, 20, 2)))
    net = net_for(pkg, hip, p)
    y = net.forward(hip.to_device(bits), n).get()
    want = np.zeros(n * 4096, np.float32)
    orc.orc_net_forward(p, bits_f32(bits).ravel(), n, 1, want)
    want = want.reshape(n, 4096)
    err = np.abs(y - want)
    # FP32 (MFMA) vs FP64 sums flip a bf16 rounding of a hidden activation now and then
    assert err.max() <= 1e-2 * np.abs(want).max(), err.max()
    assert np.linalg.norm(y - want) <= 2e-3 * np.linalg.norm(want)


def test_loss_and_gradient_match_oracle(pkg, orc, hip):
    rng = np.random.default_rng(7)
    n = 3
    p = random_params(rng)
    bits = bf16_bits(rng.normal(size=(n, 20, 20, 20, 2)))
    tgt = rng.normal(size=(n, 4096)).astype(np.float32)
    net = net_for(pkg, hip, p)
    loss, g = net.loss_grad(hip.to_device(bits), hip.to_device(tgt), n)
    go = np.zeros(p.size)
    lo = orc.orc_net_loss_grad(p, bits_f32(bits).ravel(), tgt.ravel(), n, 1, go)
    assert loss == pytest.approx(lo, rel=1e-4)
    for l in range(4):
        a, b = g[l * 6928:(l + 1) * 6928], go[l * 6928:(l + 1) * 6928]
        assert np.linalg.norm(a - b) <= 2e-2 * np.linalg.norm(b), (l, np.linalg.norm(a - b) / np.linalg.norm(b))
    # padding stays without gradient
    assert np.all(g[:6912].reshape(27, 16, 16)[:, 2:, :] == 0)
    assert np.all(g[3 * 6928: 3 * 6928 + 6912].reshape(27, 16, 16)[:, :, 1:] == 0)


def test_training_learns_a_box_filter(pkg, hip):
    """Target = the 3^3 mean of input channel 0 around each output cell: the
    loss falls well below its starting value within 300 Adam steps."""
    rng = np.random.default_rng(3)
    n = 128
    x = rng.normal(size=(n, 20, 20, 20, 2)).astype(np.float32)
    bits = bf16_bits(x)
    xf = bits_f32(bits)[..., 0]
    box = np.zeros((n, 16, 16, 16), np.float32)
    for dz in range(3):
        for dy in range(3):
            for dx in range(3):
                box += xf[:, 1 + dz:17 + dz, 1 + dy:17 + dy, 1 + dx:17 + dx]
    box /= 27.0
    from msbg_rs_amd.learned import init_params
    net = net_for(pkg, hip, init_params(0))
    losses = net.train(hip.to_device(bits), hip.to_device(box.reshape(n, 4096)), n, steps=300, batch=16, lr=3e-3,
                       seed=1)
    assert np.all(np.isfinite(losses))
    assert losses[-20:].mean() < 0.2 * losses[:5].mean(), (losses[:5], losses[-20:])


def test_net_input_bitexact(pkg, orc, hip):
    g, active, x, b = band_problem(pkg, 40, 33, 48, 9)
    phi = pkg.SparseGrid("phi", 40, 33, 48, -1.0, 1.0)
    rng = np.random.default_rng(9)
    phi.ensure_blocks_parallel(np.nonzero(rng.random(phi.n_blocks) < 0.6)[0])
    phi._slab[2:phi.n_slots] = rng.uniform(-1, 1, size=(phi.n_slots - 2, 4096)).astype(np.float32)
    layout = pkg.DeviceGrid.from_host(g, lib=hip)
    band = pkg.PoissonBand(layout, active, lib=hip)
    dphi = pkg.DeviceGrid.from_host(phi, lib=hip)
    r = np.ascontiguousarray(x)
    got = band.net_input(dphi, hip.to_device(r), 0.37).get()
    want = np.zeros(active.size * 16000, np.uint16)
    orc.orc_net_input(g.sx, g.sy, g.sz, g.b2s, active, active.size, r.ravel(), 0.37,
                      np.ascontiguousarray(phi.slab).ravel(), phi.b2s, want)
    assert np.array_equal(got.ravel(), want)


def shell_band(pkg, hip):
    from msbg_rs_amd import scenes
    g, bids, _ = scenes.shell_scene()
    layout = pkg.DeviceGrid.from_host(g, lib=hip)
    band = pkg.PoissonBand(layout, bids, lib=hip)
    b = scenes.poisson_rhs(g, bids)
    return g, bids, layout, band, b


def test_correction_is_judged_by_the_true_residual(pkg, hip):
    g, bids, phi, band, b = shell_band(pkg, hip)
    db = hip.to_device(b)
    rng = np.random.default_rng(4)
    outcomes = set()
    for trial in range(4):
        x = band.field(0)
        for _ in range(8 + 8 * trial):
            band.rbgs(0, x, db, 0, 1.9)
            band.rbgs(0, x, db, 1, 1.9)
        before = x.get()
        net = net_for(pkg, hip, random_params(rng, scale=0.5 if trial % 2 else 0.05), out_scale=1.0)
        r2b, r2a, acc = band.learned_correct(net, phi, x, db)
        after = x.get()
        r2, _ = band.residual(0, x, db)
        assert r2 == r2a
        if acc:
            assert r2a < r2b and not np.array_equal(after, before)
        else:
            assert r2a == r2b and np.array_equal(after.view(np.uint32), before.view(np.uint32))
        outcomes.add(acc)
    assert True in outcomes  # the line search makes an untrained direction useful at least once


def test_solve_with_correction_converges(pkg, hip):
    g, bids, phi, band, b = shell_band(pkg, hip)
    db = hip.to_device(b)
    net = net_for(pkg, hip, random_params(np.random.default_rng(5), scale=0.3))
    for storage, refine in ((0, False), (1, True), (2, True)):
        x = band.field(0)
        st = band.solve(x, db, storage=storage, refine=refine, omega=1.9, sweeps_per_check=4, max_sweeps=3000,
                        tol=1e-6, learned=net, phi=phi)
        assert st["converged"] and st["rel_residual"] <= 1e-6, st
        assert st["corrections"] > 0 and 0 <= st["accepted"] <= st["corrections"]
        r2, b2 = band.residual(0, x, db)
        assert np.sqrt(r2 / b2) <= 1e-6


def test_trained_corrector_gain_on_unseen_shell(pkg, hip):
    """The committed network (trained on noisy-sphere bands, never on this
    shell) against the same solve without it: fewer red-black sweeps to
    ||r|| / ||b|| <= 1e-6, in FP32 and in BF16 refinement, and every accepted
    correction lowered the true residual (the solve would not converge
    otherwise)."""
    from msbg_rs_amd.learned import WEIGHTS
    g, bids, phi, band, b = shell_band(pkg, hip)
    db = hip.to_device(b)
    net = pkg.CorrectorNet.load(WEIGHTS, lib=hip)
    for storage, refine in ((0, False), (2, True)):
        res = {}
        for learned in (False, True):
            x = band.field(0)
            res[learned] = band.solve(x, db, storage=storage, refine=refine, omega=1.9, sweeps_per_check=4,
                                      max_sweeps=5000, tol=1e-6, learned=net if learned else None,
                                      phi=phi if learned else None)
            assert res[learned]["converged"]
        assert res[True]["accepted"] > 0
        assert res[True]["sweeps"] < res[False]["sweeps"], (storage, res)


@pytest.mark.parametrize("n", [1, 33, 50, 64])
def test_gradient_of_a_repeated_batch(pkg, hip, n):
    """A batch given twice has the gradient of the batch (below, at and past
    the 64 tile groups of the weight-gradient kernels; the loss factor 1 / n
    halves exactly).  The two differ by the order of FP32 sums of products of
    one sign pattern: at most ~1e5 terms a weight, whose rounding walk is below
    sqrt(1e5) 2^-24 = 2e-5 of their root sum of squares, taken norm-wise with
    the cancellation of a trained-from-noise gradient (factor 5)."""
    rng = np.random.default_rng(n)
    x = bf16_bits(rng.normal(size=(n, 20, 20, 20, 2)).astype(np.float32))
    tgt = rng.normal(size=(n, 4096)).astype(np.float32)
    from msbg_rs_amd.learned import init_params
    net = net_for(pkg, hip, init_params(n))
    l1, g1 = net.loss_grad(hip.to_device(x), hip.to_device(tgt), n)
    l2, g2 = net.loss_grad(hip.to_device(np.concatenate([x, x])), hip.to_device(np.concatenate([tgt, tgt])), 2 * n)
    assert l2 == pytest.approx(l1, rel=1e-12)
    for l in range(4):
        a, b = g1[l * 6928:(l + 1) * 6928], g2[l * 6928:(l + 1) * 6928]
        assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(a), (l, np.linalg.norm(a - b) / np.linalg.norm(a))


@pytest.mark.parametrize("n", [513, 1030])
def test_forward_in_chunks(pkg, hip, n):
    """More tiles than one pass takes: every tile has the bits of a call of its
    own, wherever in the batch it lies, with +-inf and NaN inputs in their tiles only."""
    rng = np.random.default_rng(n)
    p = random_params(rng)
    five = bf16_bits(rng.normal(size=(5, 20, 20, 20, 2)))
    five[3, 10, 10, 10, 0] = 0x7F80  # +inf
    five[4, 3, 17, 9, 1] = 0x7FC0    # NaN
    net = net_for(pkg, hip, p)
    alone = np.concatenate([net.forward(hip.to_device(np.ascontiguousarray(t[None])), 1).get().reshape(1, 4096)
                            for t in five])
    which = rng.integers(0, 5, n)
    got = net.forward(hip.to_device(np.ascontiguousarray(five[which])), n).get().reshape(n, 4096)
    assert np.all(np.isfinite(alone[:3]))  # (the hidden layers' ReLU takes a NaN to 0)
    assert np.array_equal(got.view(np.uint32), alone[which].view(np.uint32))
