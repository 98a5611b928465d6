"""Learned closure kernels on the GPU against the CPU oracle
(oracle/closure_oracle.py, FP64 with bf16 rounding where the GPU stores
bf16), and the fine <-> coarse plumbing against numpy and the step oracle.

Tolerances: the GPU accumulates in FP32 in a different order and rounds
activations and gradients to bf16 (8-bit significand), so outputs and
gradients agree to a relative L2 error of a few 1e-3; the tests allow
1e-2 (forward) and 3e-2 (gradients)."""
from __future__ import annotations

import ctypes as C
import math
from dataclasses import replace

import numpy as np
import pytest

import oracle
import oracle.closure_oracle as co
from helpers import assert_bitwise
from psyclonebench_amd import _native
from psyclonebench_amd.closure import (ClosureNet, coarse_model, conv_form, init_params,
                                       layer_offsets, set_conv_form)
from psyclonebench_amd.model import MASK_WEST_OPEN, Bathymetry, Model, NemoConfig, c1_config
from psyclonebench_amd.psy import TimeStepper

pytestmark = pytest.mark.gpu

FWD_TOL = 1e-2
GRAD_TOL = 3e-2


@pytest.fixture(autouse=True)
def _release():
    yield
    _native.hip_lib().nemo_hip_release_all()


def coarse_test_model(nx=64, ny=16) -> Model:
    return Model(NemoConfig(jpiglo=nx + 2, jpjglo=ny + 2, jphgr_msh=MASK_WEST_OPEN,
                            dx=4000.0, dy=4000.0, rdt=80.0, cbfr=0.0015, tide_amp=1.0,
                            tide_omega=2 * math.pi / 44712.0))


def net_params(seed=3) -> np.ndarray:
    rng = np.random.default_rng(seed + 100)
    p = init_params(seed)
    offs = layer_offsets()
    for l, (cin, cout) in enumerate(co.LAYERS):
        b0 = offs[l] + 25 * cin * cout
        used = 3 if l == 3 else cout
        p[b0:b0 + used] = 0.1 * rng.standard_normal(used)
    p[offs[3]:offs[3] + 25 * 32 * 16] *= 10.0   # output layer at full scale
    return p


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def test_forward_matches_oracle():
    m = coarse_test_model(64, 16)
    p = net_params()
    net = ClosureNet(m, params=p)
    x = np.random.default_rng(0).standard_normal((16, 64, 4))
    gpu = net.forward_host(x)
    ref, _ = co.forward(p.astype(np.float64), x, quant=True)
    errs = [rel(gpu[..., k], ref[..., k]) for k in range(3)]
    print("forward rel L2 error per channel:", errs, flush=True)
    assert max(errs) < FWD_TOL
    net.release()


def test_conv_forms_bitwise_equal():
    """Both launch forms of the 32 -> 32 convolutions (two tiles per
    wavefront pass, or one) give the same bits: the forward output, the loss
    and every gradient, on a 96 x 37 grid (the last 28-pixel column tile
    overlaps its neighbour)."""
    m = coarse_test_model(96, 37)
    p = net_params(6)
    rng = np.random.default_rng(7)
    x = rng.standard_normal((37, 96, 4))
    t = rng.standard_normal((37, 96, 3))
    out = {}
    default = conv_form()
    try:
        for form in (0, 1):
            set_conv_form(form)
            net = ClosureNet(m, params=p)
            y = net.forward_host(x)
            loss, g = net.grad_host(x, t)
            out[form] = (y, loss, g)
            net.release()
    finally:
        set_conv_form(default)
    assert_bitwise(out[1][0], out[0][0], "forward")
    assert out[1][1] == out[0][1]
    assert_bitwise(out[1][2], out[0][2], "gradients")


@pytest.mark.parametrize("weights", [(1.0, 1.0, 1.0), (1.0, 3.0, 0.5)])
def test_gradients_match_oracle(weights):
    m = coarse_test_model(64, 16)
    p = net_params(4)
    net = ClosureNet(m, params=p)
    net.set_loss_weights(*weights)
    rng = np.random.default_rng(1)
    x = rng.standard_normal((16, 64, 4))
    t = rng.standard_normal((16, 64, 3))
    loss_g, g = net.grad_host(x, t)
    loss_o, go = co.loss_and_grad(p.astype(np.float64), x, t, quant=True, weights=weights)
    # the reported loss is the unweighted mean squared error
    loss_u, _ = co.loss_and_grad(p.astype(np.float64), x, t, quant=True)
    print("weights", weights, "loss gpu / oracle:", loss_g, loss_u, flush=True)
    assert abs(loss_g - loss_u) / loss_u < FWD_TOL
    offs = layer_offsets()
    for l, (cin, cout) in enumerate(co.LAYERS):
        nw = 25 * cin * cout
        ci_used = 4 if l == 0 else cin
        co_used = 3 if l == 3 else cout
        gw = g[offs[l]:offs[l] + nw].reshape(25, cout, cin)[:, :co_used, :ci_used]
        ow = go[offs[l]:offs[l] + nw].reshape(25, cout, cin)[:, :co_used, :ci_used]
        gb = g[offs[l] + nw:offs[l] + nw + co_used]
        ob = go[offs[l] + nw:offs[l] + nw + co_used]
        ew, eb = rel(gw, ow), rel(gb, ob)
        print(f"layer {l}: weight grad rel err {ew:.2e}, bias grad rel err {eb:.2e}", flush=True)
        assert ew < GRAD_TOL and eb < GRAD_TOL
        # padded channels receive exactly zero gradient
        full = g[offs[l]:offs[l] + nw].reshape(25, cout, cin)
        assert not np.any(full[:, co_used:, :]) and not np.any(full[:, :, ci_used:])
    net.release()


@pytest.mark.parametrize("nx, ny", [(32, 3), (32, 12), (96, 37), (256, 400)])
def test_gradient_partials_over_sizes(nx, ny):
    """Weight and bias gradients where the row chunks change: fewer rows than
    one team takes, an idle second team, a remainder, more than two groups of
    rows a team. The bound is that of the gradients against the oracle."""
    print("gradients", nx, ny, flush=True)
    p = net_params(8)
    net = ClosureNet(coarse_test_model(nx, ny), params=p)
    rng = np.random.default_rng(9)
    x, t = rng.standard_normal((ny, nx, 4)), rng.standard_normal((ny, nx, 3))
    _, g = net.grad_host(x, t)
    net.release()
    _, go = co.loss_and_grad(p.astype(np.float64), x, t, quant=True)
    offs = layer_offsets()
    for l, (cin, cout) in enumerate(co.LAYERS):
        n = 25 * cin * cout
        for what, sl in (("weights", slice(offs[l], offs[l] + n)),
                         ("biases", slice(offs[l] + n, offs[l] + n + cout))):
            e = rel(g[sl], go[sl])
            print(f"layer {l} {what}: {e:.2e}", flush=True)
            assert e < GRAD_TOL


def test_adam_step_matches_formula():
    m = coarse_test_model(64, 16)
    p = net_params(5)
    net = ClosureNet(m, params=p)
    net.set_optimizer("adam", lr=1e-3)
    rng = np.random.default_rng(2)
    x, t = rng.standard_normal((16, 64, 4)), rng.standard_normal((16, 64, 3))
    _, g = net.grad_host(x, t)
    net.train_host(x, t)
    p1 = net.params()
    b1, b2, eps, lr = np.float32(0.9), np.float32(0.999), np.float32(1e-8), np.float32(1e-3)
    mh = ((1 - b1) * g) / (1 - b1)
    vh = ((1 - b2) * g * g) / (1 - b2)
    expect = p - lr * mh / (np.sqrt(vh) + eps)
    np.testing.assert_allclose(p1, expect, rtol=1e-5, atol=1e-7)
    net.release()


def test_training_fits_a_learnable_map():
    """Targets that are a fixed local linear map of the inputs: 300 Adam
    steps on the GPU cut the loss by more than 5x (the best of the last 100
    steps), and the run has not diverged at its end (the mean of the last 10
    below 0.6x the first). The trajectory amplifies FP32 rounding: two
    bias-gradient reductions that agree to 1e-8 (a different summation
    order) end this run at 0.022 and 0.037 from 0.263, and two input-layer
    kernels that sum the 5x5 taps in different orders reach 0.019 and 0.024
    and then, for one of them, a late spike of Adam at this learning rate
    (0.134 over the last 10 steps); seeds 7-11 end at 0.013-0.035 with
    either kernel."""
    m = coarse_test_model(64, 32)
    net = ClosureNet(m, seed=6)
    net.set_optimizer("adam", lr=3e-3)
    rng = np.random.default_rng(3)
    losses = []
    for k in range(300):
        x = rng.standard_normal((32, 64, 4))
        t = np.stack([0.5 * np.roll(x[..., 2], 1, axis=1) - 0.3 * x[..., 0],
                      0.4 * x[..., 1] * 1.0 - 0.2 * np.roll(x[..., 2], 1, axis=0),
                      0.3 * (x[..., 0] - np.roll(x[..., 0], 1, axis=1))], axis=-1)
        losses.append(net.train_host(x, t))
    print("loss first / best of the last 100 / last 10:", losses[0], min(losses[-100:]),
          np.mean(losses[-10:]), flush=True)
    assert min(losses[-100:]) < 0.2 * losses[0]
    assert np.mean(losses[-10:]) < 0.6 * losses[0]
    net.release()


def _fine_and_coarse(nxf=128, nyf=64, seed=9):
    cfg = replace(c1_config(10), jpiglo=nxf + 2, jpjglo=nyf + 2,
                  bathymetry=Bathymetry(seed=seed, sigma=8.0))
    fine = Model(cfg)
    coarse = coarse_model(fine, 4)
    return fine, coarse


def test_filter_and_set_state():
    fine, coarse = _fine_and_coarse()
    sf, sc = TimeStepper(fine, mode=2), TimeStepper(coarse, mode=2)
    sf.run(1)
    sc.run(1)
    gf, gc = fine.grid, coarse.grid
    rng = np.random.default_rng(4)
    lib = _native.hip_lib()
    host = {}
    for n in ("sshn_t", "un", "vn"):
        a = rng.standard_normal((gf.H, gf.W))
        host[n] = a
        lib.c_write_to_device(a.ctypes.data, fine.fields[n].device_ptr, 1, 1, gf.W, gf.H, True)
    net = ClosureNet(coarse)
    net.filter_fine(sf, 4)
    nx, ny = gc.M - 2, gc.N - 2
    s = host["sshn_t"][1:1 + 4 * ny, 1:1 + 4 * nx].reshape(ny, 4, nx, 4).mean(axis=(1, 3))
    u = host["un"][1:1 + 4 * ny, 4:4 * nx + 1:4].reshape(ny, 4, nx).mean(axis=1)
    v = host["vn"][4:4 * ny + 1:4, 1:1 + 4 * nx].reshape(ny, nx, 4).mean(axis=2)
    F = {n: net.filtered(n, (gc.H, gc.W)) for n in ("sshn_t", "un", "vn")}
    np.testing.assert_allclose(F["sshn_t"][1:ny + 1, 1:nx + 1], s, rtol=1e-13, atol=1e-15)
    np.testing.assert_allclose(F["un"][1:ny + 1, 1:nx + 1], u, rtol=1e-13, atol=1e-15)
    np.testing.assert_allclose(F["vn"][1:ny + 1, 1:nx + 1], v, rtol=1e-13, atol=1e-15)

    before = {n: sc.fetch(n) for n in ("sshn_t", "un", "vn", "sshn_u", "sshn_v")}
    net.set_state(sc)
    after = {n: sc.fetch(n) for n in ("sshn_t", "un", "vn", "sshn_u", "sshn_v")}
    exp = {n: before[n].copy() for n in before}
    exp["sshn_t"][1:ny + 1, 1:nx + 1] = F["sshn_t"][1:ny + 1, 1:nx + 1]
    exp["un"][1:ny + 1, 1:nx] = F["un"][1:ny + 1, 1:nx]
    exp["vn"][1:ny, 1:nx + 1] = F["vn"][1:ny, 1:nx + 1]
    # face ssh as next_sshu / next_sshv compute it from the new T-cell ssh
    ol = oracle.oracle_lib()
    P = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
    tm = coarse.array("tmask")
    ol.oracle_next_sshu(1, nx - 1, 1, ny, gc.W, P(exp["sshn_u"]), P(exp["sshn_t"]),
                        tm.ctypes.data_as(C.POINTER(C.c_int)), P(coarse.array("area_t")),
                        P(coarse.array("area_u")))
    ol.oracle_next_sshv(1, nx, 1, ny - 1, gc.W, P(exp["sshn_v"]), P(exp["sshn_t"]),
                        tm.ctypes.data_as(C.POINTER(C.c_int)), P(coarse.array("area_t")),
                        P(coarse.array("area_v")))
    for n in after:
        assert_bitwise(after[n], exp[n], n)
    net.release()


def test_training_step_equals_the_step_on_its_inputs():
    """train_step takes its input and target from the model's fields; the same
    input and target handed over from the host give the same loss and weights,
    bit for bit (every interior cell wet and counted, no gate)."""
    fine, coarse = _fine_and_coarse()
    sf, sc = TimeStepper(fine, mode=2), TimeStepper(coarse, mode=2)
    sf.run(3)
    sc.run(1)
    g = coarse.grid
    inner = (slice(1, g.N - 1), slice(1, g.M - 1))
    assert np.all(coarse.array("tmask")[inner] > 0)
    p, out = net_params(12), []
    for from_model in (True, False):
        net = ClosureNet(coarse, params=p)
        net.set_ssh_cells(True)
        net.set_optimizer("sgd", lr=1e-2)
        net.filter_fine(sf, 4)
        if from_model:
            net.train_step(sc)
            loss = net.last_loss()
        else:
            names = ("un", "vn", "sshn_t")
            state = [sc.fetch(n) for n in names]
            x = np.stack([a[inner] for a in state] + [coarse.array("ht")[inner]], -1)
            t = np.stack([(net.filtered(n, (g.H, g.W)) - a)[inner]
                          for n, a in zip(names, state)], -1)
            loss = net.train_host(x, t)
        out.append((loss, net.params()))
        net.release()
    assert out[0][0] == out[1][0] > 0.0
    assert_bitwise(out[0][1], out[1][1], "weights")
    assert np.any(out[0][1] != p.astype(np.float32))


def test_guard_keeps_plain_step_on_blowup():
    fine, coarse = _fine_and_coarse()
    sc = TimeStepper(coarse, mode=2)
    sc.run(5)
    net = ClosureNet(coarse, params=net_params(7))
    net.set_norm([0, 0, 0, 100], [1, 1, 1, 50], [1e30, 1e30, 1e30])
    net.set_guard(0.05, 0.0)
    before = {n: sc.fetch(n) for n in ("sshn_t", "un", "vn", "sshn_u", "sshn_v")}
    net.correct(sc, guard=True)
    assert net.guard_trips() == 1
    for n in before:
        assert_bitwise(sc.fetch(n), before[n], n)
    # a small correction passes and changes the state
    net.set_norm([0, 0, 0, 100], [1, 1, 1, 50], [1e-9, 1e-9, 1e-9])
    net.set_guard(0.05, 1e-6)
    net.correct(sc, guard=True)
    assert net.guard_trips() == 1
    assert np.any(sc.fetch("sshn_t") != before["sshn_t"])
    net.release()


def test_guard_sums_equal_energy_of_the_state():
    """The energy sums the output layer folds in (E before and after the
    correction, the non-finite count) against numpy over the interior of
    the coarse state fetched before and after an accepted correction:
    E = sum g ssh^2 + ht (u^2 + v^2), to 1e-12 relative (the GPU sums in
    another order)."""
    _, coarse = _fine_and_coarse()
    sc = TimeStepper(coarse, mode=2)
    sc.run(5)
    g = coarse.grid
    nx, ny = g.M - 2, g.N - 2
    net = ClosureNet(coarse, params=net_params(7))
    net.set_norm([0, 0, 0, 100], [1, 1, 1, 50], [1e-4, 1e-4, 1e-4])
    net.set_guard(1e6, 1e6)  # accept
    grav = 9.80665
    ht = coarse.array("ht")[1:ny + 1, 1:nx + 1]

    def energy(st):
        s_, u_, v_ = (st[n][1:ny + 1, 1:nx + 1] for n in ("sshn_t", "un", "vn"))
        return float(np.sum(grav * s_ * s_ + ht * (u_ * u_ + v_ * v_)))

    before = {n: sc.fetch(n) for n in ("sshn_t", "un", "vn")}
    net.correct(sc, guard=True)
    after = {n: sc.fetch(n) for n in ("sshn_t", "un", "vn")}
    assert net.guard_trips() == 0
    assert any(np.any(after[n] != before[n]) for n in after)
    st = net.last_stats()
    e0, e1 = energy(before), energy(after)
    print("guard energies", st["energy_before"], e0, st["energy_after"], e1, flush=True)
    assert st["nonfinite"] == 0.0
    assert abs(st["energy_before"] - e0) <= 1e-12 * abs(e0)
    assert abs(st["energy_after"] - e1) <= 1e-12 * abs(e1)
    assert e1 != e0
    net.release()


@pytest.mark.timeout(600)
def test_shipped_weights_halve_the_plain_coarse_error():
    """The bar the learned closure is built to: on held-out bathymetries
    (seeds 64 and 65) at the training size (fine 4096^2 FP64, coarse 1024^2)
    over the evaluation's 2000 coarse steps (44 h), the learned coarse model's
    error against the box-filtered fine run is at most half the plain coarse
    model's, for u, v and ssh (mean over the run, every 100 steps, relative
    RMS over the interior), with no correction rejected by the energy guard.
    The ssh is measured over the cells the coarse step evolves: the step
    clamps the wet cells next to the open edge to the tidal elevation in both
    coarse forms, so those cells carry the same error with or without the
    correction; the all-cell ratio is printed."""
    from psyclonebench_amd import closure_run as cr
    if not cr.DEFAULT_WEIGHTS.exists():
        pytest.fail(f"no trained weights at {cr.DEFAULT_WEIGHTS}")
    print("closure gain: seeds 64, 65, 2000 coarse steps at 1024^2", flush=True)
    res = cr.evaluate(4096, 4, [64, 65], 2000, 100, cr.DEFAULT_WEIGHTS,
                      log_fn=lambda *x: print(*x, flush=True))
    print("ratio (mean, final):", res["ratio_mean"], res["ratio_final"], flush=True)
    for b in (64, 65):
        s = res["seeds"][b]
        assert s["guard_trips"] == 0, b
        for f in ("un", "vn", "sshn_t_free"):
            assert s["ratio_mean"][f] <= 0.5, (b, f, s["ratio_mean"][f])


def test_training_command_end_to_end(tmp_path):
    """The `closure_run train` command at a small size (fine 256^2, coarse
    64^2): pilot normalisation, spin-ups, rollouts with spike restarts, the
    moving average of the weights, model selection on a held-out seed, the
    saved file, and an evaluation of it."""
    import json as _json

    from psyclonebench_amd import closure_run as cr
    out = tmp_path / "w.npz"
    print("closure train command: fine 256^2, 2 seeds x 30 steps", flush=True)
    cr.main(["train", "--n", "256", "--bathy", "0:2", "--steps", "30", "--pilot-steps", "100",
             "--max-spin", "5", "--rollout", "5", "--ema", "0.9", "--ema-every", "2",
             "--ema-start", "0", "--reset-spike", "4", "--log-every", "10",
             "--val-every", "1", "--val-steps", "40", "--out", str(out)])
    z = np.load(out)
    meta = _json.loads(str(z["meta"]))
    assert z["params"].shape == (_native.hip_lib().nemo_cl_param_count(),)
    assert np.all(np.isfinite(z["params"]))
    assert meta["ema"] == 0.9 and meta["reset_spike"] == 4.0
    assert len(meta["history"]) == 2
    # model selection ran after each seed and kept one of the two
    assert [v["after_seed"] for v in meta["validation"]] == [0, 1]
    assert meta["selected_after_seed"] in (0, 1)
    assert not (tmp_path / "w.validation.npz").exists()
    res = cr.evaluate(256, 4, [2], 20, 10, out, log_fn=lambda *x: None)
    for f in ("sshn_t", "un", "vn"):
        assert math.isfinite(res["ratio_mean"][f]), f


@pytest.mark.parametrize("guard", [True, False])
def test_captured_learned_steps_equal_stepwise(guard):
    """nemo_cl_steps (coarse step + correction, captured as one graph and
    replayed) against alternating c_invoke_time_step and nemo_cl_correct on
    a twin model: bitwise equal after 7 + 30 steps (two graph lengths, the
    second from the other ping-pong parity), with the same guard trips. A
    settings change (the guard) must be seen by the next replay."""
    _, coarse = _fine_and_coarse()
    twin = coarse.copy()
    a, b = TimeStepper(coarse, mode=2), TimeStepper(twin, mode=2)
    a.run(3)
    b.run(3)
    na = ClosureNet(coarse, params=net_params(5))
    nb = ClosureNet(twin, params=net_params(5))
    for net in (na, nb):
        net.set_norm([0, 0, 0, 100], [0.5, 0.5, 0.5, 50], [1e-3, 1e-3, 1e-3])
        net.set_gate(0.01)
        net.set_guard(0.05, 1e-3)
    fields = ("sshn_t", "un", "vn", "sshn_u", "sshn_v")
    for n, rel_guard, abs_tol in ((7, 0.05, 1e-3), (30, 0.05, 1e-3), (30, 1e-9, 0.0)):
        for net in (na, nb):
            net.set_guard(rel_guard, abs_tol)
        na.steps(a, n, guard=guard)
        for _ in range(n):
            b.step()
            nb.correct(b, guard=guard)
        for f in fields:
            assert_bitwise(a.fetch(f), b.fetch(f), f"{n} steps, guard {rel_guard}: {f}")
        assert na.guard_trips() == nb.guard_trips()
    print("guard trips:", na.guard_trips(), flush=True)
    na.release()
    nb.release()
