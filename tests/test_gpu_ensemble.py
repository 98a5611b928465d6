"""Batched ensemble (nemo_ens_*) on the GPU, through the C ABI.

FP64: every domain of the ensemble is bitwise the oracle run of that domain
alone (rows 0 .. N-2, the rows the fused form writes like the reference),
for every launch shape. Mixed precision: every domain is bitwise the
single-domain mixed form (nemo_mp_*), which test_gpu_mixed pins to the
oracle within its stated tolerances."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from helpers import assert_bitwise, live_state_model, rel_err
from psyclonebench_amd import _native
from psyclonebench_amd.ensemble import EnsembleStepper, ensemble_configs
from psyclonebench_amd.model import Model
from psyclonebench_amd.psy import MixedStepper, TimeStepper
from test_gpu_band import live_model as band_model

pytestmark = pytest.mark.gpu

FIELDS = ("sshn_t", "un", "vn", "sshn_u", "sshn_v")


@pytest.fixture(autouse=True)
def _release():
    yield
    _native.hip_lib().nemo_hip_release_all()


def small_ensemble(ndom=6, seed=5, nsteps=40):
    # uneven sides 20..130 (ragged strips and bands), own depth and tide
    return ensemble_configs(ndom=ndom, seed=seed, n_min=20, n_max=130, nsteps=nsteps)


def oracle_domain(cfg, nsteps):
    m = Model(cfg)
    g = m.grid
    arrays = m.arrays()
    oracle.set_tide(cfg.tide_amp, cfg.tide_omega)
    try:
        oracle.run_steps(arrays, cfg.nit000, nsteps, g.bounds, g.W, m.scalars,
                         kind="oracle_omp")
    finally:
        oracle.oracle_lib().oracle_reset_tide()
    return {n: m.array(n) for n in FIELDS}, g


def test_ensemble_f64_matches_oracle_per_domain():
    cfgs = small_ensemble()
    nsteps = 40
    ens = EnsembleStepper([Model(c) for c in cfgs], precision=64)
    print("ensemble points", ens.interior_points, flush=True)
    ens.run(nsteps)
    for d, cfg in enumerate(cfgs):
        ref, g = oracle_domain(cfg, nsteps)
        for n in FIELDS:
            assert_bitwise(ens.fetch(d, n)[:g.N - 1], ref[n][:g.N - 1],
                           f"domain {d} ({g.M}x{g.N}) {n}")
    ens.release()


@pytest.mark.parametrize("precision", [64, 32])
def test_ensemble_every_shape_bitwise_equal(precision):
    """Every launch shape (rows x columns x prefetch depth x launch form:
    one wavefront per tile, or persistent with so many wavefronts per
    workgroup and residency) gives the same bits, in both precisions."""
    cfgs = small_ensemble(ndom=5, seed=7)
    models = [Model(c) for c in cfgs]
    probe = EnsembleStepper(models, precision=precision)
    nshape = len(probe.shapes())
    shapes = probe.shapes()
    assert {s[3] for s in shapes} == {61, 56, 0}
    assert {s[4] for s in shapes} == {0, 1, 2}
    assert any(s[2] == 0 for s in shapes) and any(s[2] > 0 for s in shapes)
    probe.release()
    ref = None
    for k in range(nshape):
        ens = EnsembleStepper(models, precision=precision)
        ens.set_shape(k)
        print("precision", precision, "shape", k, ens.shapes()[k], flush=True)
        ens.run(12)
        out = [{n: ens.fetch(d, n) for n in ("sshn_t", "un", "vn")}
               for d in range(len(cfgs))]
        ens.release()
        if ref is None:
            ref = out
            continue
        for d in range(len(cfgs)):
            for n in out[d]:
                assert_bitwise(out[d][n], ref[d][n], f"shape {k} domain {d} {n}")


def test_ensemble_graph_equals_timed_and_single_calls():
    cfgs = small_ensemble(ndom=4, seed=9)
    a = EnsembleStepper([Model(c) for c in cfgs])
    b = EnsembleStepper([Model(c) for c in cfgs])
    c = EnsembleStepper([Model(c) for c in cfgs])
    a.run(17)
    ms = b.timed_run(17)
    assert ms > 0
    for _ in range(17):
        c.run(1)
    for d in range(len(cfgs)):
        for n in FIELDS:
            x = a.fetch(d, n)
            assert_bitwise(b.fetch(d, n), x, f"timed domain {d} {n}")
            assert_bitwise(c.fetch(d, n), x, f"single domain {d} {n}")
    for e in (a, b, c):
        e.release()


def test_ensemble_autotune_restores_state():
    cfgs = small_ensemble(ndom=4, seed=11)
    a = EnsembleStepper([Model(c) for c in cfgs])
    b = EnsembleStepper([Model(c) for c in cfgs])
    a.run(5)
    b.run(5)
    best, ms = a.autotune(2)
    print("autotune:", best, a.shapes()[best], [round(x, 4) for x in ms], flush=True)
    assert 0 <= best < len(ms) and all(x > 0 for x in ms)
    assert ms[best] == min(ms)
    a.run(9)
    b.run(9)
    for d in range(len(cfgs)):
        for n in FIELDS:
            assert_bitwise(a.fetch(d, n), b.fetch(d, n), f"domain {d} {n}")
    a.release()
    b.release()


def test_ensemble_autotune_before_first_step():
    cfgs = small_ensemble(ndom=3, seed=13)
    a = EnsembleStepper([Model(c) for c in cfgs])
    b = EnsembleStepper([Model(c) for c in cfgs])
    a.autotune(1)
    a.run(8)
    b.run(8)
    for d in range(len(cfgs)):
        for n in FIELDS:
            assert_bitwise(a.fetch(d, n), b.fetch(d, n), f"domain {d} {n}")
    a.release()
    b.release()


def test_ensemble_mixed_matches_single_domain_mixed():
    cfgs = small_ensemble(ndom=5, seed=17, nsteps=60)
    ens = EnsembleStepper([Model(c) for c in cfgs], precision=32)
    ens.run(60)
    for d, cfg in enumerate(cfgs):
        mp = MixedStepper(Model(cfg))
        mp.run(60)
        for n in FIELDS:
            assert_bitwise(ens.fetch(d, n), mp.fetch(n), f"domain {d} {n}")
        mp.release()
    ens.release()


def test_ensemble_mixed_error_against_f64():
    cfgs = small_ensemble(ndom=4, seed=19, nsteps=400)
    f64 = EnsembleStepper([Model(c) for c in cfgs], precision=64)
    f32 = EnsembleStepper([Model(c) for c in cfgs], precision=32)
    f64.run(400)
    f32.run(400)
    for d, cfg in enumerate(cfgs):
        g = f64.models[d].grid
        sl = (slice(g.ys, g.ye + 1), slice(g.xs, g.xe + 1))
        e = {n: rel_err(f32.fetch(d, n)[sl], f64.fetch(d, n)[sl]) for n in ("sshn_t", "un", "vn")}
        print("domain", d, e, flush=True)
        assert e["sshn_t"][0] <= 1e-5, e
        assert e["un"][0] <= 1e-4 and e["vn"][0] <= 1e-4, e
    f64.release()
    f32.release()


@pytest.mark.slow
def test_ensemble_256_domains_sample_equals_single_domain_fused():
    """The 256-domain ensemble (sides 64..1024): 30 graph-replayed steps;
    a sample of domains, smallest and largest included, is bitwise the
    single-domain fused form of that domain."""
    cfgs = ensemble_configs(ndom=256, seed=0, nsteps=30)
    ens = EnsembleStepper([Model(c) for c in cfgs], precision=64)
    print("256 domains, interior points", ens.interior_points, flush=True)
    ens.run(30)
    sizes = [(c.jpiglo - 2) * (c.jpjglo - 2) for c in cfgs]
    sample = sorted({int(np.argmin(sizes)), int(np.argmax(sizes)), 0, 100, 255})
    for d in sample:
        st = TimeStepper(Model(cfgs[d]), mode=2)
        st.run(30)
        g = st.model.grid
        for n in FIELDS:
            assert_bitwise(ens.fetch(d, n)[:g.N - 1], st.fetch(n)[:g.N - 1],
                           f"domain {d} {n}")
        st.release()
    ens.release()


def test_ensemble_random_masks_match_oracle_and_mixed():
    """Three domains with every array random and random {-1, 0, 1} masks
    (wet cells between open cells: bc_flather reads a face's value from the
    end of the previous step), 8 steps. FP64: each domain bitwise the
    oracle on all fields. FP32: each domain bitwise the single-domain mixed
    form."""
    models = [live_state_model(n, seed=60 + n, random_mask=True) for n in (40, 77, 96)]
    nsteps = 8
    ens = EnsembleStepper([m.copy() for m in models], precision=64)
    ens.run(nsteps)
    for d, m in enumerate(models):
        g = m.grid
        host = [a.copy() for a in m.arrays()]
        oracle.set_tide(m.cfg.tide_amp, m.cfg.tide_omega)
        try:
            oracle.run_steps(host, 1, nsteps, g.bounds, g.W, m.scalars)
        finally:
            oracle.oracle_lib().oracle_reset_tide()
        ref = dict(zip(oracle.ARRAY_NAMES, host))
        for n in ("sshn_u", "sshn_v"):
            assert_bitwise(ens.fetch(d, n), ref[n], f"f64 domain {d} {n}")
        for n in ("sshn_t", "un", "vn"):
            assert_bitwise(ens.fetch(d, n)[:g.N - 1, :g.M], ref[n][:g.N - 1, :g.M],
                           f"f64 domain {d} {n}")
    ens.release()
    ens = EnsembleStepper([m.copy() for m in models], precision=32)
    ens.run(nsteps)
    for d, m in enumerate(models):
        g = m.grid
        single = MixedStepper(m.copy())
        single.run(nsteps)
        for n in FIELDS:
            assert_bitwise(ens.fetch(d, n)[:g.N - 1, :g.M], single.fetch(n)[:g.N - 1, :g.M],
                           f"f32 domain {d} {n}")
        single.release()
    ens.release()


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("metrics", ["row", "point"])
@pytest.mark.parametrize("sizes", [((3, 3), (40, 33), (130, 61)), ((300, 290), (200, 150)),
                                   ((61, 64), (700, 620)), ((57, 4), (1101, 1400)),
                                   ((2501, 2403),)],
                         ids=["shared", "one", "two", "more", "largest"])
def test_ensemble_default_tiles_equal_the_persistent_kernel(sizes, metrics, precision):
    """The default shape, whose tiles follow the ensemble's size, has the bits
    of the persistent kernel with its separate Flather launch, on random masks
    and metrics."""
    print("default tiles", sizes, metrics, precision, flush=True)
    models = [band_model(nx, ny, metrics, seed=20 + k) for k, (nx, ny) in enumerate(sizes)]
    out = []
    for persistent in (False, True):
        ens = EnsembleStepper(models, precision=precision)
        if persistent:
            ens.set_shape([s[2] > 0 for s in ens.shapes()].index(True))
        ens.run(3)
        out.append([{n: ens.fetch(d, n) for n in FIELDS} for d in range(len(models))])
        ens.release()
    for d in range(len(models)):
        for n in FIELDS:
            assert_bitwise(out[0][d][n], out[1][d][n], f"domain {d} {n}")


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("metrics, sizes", [
    ("point", ((181, 300), (301, 590))), ("point", ((181, 300), (301, 640))),
    ("row", ((601, 500), (301, 960))), ("row", ((601, 500), (301, 1010)))],
    ids=["point 3866", "point 4116", "row 9830", "row 10080"])
def test_ensemble_shapes_on_both_sides_of_their_lines(metrics, sizes, precision):
    """Shapes of 4 and 8 rows, one wavefront a tile, run band tiles or
    overlapped-wavefront tiles by the number of one-row tiles (the ids; lines at
    4000 and 10000): the bits of the persistent kernel on either side."""
    print("shapes", metrics, sizes, precision, flush=True)
    models = [band_model(nx, ny, metrics, seed=40 + k) for k, (nx, ny) in enumerate(sizes)]
    probe = EnsembleStepper(models[:1], precision=precision)
    shapes = [k for k, s in enumerate(probe.shapes()) if s[2] == 0 and s[0] in (4, 8)]
    probe.release()
    assert len(shapes) == 18
    ref = None
    for k in [None] + shapes:
        ens = EnsembleStepper(models, precision=precision)
        ens.set_shape([s[2] > 0 for s in ens.shapes()].index(True) if k is None else k)
        ens.run(3)
        out = [{n: ens.fetch(d, n) for n in FIELDS} for d in range(len(models))]
        ens.release()
        ref = ref or out
        for d in range(len(models)):
            for n in FIELDS:
                assert_bitwise(out[d][n], ref[d][n], f"shape {k} domain {d} {n}")


def test_autotune_times_whole_steps():
    """A shape with a Flather launch of its own is compared with the band tiles,
    which need none, by the whole step: its time is that of the step kernel and
    of at least the shortest launch (over 1 us; the median of several tries)."""
    models = [band_model(64, 64, "row", seed=50 + k) for k in range(3)]
    ens = EnsembleStepper(models)
    shapes = ens.shapes()
    k = [s[:1] + s[2:] for s in shapes].index((16, 0, 61, 0))
    extra = []
    for _ in range(7):
        _, ms = ens.autotune(50)
        ens.set_shape(k)
        extra.append((ms[k] - ens.timed_run(50)) * 1e3)
    ens.release()
    print("whole step less its kernel, us:", [round(x, 2) for x in extra], flush=True)
    assert sorted(extra)[3] > 1.0
