"""Masks with wet cells in the first row and column, whose Flather faces read a
neighbour before the extent (read as 0 where it lies before the allocation,
where the reference reads out of bounds): the band tiles against the kernels
that run the Flather faces from host-built lists, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import assert_bitwise
from psyclonebench_amd import _native
from psyclonebench_amd.ensemble import EnsembleStepper
from psyclonebench_amd.psy import MixedStepper, TimeStepper
from test_gpu_band import OUT, live_model
from test_zz_no_alloc import OUT as INPLACE, _run_host, _run_noalloc

pytestmark = pytest.mark.gpu

FIELDS = ("sshn_t", "un", "vn", "sshn_u", "sshn_v")


@pytest.fixture(autouse=True)
def _release():
    yield
    _native.hip_lib().nemo_hip_release_all()


def edge_model(nx: int, ny: int, metrics: str, seed: int):
    """Wet, dry and open cells in the first row and column as everywhere, the
    corner wet; no wet cell in the last T row (which the fused form needs)."""
    m = live_model(nx, ny, metrics, seed=seed)
    g = m.grid
    t = np.random.default_rng(seed).choice(np.array([-1, 0, 1], np.int32), size=(g.N, g.M),
                                           p=[0.15, 0.05, 0.8])
    t[g.N - 1] = np.minimum(t[g.N - 1], 0)
    t[0, 0], t[0, 1], t[1, 0] = 1, -1, -1
    g.tmask[:g.N, :g.M] = t
    return m


@pytest.mark.parametrize("metrics", ["row", "point"])
@pytest.mark.parametrize("nx, ny", [(3, 3), (64, 61), (300, 290), (500, 450), (1501, 1200)])
def test_first_row_and_column(nx, ny, metrics):
    print("edges", nx, ny, metrics, flush=True)
    m = edge_model(nx, ny, metrics, seed=61)
    lib, out = _native.hip_lib(), []
    default = lib.nemo_hip_fused_variant()
    try:
        for variant in (default, 30):
            lib.nemo_hip_set_fused_variant(variant)
            st = TimeStepper(m.copy(), mode=2)
            st.run(3)
            out.append({n: st.fetch(n) for n in OUT})
    finally:
        lib.nemo_hip_set_fused_variant(default)
    for n in OUT:
        assert_bitwise(out[0][n], out[1][n], f"{nx}x{ny} {metrics} {n}")
    out = []
    for rows, cols in ((32, 61), (16, 48)):
        mp = MixedStepper(m, rows=rows, cols=cols)
        mp.run(3)
        out.append({n: mp.fetch(n) for n in FIELDS})
        mp.release()
    for n in FIELDS:
        assert_bitwise(out[0][n], out[1][n], f"FP32 {nx}x{ny} {metrics} {n}")


@pytest.mark.parametrize("nx, ny", [(3, 3), (300, 290), (1201, 900)])
def test_first_row_and_column_in_place(nx, ny):
    m = edge_model(nx, ny, "point", seed=62)
    m.array("gphiu")[:] = 0.0
    m.array("gphiv")[:] = 0.0
    _native.hip_lib().nemo_hip_set_tide(m.cfg.tide_amp, m.cfg.tide_omega)
    ref = _run_host(m.copy(), 1, 2)
    got = _run_noalloc(m.copy(), 1, 2)
    for n in INPLACE:
        assert_bitwise(got[n], ref[n], f"in place {nx}x{ny} {n}")


@pytest.mark.parametrize("precision", [64, 32])
def test_first_row_and_column_in_an_ensemble(precision):
    """The second domain's first faces lie behind the first domain's last values."""
    models = [edge_model(nx, ny, "row", seed=63 + k)
              for k, (nx, ny) in enumerate(((61, 40), (130, 61), (300, 290)))]
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
