"""States that are no longer physical: the kernel variants agree there too, so
that a result does not depend on the size of the mesh."""
import numpy as np
import pytest

from fooskagpu_amd import GpuSolver, Mesh, _lib, cases
from test_gpu_kernels import rough_state

pytestmark = pytest.mark.gpu

VALUES = {"nan": np.nan, "inf": np.inf, "-inf": -np.inf, "huge": 1e300, "negative": -1.0}


@pytest.mark.parametrize("precision", [_lib.FP64, _lib.MIXED])
@pytest.mark.parametrize("elements", ["tets", "mixed"])
@pytest.mark.parametrize("model", [_lib.MODEL_SINGLE, _lib.MODEL_TWO_PHASE])
@pytest.mark.parametrize("value", sorted(VALUES))
def test_variants_agree_on_states_that_are_not_physical(gpu, model, elements, precision, value):
    """Cells with one variable set to a NaN, an infinity or the like, alone and
    next to each other (faces with such a state on both sides): face states,
    limiter, residual, signal speeds and time step of four lanes per cell, of
    one with LDS and of one without, bit for bit."""
    p = dict(cases.BASE, viscFlag=0) if model == _lib.MODEL_SINGLE else cases._two_phase_params()
    m = Mesh.box(4, 4, 4, jitter=0.1, seed=5) if elements == "tets" else Mesh.mixed_box(7, 3, 3, jitter=0.1, seed=5)
    neq = 5 if model == _lib.MODEL_SINGLE else 10
    U = rough_state(neq, m.n_cells, "random", 7)
    rng = np.random.default_rng(11)
    for c in rng.choice(m.n_cells, m.n_cells // 20, replace=False):
        U[c, rng.integers(neq)] = VALUES[value]
    for f in rng.choice(np.flatnonzero(m.fc2el[:, 1] >= 0), m.n_cells // 12, replace=False):
        U[m.fc2el[f], 3] = VALUES[value]
    print(f"[nonfinite] {value} {model} {elements} {precision}", flush=True)
    out = []
    for stage in (1, 2, 0):
        with GpuSolver(dict(p, precision=precision), m, U) as g:
            g.set_tuning("stage_f", stage)
            g.set_tuning("stage_g", stage)
            g.set_debug(True)
            g.compute_face_values()
            live = g.download("slots") >= 0
            g.compute_rhs()
            out.append((g.download("theta"), g.download("grad"), g.download("face")[live], g.download("rhs"),
                        g.download("signal"), np.array(g.compute_time_step())))
    for k, o in enumerate(out[1:]):
        for name, a, b in zip(("theta", "grad", "face", "rhs", "signal", "dt"), out[0], o):
            same = (a == b) | (np.isnan(a) & np.isnan(b))
            assert same.all(), (name, (2, 0)[k], int((~same).sum()), a[~same][:3], b[~same][:3])
