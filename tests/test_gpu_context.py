"""A context whose parameters change while it lives: the same results as one
made with those parameters."""
import numpy as np
import pytest

from fooskagpu_amd import GpuSolver, _lib, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [_lib.RELAX_COLD, _lib.RELAX_PLAIN])
def test_precision_of_a_live_context_changes(gpu, mode):
    """178,746 tetrahedra, between the sizes up to which pass F with the
    relaxation takes four lanes per cell in mixed precision (50,000 and
    160,000) and in FP64 (220,000): mixed first, then FP64, then mixed again,
    against contexts of one precision; states, time step and counts."""
    c = cases.shock_bubble(n=31, nbub=5)
    assert 160000 < c.mesh.n_cells <= 220000
    print(f"[precision] {c.mesh.n_cells} cells, mode {mode}", flush=True)
    want = {}
    for prec in (_lib.FP64, _lib.MIXED):
        with GpuSolver(dict(c.params, precision=prec, relaxMode=mode), c.mesh, c.U) as g:
            want[prec] = (g.run_steps(2), g.download_state(), g.relax_totals())
    with GpuSolver(dict(c.params, precision=_lib.MIXED, relaxMode=mode), c.mesh, c.U) as g:
        for prec in (_lib.MIXED, _lib.FP64, _lib.MIXED):
            g.set_params(dict(c.params, precision=prec, relaxMode=mode))
            g.upload_state(c.U)
            g.set_clock(0.0, 0.0, 0)
            g.relax_totals(reset=True)
            got = (g.run_steps(2), g.download_state(), g.relax_totals())
            assert got[0] == want[prec][0] and got[2] == want[prec][2]
            assert np.array_equal(got[1], want[prec][1])
