"""WALE eddy viscosity in mixed precision where its FP32 powers are near the
end of their range."""
import numpy as np
import pytest

from fooskagpu_amd import GpuSolver, Mesh, _lib, cases
from fooskagpu_amd.mesh import KIND_HEX

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stage", [1, 2, 0])
@pytest.mark.parametrize("shear", [2e7, 5.7e7])
def test_eddy_viscosity_of_a_strong_shear(gpu, shear, stage):
    """u = G y with G from `shear` to 1.25 shear (1/s) and v = 1e5 x on 1 mm:
    the fifth power of the strain rate, the divisor of the eddy viscosity,
    lies between 2^126 and 2^128 in the second case (8.5e37 to 3.4e38; its
    reciprocal is no normal FP32 number), far below in the first.  The
    momentum that the eddies move, the difference of a stage with and without
    them (molecular viscosity 0), against the same difference in FP64.  FP32
    velocities of 6e4 m/s over cells of 1e-4 m leave a gradient error of 6e4
    2^-24 / 1e-4 = 40 1/s; it enters the limiter of the powers as u_x G beside
    v_x G, 4e-4, so 1 % leaves a factor of 10 for powers and sums."""
    L, n, dt = 1e-3, 8, 1e-6
    m = Mesh.box(n, n, n, hi=(L, L, L), kinds=KIND_HEX, bc=(2,) * 6)
    x, y = m.cell_center[:, 0], m.cell_center[:, 1]
    u, v = shear * y + 0.25 * shear * y * y / (2 * L), 1e5 * x
    U = np.stack([np.ones_like(u), u, v, 0 * u, 1e9 / 0.4 + 0.5 * (u * u + v * v)], 1)
    p = dict(cases.BASE, viscFlag=1, rkSteps=1, adaptDt=0, dt=dt, dynVisc=[0.0, 0.0])
    den = (0.5 * np.array([shear, 1.25 * shear]) ** 2) ** 2.5
    assert (den < 2.0 ** 126).all() if shear < 5e7 else (den > 2.0 ** 126).all() and (den < 2.0 ** 128).all()
    move = {}
    for prec in (_lib.FP64, _lib.MIXED):
        new = []
        for turb in (1, 0):
            with GpuSolver(dict(p, precision=prec, turbulence=turb), m, U) as g:
                g.set_tuning("stage_f", stage)
                g.compute_face_values()
                g.compute_rhs_update(0, dt)
                new.append(g.download_state()[:, 1])
        move[prec] = new[0] - new[1]
    err = np.linalg.norm(move[_lib.MIXED] - move[_lib.FP64]) / np.linalg.norm(move[_lib.FP64])
    print(f"[wale] shear {shear:.2g}, divisor {den[0]:.2e} to {den[1]:.2e}, moved {np.abs(move[_lib.FP64]).max():.2e}, "
          f"mixed off by {err:.2e}", flush=True)
    assert err < 1e-2
