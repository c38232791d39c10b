"""Kernel variants at the sizes and values where they can go wrong: edges of
workgroups, remainders, one-sided and empty slopes, against the FP64 oracle."""
import numpy as np
import pytest

from fooskagpu_amd import GpuSolver, Mesh, _lib, cases
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu


def rough_state(neq, n, kind, seed=0):
    """Positive states without smoothness ("random"), all alike ("uniform":
    every slope 0) or with one cell raised ("spike": slopes of one sign)."""
    rng = np.random.default_rng(seed)
    f = {"random": rng.uniform(0.5, 1.5, (n, neq)), "uniform": np.ones((n, neq)), "spike": np.ones((n, neq))}[kind]
    if kind == "spike":
        f[n // 2] = 1.4
    if neq == 5:
        return f * [1.0, 0.3, -0.2, 0.1, 2.5]
    a = 0.5 * f[:, :1]
    return np.concatenate([a, a * 900 * f[:, 1:2], (1 - a) * 20 * f[:, 2:3], 300 * (f[:, 3:6] - 0.7),
                           a * 900 * 1.5e6 * f[:, 6:7], (1 - a) * 20 * 2.4e6 * f[:, 7:8], 8e8 * f[:, 8:9],
                           0.01 * f[:, 9:]], 1)


@pytest.mark.parametrize("kind", ["random", "uniform", "spike"])
@pytest.mark.parametrize("elements", ["tets", "mixed"])
@pytest.mark.parametrize("model", [_lib.MODEL_SINGLE, _lib.MODEL_TWO_PHASE])
def test_limiter_and_gradients_are_the_oracles_bits(gpu, model, elements, kind):
    """Gradients (shared-divisor quotients), limiter (two quotients per
    variable) and face states: the oracle's operations with the same rounding,
    so equal bits."""
    p = dict(cases.BASE) if model == _lib.MODEL_SINGLE else cases._two_phase_params()
    m = Mesh.box(3, 5, 5, jitter=0.1, seed=5) if elements == "tets" else Mesh.mixed_box(7, 3, 3, jitter=0.1, seed=5)
    U = rough_state(5 if model == _lib.MODEL_SINGLE else 10, m.n_cells, kind)
    o = Oracle(p, m, U)
    o.compute_face_values()
    with GpuSolver(p, m, U) as g:
        g.set_debug(True)
        g.compute_face_values()
        live = g.download("slots") >= 0
        for name in ("grad", "theta", "face"):
            a, b = g.download(name), o.get(name)
            if name == "face":
                a, b = a[live], b[live]
            assert np.array_equal(a, b), (name, np.abs(a - b).max())


@pytest.mark.parametrize("mode", [_lib.RELAX_PLAIN, _lib.RELAX_COLD])
def test_relaxation_of_a_cell_does_not_depend_on_the_list_length(gpu, mode):
    """The listed cells are solved by groups of lanes in short lists and one
    lane each in long ones (thresholds 65,536 and 49,152): the first cells of
    a long list against the same cells alone, bit for bit, and the counts."""
    from fooskagpu_amd import surrogate
    p = dict(cases._two_phase_params(), relaxFlag=1)
    big, small = Mesh.box(38, 38, 38), Mesh.box(11, 11, 11)
    U = surrogate.uniform_states(big.n_cells, p, seed=9)
    with GpuSolver(p, big, U) as a, GpuSolver(p, small, U[:small.n_cells]) as b:
        sa, sb = a.relaxation(mode), b.relaxation(mode)
        Ua, Ub = a.download_state(), b.download_state()
    print(f"[lists] chemical cells {sa['n_chem']} / {sb['n_chem']}, fallbacks {sa['n_fallback']} / {sb['n_fallback']}")
    assert sa["n_chem"] > 65536 > 49152 > sb["n_chem"] > 0
    assert np.array_equal(Ua[:small.n_cells], Ub, equal_nan=True)


@pytest.mark.parametrize("n", [9, 25, 34, 50])
def test_states_pass_through_the_copies_unchanged(gpu, n):
    """Uploads and downloads below, between and above the sizes where they go
    through page-locked slots (5 MB down, 16 MB up; pieces of 1, 2 and 4 MB,
    the last one part full): bytes are bytes."""
    m = Mesh.box(n, n, n, rcm=False)
    U = np.random.default_rng(n).uniform(0.1, 1, (m.n_cells, 10))
    with GpuSolver(cases._two_phase_params(), m, U) as g:
        print(f"[copies] {U.nbytes} bytes", flush=True)
        assert np.array_equal(g.download_state(), U)
        g.upload_state(2 * U)
        assert np.array_equal(g.download_state(), 2 * U)


def test_copies_of_several_threads(gpu):
    """The page-locked slots are lent to one copy at a time: contexts that
    copy from several threads at once all get their own bytes."""
    import threading
    m = Mesh.box(26, 26, 26, rcm=False)
    wrong = []

    def work(k):
        U = np.full((m.n_cells, 10), float(k + 1))
        with GpuSolver(cases._two_phase_params(), m, U) as g:
            for _ in range(4):
                g.upload_state(U)
                if not np.array_equal(g.download_state(), U):
                    wrong.append(k)

    th = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not wrong


@pytest.mark.parametrize("batch", [1, 31, 33, 1057])
def test_training_step_is_adam_on_the_gradient(gpu, batch):
    """One training step on device-drawn samples (splitmix64 of the seed)
    against Adam in NumPy on fk_mlp_grad's gradient of the same samples, at
    batches that leave blocks of 32 samples and runs of 32 partials part
    full.  The step's arithmetic is FP32 with the operations of the formula:
    a few ulp (the device's square root and division, 1 ulp each) of the
    update lr = 2e-3, far below 1e-6."""
    from fooskagpu_amd import surrogate
    rng = np.random.default_rng(batch)
    n, seed = 777, 12345
    x = rng.normal(size=(n, 3)).astype(np.float32)
    y = rng.normal(size=(n, 3)).astype(np.float32)
    z = np.uint64(seed) + np.arange(1, batch + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    idx = ((z ^ (z >> np.uint64(31))) % np.uint64(n)).astype(np.int64)
    w0, norm = surrogate.init_weights(2), surrogate.fit_norm(x, y)
    with GpuSolver(cases._two_phase_params()) as g:
        sg = surrogate.Surrogate(g)
        sg.set_data(x, y)
        sg.set_weights(w0, norm)
        grad, loss = sg.grad(idx)
        l0, l1 = sg.train(1, batch=batch, lr=2e-3, seed=seed)
        w1 = sg.weights()[0]
    gr = grad.astype(np.float64)
    want = w0 - 2e-3 * gr / (np.sqrt(gr * gr) + 1e-8)  # first step: m / (1 - b1) = g, v / (1 - b2) = g^2
    print(f"[train] batch {batch}: loss {loss:.5f} {l0:.5f}, max |dw| {np.abs(w1 - want).max():.2e}")
    assert l0 == l1 == loss
    assert np.abs(w1 - want).max() < 1e-6


QUAD_CASES = {
    "sod": lambda: cases.sod(nx=7, ny=3, nz=3),
    "tgv": lambda: cases.tgv(n=7),
    "bubble": lambda: cases.bubble(n=9),
    "shock_bubble": lambda: cases.shock_bubble(n=9, nbub=3),
    "elements": lambda: _elements(_lib.MODEL_TWO_PHASE),
    "elements_sp": lambda: _elements(_lib.MODEL_SINGLE),
}


def _elements(model):
    m = Mesh.mixed_box(7, 3, 4, (0, 0, 0), (1.0, 0.4, 0.4), 0.10, 11, bc=(3, 2, 4, 5, 1, 2))
    if model == _lib.MODEL_SINGLE:
        p = dict(cases.BASE, viscFlag=1, turbulence=1, heatFlux=1, dynVisc=[1e-3, 1e-3], inletP=1.1, inletT=0.004)
        return cases.Case("elements_sp", p, m, m.init_sod(1.4, 0.0, 0.45, (1.0, 0.2, 0, 0, 1.0), (0.125, 0, 0, 0, 0.1)), 3)
    p = cases._two_phase_params(viscFlag=1, turbulence=1, inletP=1e7, inletT=cases.T_WATER)
    am = p["avfMin"]
    regions = [dict(kind=0, alphaL=1 - am, p=1e7, T=cases.T_WATER, u=(3.0, 0, 0)),
               dict(kind=1, c=(0.5, 0.2, 0.2), r=0.15, alphaL=am, p=2340.0, T=cases.T_WATER)]
    return cases.Case("elements", p, m, m.init_regions(p, regions), 3)


@pytest.mark.parametrize("precision", [_lib.FP64, _lib.MIXED])
@pytest.mark.parametrize("name", sorted(QUAD_CASES))
def test_four_lanes_per_cell_give_the_bits_of_one(gpu, name, precision):
    """Small meshes run pass G and pass F on quads (stage 1); the kernels of
    one lane per cell, with LDS (2) and without (0), give the same states and
    counts bit for bit: all stages, both relaxations fused and apart, sizes
    that leave the last wave part full, every boundary code."""
    c = QUAD_CASES[name]()
    print(f"[quads] {name} {c.mesh.n_cells} cells", flush=True)
    modes = [_lib.RELAX_PLAIN, _lib.RELAX_COLD] if c.neq == 10 else [_lib.RELAX_PLAIN]
    for mode in modes:
        for fuse in (1, 0):
            out = []
            for stage in (1, 2, 0):
                with GpuSolver(dict(c.params, precision=precision, relaxMode=mode), c.mesh, c.U) as g:
                    g.set_tuning("stage_f", stage)
                    g.set_tuning("stage_g", stage)
                    g.set_tuning("fuse_update", fuse)
                    dt = g.run_steps(3)
                    out.append((g.download_state(), dt, g.relax_totals() if c.neq == 10 else None))
            for o in out[1:]:
                assert np.array_equal(o[0], out[0][0]) and o[1:] == out[0][1:]


@pytest.mark.parametrize("precision", [_lib.FP64, _lib.MIXED])
@pytest.mark.parametrize("name", ["tgv", "shock_bubble"])
def test_workgroups_of_one_lane_per_cell_with_a_remainder(gpu, name, precision):
    """The LDS kernels at a size that fills many workgroups and leaves the last
    part full, against direct loads and stores, bit for bit."""
    c = cases.tgv(n=23) if name == "tgv" else cases.shock_bubble(n=23, nbub=5, order="morton")
    out = []
    for stage in (2, 0, 1):
        with GpuSolver(dict(c.params, precision=precision), c.mesh, c.U) as g:
            g.set_tuning("stage_f", stage)
            g.set_tuning("stage_g", stage)
            g.run_steps(2)
            out.append(g.download_state())
    assert all(np.array_equal(o, out[0]) for o in out[1:])


@pytest.mark.parametrize("stage", [1, 2, 0])
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 3, 1), (8, 4, 4), (17, 13, 11)])
def test_time_step_is_that_of_the_last_state(gpu, n, stage):
    """The step's minimum of the cells of the state at hand, whatever stages
    ran before it: a fast state, then a slow one, residuals without a time
    step in between; from a part of a wave to more waves than the words that
    hold the minima.  Against the oracle (1e-14, as for the step of one
    state), and run_steps' first dt the same."""
    m = Mesh.box(*n)
    p = dict(cases.tgv(n=4).params, cfl=0.3)
    slow = rough_state(5, m.n_cells, "random", 3)
    fast = slow * [1, 5, 5, 5, 25]
    want = []
    for U in (slow, fast):
        o = Oracle(p, m, U)
        o.compute_face_values()
        o.compute_rhs()
        want.append(o.compute_time_step())
    assert want[1] < want[0]
    with GpuSolver(p, m, fast) as g:
        g.set_tuning("stage_f", stage)

        def dt_of(U, passes=1):
            g.upload_state(U)
            g.compute_face_values()
            for _ in range(passes):
                g.compute_rhs()
            return g.compute_time_step()

        got = [dt_of(slow), dt_of(fast), dt_of(slow), dt_of(fast, 3), dt_of(slow, 2)]
        got.append(g.compute_time_step())
        print(f"[dt] {m.n_cells} cells, stage_f {stage}: {got} oracle {want}", flush=True)
        assert np.allclose(got, [want[0], want[1], want[0], want[1], want[0], want[0]], rtol=1e-14, atol=0)
        for U, dt in ((slow, got[0]), (fast, got[1]), (slow, got[0])):
            g.upload_state(U)
            g.set_clock(0.0, 0.0, 0)
            assert g.run_steps(1)[0] == dt


@pytest.mark.parametrize("kind", ["random", "uniform", "spike"])
@pytest.mark.parametrize("elements", ["tets", "mixed"])
@pytest.mark.parametrize("model", [_lib.MODEL_SINGLE, _lib.MODEL_TWO_PHASE])
def test_limiter_of_the_variants_in_mixed_precision(gpu, model, elements, kind):
    """FP32 quotients at the steepest slope of either sign (one lane per cell)
    against the smallest of a quotient at every face (four lanes): limiter and
    face states of rough states, bit for bit."""
    p = dict(cases.BASE) if model == _lib.MODEL_SINGLE else cases._two_phase_params()
    m = Mesh.box(14, 14, 14, jitter=0.1, seed=5) if elements == "tets" else Mesh.mixed_box(21, 14, 14, jitter=0.1, seed=5)
    out = []
    for stage in (1, 2, 0):
        with GpuSolver(dict(p, precision=_lib.MIXED), m, rough_state(5 if model == _lib.MODEL_SINGLE else 10, m.n_cells, kind)) as g:
            g.set_tuning("stage_g", stage)
            g.set_debug(True)
            g.compute_face_values()
            out.append((g.download("theta"), g.download("face")[g.download("slots") >= 0]))
    assert kind == "uniform" or (out[0][0] < 1).any()
    for o in out[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(o, out[0]))
