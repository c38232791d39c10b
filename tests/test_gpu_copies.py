"""Large host copies where several of their parts meet: slots that one copy
fills more than once, consecutive copies of different contents, contexts that
copy from several threads at once."""
import threading

import numpy as np
import pytest

from fooskagpu_amd import GpuSolver, Mesh, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [33, 53, 60])
def test_consecutive_copies_fill_the_slots_again(gpu, n):
    """17 MB in 2 MB pieces, 71 and 104 MB in 4 MB pieces (the last part full,
    the largest through every slot more than once): each copy brings its own
    bytes, none of the copy before."""
    m = Mesh.box(n, n, n, rcm=False)
    U = np.random.default_rng(n).uniform(0.1, 1, (m.n_cells, 10))
    print(f"[copies] {U.nbytes} bytes", flush=True)
    with GpuSolver(cases._two_phase_params(), m, U) as g:
        for k in range(5):
            g.upload_state(U + k)
            assert np.array_equal(g.download_state(), U + k)


def test_uploads_of_several_threads(gpu):
    """Three contexts, each with uploads and downloads large enough for the
    slots (17 MB), at the same time."""
    m = Mesh.box(33, 33, 33, rcm=False)
    wrong = []

    def work(k):
        U = np.full((m.n_cells, 10), float(k + 1))
        assert U.nbytes > 16 << 20
        with GpuSolver(cases._two_phase_params(), m, U) as g:
            for i in range(4):
                g.upload_state(U + 10 * i)
                if not np.array_equal(g.download_state(), U + 10 * i):
                    wrong.append((k, i))

    th = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not wrong


@pytest.mark.parametrize("n", [450001, 450002, 450003])
def test_labels_and_predictions_of_odd_counts(gpu, n):
    """Features, targets and predictions large enough for the slots (5.4 MB)
    that lie behind each other on the device and end between 16-byte words:
    the same rows as in calls of a third."""
    from fooskagpu_amd import surrogate
    p = cases._two_phase_params()
    U = surrogate.uniform_states(n, p, seed=n)
    with GpuSolver(p) as g:
        sg = surrogate.Surrogate(g)
        print(f"[copies] {n} states", flush=True)
        x, y = sg.label(U)
        ok = surrogate.finite(x, y)
        sg.set_weights(surrogate.init_weights(1), surrogate.fit_norm(*ok))
        x = np.nan_to_num(x, posinf=0, neginf=0)
        pred = sg.infer(x)
        part = [slice(0, n // 3), slice(n // 3, 2 * n // 3), slice(2 * n // 3, n)]
        xs, ys = zip(*[sg.label(U[s]) for s in part])
        assert np.array_equal(np.nan_to_num(np.concatenate(xs), posinf=0, neginf=0), x)
        assert np.array_equal(np.concatenate(ys), y, equal_nan=True)
        assert np.array_equal(np.concatenate([sg.infer(x[s]) for s in part]), pred)
