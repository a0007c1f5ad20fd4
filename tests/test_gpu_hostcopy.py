"""Results that leave in pieces equal the same results fetched a few at a time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [255, 256, 257, 700])
def test_large_results_equal_small_ones(gpu, n):
    """64^2 frames of 16 KiB around the 4 MiB from which the copy is shared out, and to odd ends."""
    from ptychopy_amd._engine import Engine
    g = np.random.default_rng(n)
    m = 64
    obj = (g.normal(size=(150, 170)) + 1j * g.normal(size=(150, 170))).astype(np.complex64)
    probe = (g.normal(size=(m, m)) + 1j * g.normal(size=(m, m))).astype(np.complex64)
    pos = g.uniform(1, 80, size=(n, 2)).astype(np.float32)
    with Engine(n, m, (150, 170)) as e:
        whole = e.simulate(obj, probe, pos)
        for i in range(0, n, 100):
            assert np.array_equal(whole[i:i + 100], e.simulate(obj, probe, pos[i:i + 100]))


@pytest.mark.parametrize("n", [1, 3, 4, 5, 131])
def test_predictions_of_many_batches_equal_those_of_one(gpu, n):
    """A single short batch, a whole one, one sample more, and more batches than are held at once."""
    from ptychopy_amd.warmstart import Net
    x = np.random.default_rng(n).uniform(0, 50, size=(n, 64, 64)).astype(np.float32)
    with Net(64, c=8, batch=4, seed=3) as net:
        for f in (net.predict, net.predict_amplitudes):
            whole = f(x)
            for i in range(0, n, 4):
                assert np.array_equal(whole[i:i + 4], f(x[i:i + 4]))


@pytest.mark.parametrize("m,rows,cols", [(256, 456, 456), (256, 457, 301), (128, 481, 487), (512, 700, 700)])
def test_frames_simulated_together_equal_single_ones(gpu, m, rows, cols):
    """Buffers in one allocation or in two, objects of odd sizes among them."""
    from ptychopy_amd._engine import Engine
    g = np.random.default_rng(rows + cols)
    obj = (g.normal(size=(rows, cols)) + 1j * g.normal(size=(rows, cols))).astype(np.complex64)
    probe = (g.normal(size=(m, m)) + 1j * g.normal(size=(m, m))).astype(np.complex64)
    pos = (g.uniform(0, 1, size=(12, 2)) * (rows - m, cols - m)).astype(np.float32)
    with Engine(1, m, (rows, cols)) as e:
        whole = e.simulate(obj, probe, pos)
        for i in range(len(pos)):
            assert np.array_equal(whole[i:i + 1], e.simulate(obj, probe, pos[i:i + 1]))
