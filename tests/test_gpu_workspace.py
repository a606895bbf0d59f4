"""The C ABI's simulations share one device workspace and pinned staging: outputs
that come back in several pieces, batches whose states are carried, systems
larger than the workspace, calls of other shapes between, two threads."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import oracle as orc
from parode_amd import api, synth

pytestmark = pytest.mark.gpu

BAR = 1e-7   # FP64 mode: one rounding of the outputs to float (6e-8)


@pytest.fixture(scope="module", autouse=True)
def gpu():
    ids, e = api.get_available_gpus()
    assert e == 0 and ids, "no GPU visible"
    assert api.initialize_selected_gpus(ids[:1]) == 0
    api.set_precision(api.FP64)
    api.set_max_batch_steps(0)
    yield
    api.set_precision(api.PLAIN32)
    api.set_max_batch_steps(0)
    api.close_gpu()


def _run(s, U):
    tv, y, e = api.simulate_ode_sampled(s.method, s.A, s.B, s.C, s.D, U, s.t0, s.t_end, s.h, s.x0)
    assert e == 0, api.last_error_message()
    return y


# method, n, m, p, points, batch (0: one)
CASES = [(0, 2, 1, 4, 300007, 0), (1, 3, 2, 5, 150001, 0), (0, 80, 2, 70, 9001, 2048),
         (1, 40, 3, 2, 5003, 1024), (1, 4, 1, 1, 4, 0), (0, 1, 1, 1, 1, 0),
         (0, 20, 40, 3, 500001, 0)]


def _case(method, n, m, p, points, seed):
    s = synth.make_system(method, n, m, p, -5.0, -0.1, 1e-3, points, seed=seed, noise_sigma=0.1)
    return s, synth.samples_f64(s)


@pytest.mark.parametrize("method,n,m,p,points,batch", CASES)
def test_outputs_through_the_shared_memory(method, n, m, p, points, batch):
    s, U = _case(method, n, m, p, points, 17 + points)
    api.set_max_batch_steps(batch)
    try:
        y = _run(s, U)
    finally:
        api.set_max_batch_steps(0)
    f = lambda a: a.astype(np.float64)
    ye = orc.simulate_f64(method, f(s.A), f(s.B), f(s.C), f(s.D), f(s.x0), U, points, s.h)
    assert np.abs(y - ye).max() <= BAR * np.abs(ye).max()


def test_other_calls_between_and_beside():
    made = [_case(*c[:5], seed=3 + i) for i, c in enumerate(CASES[:6])]
    first = [_run(s, U) for s, U in made]
    for (s, U), y in zip(reversed(made), reversed(first)):
        np.testing.assert_array_equal(_run(s, U), y)
    with ThreadPoolExecutor(2) as pool:
        for y, z in zip(first * 2, pool.map(lambda c: _run(*c), made * 2)):
            np.testing.assert_array_equal(z, y)
