"""Block responses (T steps at a time): shapes at the edges of their tiles and
of their rule against the FP64 oracle, and the same calls with the kernel
switch that keeps the general path, including samples that are not finite."""
import numpy as np
import pytest

import oracle as orc
from parode_amd import api, synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

BAR = {api.PLAIN32: 1e-5, api.MIXED: 1e-6, api.FP64: 1e-7}


def _plan(s, U, precision, states=False, general=False):
    dev = "cuda:0"
    t = [torch.from_numpy(np.ascontiguousarray(v)).to(dev) for v in (s.A, s.B, s.C, s.D, s.x0, U)]
    p = s.n if states else s.p
    y = torch.full((s.steps, p), 7.0, dtype=torch.float32, device=dev)
    ptr = [v.data_ptr() for v in t] + [y.data_ptr()]
    if states:
        ptr[2] = ptr[3] = 0
    api.set_level_kernel(api.NO_CHUNKS if general else 0)
    try:
        plan = api.Plan(s.method, s.n, s.m, p, states, states, s.steps, s.h, precision,
                        U.dtype == np.float64)
        plan.execute(*ptr)
        torch.cuda.synchronize()
        plan.close()
    finally:
        api.set_level_kernel(0)
    return y.cpu().numpy()


def _oracle(s, U, states):
    f = lambda a: a.astype(np.float64)
    C, D = (np.eye(s.n), np.zeros((s.n, s.m))) if states else (f(s.C), f(s.D))
    return orc.simulate_f64(s.method, f(s.A), f(s.B), C, D, f(s.x0), U, s.steps, s.h)


@pytest.mark.parametrize("method,n,m,p,steps", [
    (0, 1, 1, 1, 64), (0, 2, 3, 5, 65), (0, 15, 1, 17, 513), (0, 16, 16, 16, 1024),
    (0, 17, 31, 33, 2049), (0, 63, 32, 2, 777), (0, 64, 32, 64, 9001), (0, 64, 1, 1, 70001),
    (0, 65, 33, 9, 1500), (0, 5, 2, 3, 300007),
    (1, 1, 1, 1, 67), (1, 4, 2, 1, 131), (1, 15, 32, 64, 1030), (1, 16, 7, 15, 40003),
    (1, 17, 3, 2, 600), (1, 3, 5, 4, 270001),
    # maps made by products over many work-groups
    (0, 96, 40, 70, 1100), (0, 128, 16, 16, 20000), (0, 130, 1, 1, 64), (0, 200, 25, 7, 3001),
    (1, 33, 4, 4, 7000), (1, 64, 8, 8, 30003), (1, 129, 5, 9, 2500)])
@pytest.mark.parametrize("precision", [api.PLAIN32, api.MIXED, api.FP64])
def test_block_shapes_meet_the_bars(method, n, m, p, steps, precision):
    s = synth.make_system(method, n, m, p, -5.0, -0.1, 1e-3, steps, seed=31 * n + steps,
                          noise_sigma=0.1)
    U = synth.samples_f64(s)
    if precision == api.PLAIN32:
        U = U.astype(np.float32)
        ye = orc.simulate_mirror_exact(method, s.A, s.B, s.C, s.D, s.x0, s.t0, s.t_end, s.h,
                                       Uhalf=U)
    else:
        ye = _oracle(s, U, False)
    err = orc.max_rel_err(_plan(s, U, precision), ye)
    print(f"max rel err {err:.3e}")
    assert err <= BAR[precision]


@pytest.mark.parametrize("method,n,steps", [(0, 1, 64), (0, 48, 5001), (0, 64, 999), (0, 70, 3000), (1, 16, 2500), (1, 20, 1500),
                                            (1, 5, 100)])
def test_states_as_outputs(method, n, steps):
    s = synth.make_system(method, n, 3, 2, -5.0, -0.1, 1e-3, steps, seed=9 * n)
    U = synth.samples_f64(s)
    y = _plan(s, U, api.MIXED, states=True)
    assert orc.max_rel_err(y, _oracle(s, U, True)) <= 1e-6


@pytest.mark.parametrize("method,n,m,p,steps,row", [
    (0, 6, 2, 3, 2000, 1501), (0, 6, 2, 3, 2000, 0), (0, 40, 3, 40, 60000, 77777), (0, 80, 3, 5, 9000, 8191), (1, 40, 2, 3, 9000, 8190),
    (1, 8, 2, 3, 3000, 2466), (1, 12, 1, 30, 40000, 40404)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_a_sample_that_is_not_finite_reaches_only_what_depends_on_it(method, n, m, p, steps, row,
                                                                     value):
    s = synth.make_system(method, n, m, p, -5.0, -0.1, 1e-3, steps, seed=n + row)
    U = synth.samples_f64(s)
    U[row, m - 1] = value
    y = _plan(s, U, api.MIXED)
    yg = _plan(s, U, api.MIXED, general=True)
    ok = np.isfinite(yg).all(axis=1)
    np.testing.assert_array_equal(np.isfinite(y).all(axis=1), ok)
    k = int(ok.sum())
    assert ok[:k].all()
    if k:
        assert orc.max_rel_err(y[:k], yg[:k].astype(np.float64)) <= 2e-6
