"""Solves that diverge until the powers of their step map leave the FP64 range:
the outputs before that are those of the FP64 recurrence, at every width of the
block scan, with groups of blocks and without, and for maps of many work-groups."""
import numpy as np
import pytest

import oracle as orc
from parode_amd import api, synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# each output against the largest one so far: the bars of the stable solves
BAR = {api.PLAIN32: 1e-5, api.MIXED: 1e-6, api.FP64: 1e-7}


def _system(method, n, m, p, growth, steps):
    """One mode grows by about e^growth a step, the others decay."""
    s = synth.make_system(method, n, m, p, -0.5, -0.01, 1.0, steps, seed=n + steps)
    rng = np.random.default_rng(n)
    Q = synth._orthogonal(rng, n)
    lam = np.concatenate([[growth], rng.uniform(-0.5, -0.01, n - 1)])
    s.A = np.ascontiguousarray((Q * lam) @ Q.T, dtype=np.float32)
    return s


def _solve(s, U, precision):
    t = [torch.from_numpy(np.ascontiguousarray(v)).to("cuda:0")
         for v in (s.A, s.B, s.C, s.D, s.x0, U)]
    y = torch.zeros((s.steps, s.p), dtype=torch.float32, device="cuda:0")
    plan = api.Plan(s.method, s.n, s.m, s.p, 0, 0, s.steps, s.h, precision, U.dtype == np.float64)
    plan.execute(*[v.data_ptr() for v in t], y.data_ptr())
    torch.cuda.synchronize()
    plan.close()
    return y.cpu().numpy()


@pytest.mark.parametrize("method,n,m,p,growth,steps", [
    # the widths of the scan: 16, 32, 48 and 64 states
    (0, 1, 1, 1, 0.5, 4096), (0, 3, 2, 2, 0.5, 4096), (0, 24, 3, 2, 0.5, 4096),
    (0, 40, 3, 2, 0.5, 4096), (0, 60, 3, 3, 0.5, 4096), (0, 64, 3, 3, 0.5, 4096),
    (1, 4, 2, 2, 0.5, 4096), (1, 16, 2, 2, 0.5, 4096),
    # a step chosen too large: the RK4 factor of -5 is 13.7, of -60 5e5 (the powers
    # overflow inside a block)
    (0, 3, 2, 2, -5.0, 4096), (0, 3, 2, 2, -60.0, 200000), (0, 40, 2, 2, -60.0, 200000),
    (0, 70, 2, 2, -60.0, 200000),
    # blocks in groups
    (0, 3, 1, 2, 0.02, 131072), (0, 60, 1, 2, 0.02, 131072), (1, 5, 1, 2, 0.02, 131072),
    # maps made by products over many work-groups
    (0, 70, 3, 3, 0.5, 4096), (1, 20, 2, 2, 0.5, 4096)])
@pytest.mark.parametrize("precision", [api.PLAIN32, api.MIXED, api.FP64])
def test_outputs_before_the_overflow_are_right(method, n, m, p, growth, steps, precision):
    s = _system(method, n, m, p, growth, steps)
    U = synth.samples_f64(s)
    if precision == api.PLAIN32:
        U = U.astype(np.float32)
    with np.errstate(all="ignore"):
        if precision == api.PLAIN32:
            ye = orc.simulate_mirror_exact(method, s.A, s.B, s.C, s.D, s.x0, s.t0, s.t_end, s.h,
                                           Uhalf=U)
        else:
            f = lambda a: a.astype(np.float64)
            ye = orc.simulate_f64(method, f(s.A), f(s.B), f(s.C), f(s.D), f(s.x0), U, steps, s.h)
        ye = np.asarray(ye, np.float64)
        within = (np.abs(ye) < 1e38).all(axis=1)   # (float outputs)
    k = int(np.argmin(within))
    assert 0 < k < steps and within[:k].all()
    y = _solve(s, U, precision)[:k]
    assert np.isfinite(y).all()
    top = np.maximum.accumulate(np.abs(ye[:k]).max(axis=1))[:, None]
    err = (np.abs(y - ye[:k]) / top).max()
    print(f"{k} outputs before the overflow, max rel err {err:.3e}")
    assert err <= BAR[precision]
