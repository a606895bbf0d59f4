"""The ABM start-up at the edges of its splits over lanes: the first states of a
solve against the oracle's three RK4 steps, bit for bit in the reference's float
rounding."""
import numpy as np
import pytest

import oracle as orc
from parode_amd import api, synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,m", [(1, 1), (3, 5), (4, 4), (5, 1), (15, 32), (16, 3), (17, 2), (63, 9),
                                 (64, 1), (65, 4), (128, 17), (129, 3), (255, 33), (256, 256)])
@pytest.mark.parametrize("points", [4, 70])
@pytest.mark.parametrize("precision", [api.PLAIN32, api.FP64])
def test_first_states(n, m, points, precision):
    s = synth.make_system(1, n, m, 1, -5.0, -0.1, 1e-2, points, seed=7 * n + m)
    U = synth.samples_f64(s)
    if precision == api.PLAIN32:
        U = U.astype(np.float32)
        X = orc.abm_startup_f32(s.A, s.B, s.x0, U[:7], s.h)
    else:
        f = lambda a: a.astype(np.float64)
        X = orc.abm_startup_f64(f(s.A), f(s.B), f(s.x0), U[:7], s.h)
    t = [torch.from_numpy(np.ascontiguousarray(v)).to("cuda:0") for v in (s.A, s.B, s.x0, U)]
    y = torch.zeros((points, n), dtype=torch.float32, device="cuda:0")
    plan = api.Plan(1, n, m, n, 1, 1, points, s.h, precision, U.dtype == np.float64)
    plan.execute(t[0].data_ptr(), t[1].data_ptr(), 0, 0, t[2].data_ptr(), t[3].data_ptr(),
                 y.data_ptr())
    torch.cuda.synchronize()
    plan.close()
    got, ye = y.cpu().numpy()[:3], np.asarray(X, np.float64).reshape(4, n)[:3]
    if precision == api.PLAIN32:
        np.testing.assert_array_equal(got, ye.astype(np.float32))
    else:   # one rounding to float
        assert (np.abs(got - ye) <= 2.0 ** -23 * np.abs(ye) + 1e-12).all()
