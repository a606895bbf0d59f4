"""The general path (the tree of scan levels with its chunk recurrences, leaves and
output kernels), which short horizons, systems without inputs and outputs without
states take, and every system under a kernel switch: grouped launches and single
plans against the FP64 recurrence, since systems with inputs, outputs and 64 points
or more run as block responses otherwise."""
import numpy as np
import pytest

# torch before the library starts the HIP runtime (its own start-up then finds the GPU)
torch = pytest.importorskip("torch")

import oracle as orc  # noqa: E402
from parode_amd import api, synth  # noqa: E402
from test_gpu_batch import SHAPES, _serve, _systems  # noqa: E402

pytestmark = pytest.mark.gpu

BAR = {api.PLAIN32: 1e-5, api.MIXED: 1e-6, api.FP64: 1e-7}


@pytest.fixture(scope="module", autouse=True)
def gpu():
    ids, e = api.get_available_gpus()
    assert e == 0 and ids, "no GPU visible"
    assert api.initialize_selected_gpus(ids[:1]) == 0
    yield
    api.close_gpu()


@pytest.fixture
def switch():
    yield api.set_level_kernel
    api.set_level_kernel(0)


def _f64(s):
    f = lambda a: a.astype(np.float64)
    return orc.simulate_f64(s.method, f(s.A), f(s.B), f(s.C), f(s.D), f(s.x0),
                            synth.samples_f64(s), s.steps, s.h)


def _cut(s, points):
    s.steps = min(s.steps, points)
    return s


def _check_group(systems):
    ys, gs = _serve(systems)
    assert gs["grouped_requests"] == len(systems)
    for s, y in zip(systems, ys):
        err = orc.max_rel_err(y, _f64(s))
        print(f"{'ABM' if s.method else 'RK4'} n={s.n} N={s.steps}: {err:.3e}")
        assert err <= BAR[api.MIXED], (s.method, s.n, s.steps, err)


@pytest.mark.parametrize("points", [4, 5, 17, 63])
def test_grouped_short_horizons(points):
    """Fewer than 64 points: the grouped tree, leaves and outputs of every width."""
    _check_group([_cut(s, points) for s in _systems()])


def test_grouped_tree_of_every_width(switch):
    """The switch that takes every level as a tree level (grouped up to 8192 points)."""
    switch(api.NO_CHUNKS)
    _check_group([_cut(s, 8192) for s in _systems()])


def test_grouped_outputs_without_states():
    """D without C: y = D u, beside systems that run as block responses."""
    systems = _systems()
    need = sum(api.Server.footprint(s.method, s.n, s.m, s.p, s.steps) for s in systems)
    srv = api.Server(lanes=4, device_bytes=int(need * 1.2) + (256 << 20), pinned_bytes=512 << 20,
                     precision=api.MIXED)
    try:
        got = [srv.submit(s.method, s.A, s.B, s.C if k % 3 == 2 else None, s.D, s.x0, s.steps, s.h,
                          coef=s.ucoef) for k, s in enumerate(systems)]
        for t, _ in got:
            assert srv.wait(t)[0] == 0
        gs = srv.group_stats()
    finally:
        srv.close()
    assert gs["grouped_requests"] == len(systems)
    for k, (s, (_, y)) in enumerate(zip(systems, got)):
        ye = (_f64(s) if k % 3 == 2 else
              synth.samples_f64(s)[:2 * s.steps:2] @ s.D.T.astype(np.float64))
        assert orc.max_rel_err(y, ye) <= BAR[api.MIXED], (s.method, s.n, s.steps)


def _plan(s, U, precision, m=None):
    m = s.m if m is None else m
    t = [torch.from_numpy(np.ascontiguousarray(v)).to("cuda:0")
         for v in (s.A, s.B, s.C, s.D, s.x0, U)]
    ptr = [v.data_ptr() for v in t]
    y = torch.zeros((s.steps, s.p), dtype=torch.float32, device="cuda:0")
    if m == 0:
        ptr[1] = ptr[3] = ptr[5] = 0
    plan = api.Plan(s.method, s.n, m, s.p, 0, 1 if m == 0 else 0, s.steps, s.h, precision,
                    U.dtype == np.float64)
    plan.execute(*ptr, y.data_ptr())
    torch.cuda.synchronize()
    plan.close()
    return y.cpu().numpy()


@pytest.mark.parametrize("k", range(len(SHAPES)))
def test_chunk_recurrences_of_every_width(switch, k):
    """The chunk recurrences with their outputs, the power table on the vector ALUs."""
    s = _systems()[k]
    switch(api.VECTOR_GEMM)
    y = _plan(s, synth.samples_f64(s), api.MIXED)
    assert orc.max_rel_err(y, _f64(s)) <= BAR[api.MIXED]


@pytest.mark.parametrize("method,n,p,steps", [(0, 1, 1, 70), (0, 8, 3, 5000), (0, 50, 5, 20000),
                                              (0, 130, 4, 3000), (1, 5, 2, 3000), (1, 70, 4, 9000)])
@pytest.mark.parametrize("precision", [api.PLAIN32, api.MIXED, api.FP64])
def test_systems_without_inputs(method, n, p, steps, precision):
    s = synth.make_system(method, n, 1, p, -5.0, -0.1, 1e-3, steps, seed=n)
    y = _plan(s, np.zeros((2 * steps + 1, 1)), precision, m=0)
    f = lambda a: a.astype(np.float64)
    if precision == api.PLAIN32:
        ye = orc.simulate_mirror_exact(method, s.A, 0 * s.B, s.C, 0 * s.D, s.x0, 0.0, s.t_end, s.h,
                                       Uhalf=np.zeros((2 * steps + 1, 1), np.float32))
    else:
        ye = orc.simulate_f64(method, f(s.A), 0 * f(s.B), f(s.C), 0 * f(s.D), f(s.x0),
                              np.zeros((2 * steps + 1, 1)), steps, s.h)
    assert orc.max_rel_err(y, ye) <= BAR[precision]
