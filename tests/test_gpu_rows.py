"""The kernels that give a system several lanes (kernels_row.h) against the lane-per-system kernels and the oracle:
bit-identical states, sub-step counts and status in exact mode, at the edges of their ranges."""
import numpy as np
import pytest

import oracle_lib as O
import test_gpu_trace
from wind_amd import api
from wind_amd import networks as W

pytestmark = pytest.mark.gpu


def same(a, b):
    na, nb = np.isnan(a), np.isnan(b)
    return np.array_equal(na, nb) and np.array_equal(a[~na].view(np.uint32), b[~nb].view(np.uint32))


def run(net, n, y0, c, kernel, **kw):
    y = y0.copy()
    steps, status = np.zeros(n, np.int32), np.full(n, -1, np.int32)
    kw = {"tend": 1.0, "nfix": 1, "tol": 1e-3, **kw}
    tol = kw.pop("tol")
    total, _ = api.integrate(net, 0.0, kw.pop("tend"), kw.pop("nfix"), c, y, n, tol, kw.pop("rel", tol), kernel=kernel,
                             steps_out=steps, status_out=status, **kw)
    assert total == int(steps.astype(np.int64).sum())
    return y, steps, status


NETS = {
    "nr_test": (lambda: api.Network.builtin(api.NET_NR_TEST), lambda n: W.nr_test_systems(n, 5)[:2],
                {"tend": 1.0, "nfix": 1000}),
    "katz96": (lambda: api.Network.builtin(api.NET_KATZ96),
               lambda n: tuple(np.resize(a, n * k) for a, k in ((W.KATZ96_FIXTURE_Y, 5), (W.KATZ96_FIXTURE_C, 10))),
               {"tend": 200.0, "tol": 5e-3}),
    "hhe6": (lambda: api.Network.builtin(api.NET_HHE6, W.hhe6_params()), lambda n: W.hhe6_systems(n, 9),
             {"tend": 1e4}),
    "mixed5": (lambda: api.Network.plugin("mixed5"),
               lambda n: W.mass_action_systems(n, 5, 11, W.MIXED_SCALE_RANGE), {"tend": 1e7}),
}


@pytest.mark.parametrize("name", list(NETS))
@pytest.mark.parametrize("method", [api.SIE, api.RK2])
@pytest.mark.parametrize("controller", [api.CTRL_REFERENCE, api.CTRL_ADAPTIVE])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 67])
def test_row_kernel_equals_lane_kernel(name, method, controller, n):
    make, systems, kw = NETS[name]
    net, (y0, c) = make(), systems(n)
    kw = dict(kw, method=method, controller=controller, max_attempts=3000)
    a, b = (run(net, n, y0, c, k, **kw) for k in (api.KERNEL_LANE, api.KERNEL_AUTO))
    assert same(a[0], b[0]) and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("name,n,method,controller", [
    ("katz96", 16385, api.SIE, api.CTRL_REFERENCE), ("hhe6", 4097, api.SIE, api.CTRL_REFERENCE), ("katz96", 4097, api.RK2, api.CTRL_ADAPTIVE),
    ("hhe6", 17001, api.SIE, api.CTRL_ADAPTIVE), ("hhe6", 140001, api.RK2, api.CTRL_REFERENCE),
    ("mixed5", 70001, api.SIE, api.CTRL_REFERENCE), ("katz96", 300007, api.SIE, api.CTRL_REFERENCE)])
def test_tail_on_rows_equals_lane_kernel(name, n, method, controller):
    """Batches whose last systems the lane kernel hands over; an attempt cap that some reach."""
    make, systems, kw = NETS[name]
    net, (y0, c) = make(), systems(n)
    kw = dict(kw, method=method, controller=controller, max_attempts=60)
    a, b = (run(net, n, y0, c, k, **kw) for k in (api.KERNEL_LANE, api.KERNEL_AUTO))
    assert same(a[0], b[0]) and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


def num_cu():
    return pytest.importorskip("torch").cuda.get_device_properties(0).multi_processor_count


@pytest.mark.parametrize("name,per_cu,method,controller,cap,tol,hints", [
    ("hhe6", 17, api.SIE, api.CTRL_REFERENCE, 700, 1e-3, False),
    ("hhe6", 300, api.SIE, api.CTRL_REFERENCE, 700, 1e-3, False),
    ("hhe6", 300, api.SIE, api.CTRL_REFERENCE, 700, 1e-3, True),
    ("hhe6", 40, api.RK2, api.CTRL_REFERENCE, 1200, 1e-3, False),
    ("hhe6", 300, api.RK2, api.CTRL_ADAPTIVE, 1200, 1e-3, False),
    ("katz96", 300, api.SIE, api.CTRL_REFERENCE, 700, 1e-5, True),
    ("mixed5", 9, api.SIE, api.CTRL_ADAPTIVE, 700, 1e-6, False),
    ("mixed5", 300, api.SIE, api.CTRL_ADAPTIVE, 700, 1e-6, False),
    ("mixed5", 1400, api.SIE, api.CTRL_REFERENCE, 700, 1e-3, False)])
def test_long_systems_are_handed_over(name, per_cu, method, controller, cap, tol, hints):
    """One system in 50 goes on to the attempt cap, far beyond the attempts after which a wave may hand over, the
    others end soon: the second lane pass and the rows take the long ones over, in index order and in another start
    order, and also where the queue feeds lanes twice.  The same bits as the lane kernel alone."""
    make, systems, kw = NETS[name]
    net, n = make(), per_cu * num_cu() + 3
    y0, c = systems(n)
    N, NC = len(y0) // n, np.size(c) // n
    c = np.ravel(c).reshape(n, NC).copy()
    kw = dict(kw, method=method, controller=controller, max_attempts=cap, tol=tol)
    steps = run(net, n, y0, c.ravel(), api.KERNEL_LANE, **kw)[1]
    order = np.argsort(steps, kind="stable")
    long, short = order[-(n // 50 + 1):], order[:n // 2]
    pick = np.resize(short, n)
    pick[np.random.default_rng(1).permutation(n)[:n // 50]] = np.resize(long, n // 50)
    y0, c = y0.reshape(n, N)[pick].ravel(), c[pick].ravel()
    if hints:
        kw["cost_hint"] = steps[pick].astype(np.int32)
    a, b = (run(net, n, y0, c, k, **kw) for k in (api.KERNEL_LANE, api.KERNEL_AUTO))
    print(f"{name} n={n}: attempts {np.percentile(a[1] // 3, [0, 50, 97, 98.5, 100])}", flush=True)
    assert np.percentile(a[1] // 3, 98.5) >= 128
    assert same(a[0], b[0]) and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("name", list(NETS))
@pytest.mark.parametrize("method", [api.SIE, api.RK2])
def test_lanes_without_a_system_change_nothing(name, method):
    """Fast lane kernel: lanes that repeat another lane's system once the queue is empty store nothing; each
    system's state, sub-steps and status are those of the whole call, also where systems reach max_attempts."""
    make, systems, kw = NETS[name]
    net, n = make(), 300
    y0, c = systems(n)
    N, NC = len(y0) // n, np.size(c) // n
    kw = {**kw, "mode": api.MODE_FAST, "controller": api.CTRL_ADAPTIVE, "max_attempts": 150}
    y, steps, status = run(net, n, y0, c, api.KERNEL_AUTO, method=method, **kw)
    flat = np.ravel(c)
    for a, b in ((0, 1), (1, 4), (4, 68), (68, 133), (133, 300)):
        part = run(net, b - a, y0[a * N:b * N], flat[a * NC:b * NC], api.KERNEL_AUTO, method=method, **kw)
        assert same(part[0], y[a * N:b * N])
        assert np.array_equal(part[1], steps[a:b]) and np.array_equal(part[2], status[a:b])


@pytest.mark.parametrize("N", [1, 2, 7, 8, 9, 16, 31, 33, 40, 41, 55, 57, 63, 64])
@pytest.mark.parametrize("controller", [api.CTRL_REFERENCE, api.CTRL_ADAPTIVE])
def test_register_kernel_equals_oracle(N, controller):
    """Mass-action networks with the matrix in registers, at the edges of the sizes it is built for; a state that
    overflows, whose infinities pass through the elimination."""
    n = 5
    rx, k = W.mass_action_network(N, 300 + N, R=max(4 * N, 3) if N != 9 else 0)
    y0, sc = W.mass_action_systems(n, N, 5, W.MIXED_SCALE_RANGE)
    y0[N:2 * N] *= np.float32(1e30)
    y0[2 * N] = np.inf
    yr = y0.copy()
    _, sr, tr = O.gold_integrate(O.SIE, O.mass_action(N, rx, k), 0.0, 1e5, 1, sc, yr, n, 1e-6, 1e-4, const_stride=1,
                                 max_attempts=60, controller=controller)
    y, steps, status = run(api.Network.mass_action(N, rx, k), n, y0, sc, api.KERNEL_AUTO, tend=1e5, tol=1e-6,
                           rel=1e-4, controller=controller, max_attempts=60)
    assert same(y, yr) and np.array_equal(steps, sr) and np.array_equal(status, tr)


@pytest.mark.parametrize("N", [3, 16, 17, 33, 48, 50, 80, 96, 97, 113, 129, 157])
def test_dense_solver_results_do_not_depend_on_the_batch(N):
    """Fast dense solver: few systems run on eight waves each, many on four; the same bits."""
    n = 560
    net = api.Network.mass_action(N, *W.mass_action_network(N, 700 + N))
    y0, sc = W.mass_action_systems(n, N, 7, W.MIXED_SCALE_RANGE)
    kw = {"tend": 1e6, "tol": 1e-10, "rel": 8e-5, "mode": api.MODE_FAST, "controller": api.CTRL_ADAPTIVE,
          "max_attempts": 60}
    full = run(net, n, y0, sc, api.KERNEL_AUTO, **kw)
    for m in (1, 200, 512):
        part = run(net, m, y0[:m * N], sc[:m], api.KERNEL_AUTO, **kw)
        assert same(part[0], full[0][:m * N]) and np.array_equal(part[1], full[1][:m])


@pytest.mark.parametrize("N", [50, 80, 100, 157])
@pytest.mark.parametrize("controller", [api.CTRL_REFERENCE, api.CTRL_ADAPTIVE])
def test_dense_hand_over_continues_each_system(N, controller):
    """The last systems of a call go on on eight waves each: states, sub-steps, status and the sub-steps' total are
    those of calls that never hand over, also where systems reach max_attempts."""
    n = 600
    net = api.Network.mass_action(N, *W.mass_action_network(N, 700 + N))
    y0, sc = W.mass_action_systems(n, N, 7, W.MIXED_SCALE_RANGE)
    kw = {"tend": 1e6, "tol": 1e-10, "rel": 8e-5, "mode": api.MODE_FAST, "controller": controller,
          "max_attempts": 700}
    y, steps, status = run(net, n, y0, sc, api.KERNEL_AUTO, **kw)
    print(f"N={N} attempts {steps.min() // 3} .. {steps.max() // 3}", flush=True)
    for i in range(0, n, 200):
        part = run(net, 200, y0[i * N:(i + 200) * N], sc[i:i + 200], api.KERNEL_AUTO, **kw)
        assert same(part[0], y[i * N:(i + 200) * N])
        assert np.array_equal(part[1], steps[i:i + 200]) and np.array_equal(part[2], status[i:i + 200])


@pytest.mark.parametrize("N", [5, 16, 33, 40, 48])
def test_dense_solver_attempts_at_few_tiles(N):
    """Register-resident dense solver at one and three tiles per dimension: per attempt against the float
    oracle, with the bounds of the other sizes."""
    test_gpu_trace.test_fast_dense_attempts(N, 16, 200, 0)


def test_row_kernel_strides_hints_and_non_finite_states():
    net, n = api.Network.builtin(api.NET_HHE6, W.hhe6_params()), 129
    y0, c = W.hhe6_systems(n, 21)
    y0[6 * 7 + 5] = np.inf
    y0[6 * 8 + 1] = np.nan
    y0[6 * 9:6 * 10] = 3e38
    wide = np.full(3 * n, 7.0, np.float32)
    wide[::3] = c
    kw = {"tend": 1e3, "max_attempts": 500, "tol": 1e-3}
    ref = run(net, n, y0, c, api.KERNEL_LANE, **kw)
    hint = np.random.default_rng(0).integers(1, 1000, n).astype(np.int32)
    for extra in ({"const_stride": 3}, {"cost_hint": hint}):
        got = run(net, n, y0, wide if "const_stride" in extra else c, api.KERNEL_AUTO, **kw, **extra)
        assert same(ref[0], got[0]) and np.array_equal(ref[1], got[1]) and np.array_equal(ref[2], got[2])


@pytest.mark.parametrize("tiles", [4, 5, 50])
@pytest.mark.parametrize("method", [O.SIE, O.RK2])
@pytest.mark.parametrize("controller", [api.CTRL_REFERENCE, api.CTRL_ADAPTIVE])
def test_tiled_network_equals_oracle_also_where_a_tile_overflows(tiles, method, controller):
    """A tile whose state overflows: in the dense elimination its infinities reach the other tiles' equations."""
    n, N, name = 4, 5 * tiles, f"katz96_t{tiles}"
    c = W.KATZ96_FIXTURE_C.copy()
    y0 = np.tile(W.KATZ96_FIXTURE_Y.reshape(4, 5), (1, tiles)).astype(np.float32)
    rng = np.random.default_rng(tiles)
    y0 *= rng.uniform(0.5, 1.5, y0.shape).astype(np.float32)  # tiles that differ
    y0[1, 5 * (tiles - 1) + 1] = 3e38
    y0[2, 5 * (tiles // 2)] = np.inf
    y0 = y0.reshape(-1)
    yr = y0.copy()
    tend = 0.5
    _, sr, tr = O.gold_integrate(method, O.generated(name), 0.0, tend, 1, c, yr, n, 5e-3, 5e-3, const_stride=10,
                                 max_attempts=40, controller=controller)
    y, steps, status = run(api.Network.plugin(name), n, y0, c, api.KERNEL_AUTO, tend=tend, tol=5e-3, method=method,
                           controller=controller, max_attempts=40)
    if method == O.SIE and controller == api.CTRL_REFERENCE:
        assert np.isnan(yr.reshape(n, N)[2]).sum() > 5  # it does reach them
    assert same(y, yr) and np.array_equal(steps, sr) and np.array_equal(status, tr)


def test_explicit_tiles_on_both_sides_of_their_limit():
    """RK2 on a tiled network whose matrices are beyond LDS: the tile kernel up to a system per CU, the block kernel
    above, the same bits."""
    tiles = 50
    N, n = 5 * tiles, num_cu() + 1
    rng = np.random.default_rng(tiles)
    y0 = np.tile(np.resize(W.KATZ96_FIXTURE_Y, 5 * n).reshape(n, 5), (1, tiles))
    y0 = (y0 * rng.uniform(0.5, 1.5, y0.shape)).astype(np.float32).reshape(-1)
    c = np.resize(W.KATZ96_FIXTURE_C, 10 * n).astype(np.float32)
    kw = {"tend": 0.5, "tol": 5e-3, "method": api.RK2, "max_attempts": 20}
    net = api.Network.plugin(f"katz96_t{tiles}")
    y, steps, status = run(net, n, y0, c, api.KERNEL_AUTO, **kw)
    part = run(net, n - 1, y0[:-N], c[:-10], api.KERNEL_AUTO, **kw)
    assert same(part[0], y[:-N]) and np.array_equal(part[1], steps[:-1]) and np.array_equal(part[2], status[:-1])


@pytest.mark.parametrize("n", [1, 3, 32000, 33500])
def test_host_arrays_equal_device_arrays(n):
    """Host-pointer calls on both sides of the staging limit (1 MiB; 32 bytes a system here), outputs optional."""
    torch = pytest.importorskip("torch")
    net = api.Network.builtin(api.NET_NR_TEST)
    y0, c, _ = W.nr_test_systems(n, 3)
    y, steps, status = run(net, n, y0, c, api.KERNEL_AUTO, nfix=1000)
    d, dc = torch.from_numpy(y0).cuda(), torch.from_numpy(c).cuda()
    torch.cuda.synchronize()
    total, _ = api.integrate(net, 0.0, 1.0, 1000, dc, d, n, 1e-3, 1e-3, device_pointers=True)
    assert total == int(steps.astype(np.int64).sum()) and np.all(status == 0)
    assert same(y, d.cpu().numpy())
    bare = y0.copy()
    assert api.integrate(net, 0.0, 1.0, 1000, c, bare, n, 1e-3, 1e-3)[0] == total and same(bare, y)
