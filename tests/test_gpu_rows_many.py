"""Kernels that carry a workgroup or a wave on to its next system: more systems than the device holds at once, against
calls small enough that none is reused, bit for bit; hand-overs from several threads at once."""
import os
import threading

import numpy as np
import pytest

from test_gpu_rows import NETS, num_cu, run, same
from wind_amd import api
from wind_amd import networks as W

pytestmark = pytest.mark.gpu


def equal_in_parts(net, n, part, y0, c, **kw):
    """The whole call against calls of `part` systems."""
    N, NC = len(y0) // n, len(c) // n
    y, steps, status = run(net, n, y0, c, api.KERNEL_AUTO, **kw)
    for a in range(0, n, part):
        b = min(n, a + part)
        got = run(net, b - a, y0[a * N:b * N], c[a * NC:b * NC], api.KERNEL_AUTO, **kw)
        assert same(got[0], y[a * N:b * N]), a
        assert np.array_equal(got[1], steps[a:b]) and np.array_equal(got[2], status[a:b]), a
    return y, steps


@pytest.mark.parametrize("N,per_cu", [(3, 40), (8, 40), (33, 24), (64, 24)])  # at most 16 workgroups of 128 per CU
def test_register_kernel_takes_system_after_system(N, per_cu):
    n = per_cu * num_cu() + 1
    rx, k = W.mass_action_network(N, 300 + N)
    y0, sc = W.mass_action_systems(n, N, 5, W.MIXED_SCALE_RANGE)
    y0 = y0.reshape(n, N)
    y0[::97] *= np.float32(1e30)
    y0[::193, 0] = np.inf
    equal_in_parts(api.Network.mass_action(N, rx, k), n, num_cu(), y0.ravel(), sc, tend=1e5, tol=1e-6, rel=1e-4,
                   controller=api.CTRL_ADAPTIVE, max_attempts=12)


@pytest.mark.parametrize("tiles,per_cu", [(4, 70), (20, 9)])  # at most 32 waves per CU
@pytest.mark.parametrize("controller", [api.CTRL_REFERENCE, api.CTRL_ADAPTIVE])
def test_tile_kernel_takes_system_after_system(tiles, per_cu, controller):
    """Also after a system that went through the dense form."""
    N, n = 5 * tiles, per_cu * num_cu() + 1
    rng = np.random.default_rng(tiles)
    y0 = np.tile(np.resize(W.KATZ96_FIXTURE_Y, 5 * n).reshape(n, 5), (1, tiles))
    y0 = (y0 * rng.uniform(0.5, 1.5, y0.shape)).astype(np.float32)
    y0[::211, 5 * (tiles - 1) + 1] = 3e38
    y0[100::401, 5 * (tiles // 2)] = np.inf
    c = np.resize(W.KATZ96_FIXTURE_C, 10 * n).astype(np.float32)
    y, _ = equal_in_parts(api.Network.plugin(f"katz96_t{tiles}"), n, num_cu(), y0.ravel(), c, tend=0.5, tol=5e-3,
                          controller=controller, max_attempts=6)
    if controller == api.CTRL_REFERENCE:  # (the adaptive controller rejects the steps that make them)
        assert np.isnan(y.reshape(n, N)[100::401]).any()


@pytest.mark.parametrize("N", [50, 100, 157])
def test_dense_hand_over_from_the_smallest_batch_that_does(N):
    """One system more than the eight-wave form takes, and as many again as that."""
    few = (1 if N <= 80 else 2) * num_cu()
    net = api.Network.mass_action(N, *W.mass_action_network(N, 700 + N))
    for n in (few + 1, 2 * few + 1):
        y0, sc = W.mass_action_systems(n, N, 7, W.MIXED_SCALE_RANGE)
        equal_in_parts(net, n, few // 2, y0, sc, tend=1e6, tol=1e-10, rel=8e-5, mode=api.MODE_FAST,
                       controller=api.CTRL_ADAPTIVE, max_attempts=300)


@pytest.mark.parametrize("method", [api.SIE, api.RK2])
@pytest.mark.parametrize("controller", [api.CTRL_REFERENCE, api.CTRL_ADAPTIVE])
@pytest.mark.parametrize("per_cu", [0, 16, 20, 300])
def test_eight_equations_on_rows(method, controller, per_cu):
    """The largest network that rows take: small batches, the largest that is rows throughout, and hand-overs with
    and without the second lane pass, against the lane kernel."""
    net, n = api.Network.plugin("mass_action8"), per_cu * num_cu() + (5 if per_cu != 16 else 0)
    y0, c = W.mass_action_systems(n, 8, 11, W.MIXED_SCALE_RANGE)
    kw = {"tend": 1e7, "tol": 1e-8, "rel": 1e-4, "method": method, "controller": controller, "max_attempts": 700}
    a, b = (run(net, n, y0, c, k, **kw) for k in (api.KERNEL_LANE, api.KERNEL_AUTO))
    assert same(a[0], b[0]) and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


def test_plugin_that_does_not_know_the_grown_arguments(tmp_path):
    """A plugin file without the entry that tells it of them reads the part it knows: the same bits, no hand-over."""
    built = os.path.join(os.path.dirname(api.LIB_PATH), "gen", "mixed5", "libwind_net.so")
    with open(built, "rb") as f:
        body = f.read()
    assert body.count(b"\0wind_plugin_args2\0") >= 1
    old = tmp_path / "libwind_net.so"
    old.write_bytes(body.replace(b"\0wind_plugin_args2\0", b"\0wind_plugin_argsX\0"))
    make, systems, kw = NETS["mixed5"]
    n = 20 * num_cu() + 3
    y0, c = systems(n)
    kw = {**kw, "max_attempts": 300}
    a = run(make(), n, y0, c, api.KERNEL_AUTO, **kw)
    b = run(api.Network.plugin(str(old)), n, y0, c, api.KERNEL_AUTO, **kw)
    assert same(a[0], b[0]) and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


def test_hand_overs_of_several_threads_at_once():
    """Each call has its own lists: exact and dense hand-overs, rows and lanes together, repeated."""
    jobs = []
    for name, per_cu, kw in (("hhe6", 20, {"max_attempts": 400}), ("katz96", 20, {"max_attempts": 400}),
                             ("mixed5", 20, {"max_attempts": 400}), ("hhe6", 3, {"max_attempts": 400})):
        make, systems, base = NETS[name]
        n = per_cu * num_cu() + 5
        jobs.append((make(), n, *systems(n), {**base, **kw}))
    for N in (64, 100):
        n = (1 if N == 64 else 2) * num_cu() + 90
        jobs.append((api.Network.mass_action(N, *W.mass_action_network(N, 700 + N)), n,
                     *W.mass_action_systems(n, N, 7, W.MIXED_SCALE_RANGE),
                     {"tend": 1e6, "tol": 1e-10, "rel": 8e-5, "mode": api.MODE_FAST,
                      "controller": api.CTRL_ADAPTIVE, "max_attempts": 200}))
    alone = [run(net, n, y0, c, api.KERNEL_AUTO, **kw) for net, n, y0, c, kw in jobs]
    got, errors = [[] for _ in jobs], []

    def work(i):
        net, n, y0, c, kw = jobs[i]
        try:
            for _ in range(4):
                got[i].append(run(net, n, y0, c, api.KERNEL_AUTO, **kw))
        except Exception as e:  # noqa: BLE001 (reported below)
            errors.append((i, e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for i, a in enumerate(alone):
        assert len(got[i]) == 4
        for g in got[i]:
            assert same(a[0], g[0]) and np.array_equal(a[1], g[1]) and np.array_equal(a[2], g[2]), i
