"""wind_integrate's host code on a HIP runtime without a device (fake_hip.cpp)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r"""
import ctypes as C, sys
import numpy as np
fake = C.CDLL(sys.argv[1], C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
from wind_amd import api
from wind_amd import networks as W

lib = api.load()


def call(net, n, stream, kernel=api.KERNEL_AUTO, mode=api.MODE_EXACT, outputs=True):
    y, c = W.hhe6_systems(n, 1)
    before = y.copy()
    out = [np.zeros(n, np.int32) for _ in range(2)] if outputs else [None, None]
    o = api.WindOptions()
    lib.wind_options_init(C.byref(o))
    o.mode, o.kernel, o.stream = mode, kernel, stream
    if outputs:
        o.steps_out, o.status_out = (a.ctypes.data for a in out)
    rc = lib.wind_integrate(net.handle, 0.0, 1.0, 1, c.ctypes.data, y.ctypes.data, n, 6, 1e-3, 1e-3, C.byref(o))
    return rc, fake.fake_pending(), np.array_equal(y, before)


net = api.Network.builtin(api.NET_HHE6, W.hhe6_params())
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I/opt/rocm/include", "-Wno-return-type",
                    os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", so], check=True)
    return so


def child(fake, body, *args):
    r = subprocess.run([sys.executable, "-c", CHILD + body, fake, ROOT, *map(str, args)], capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("n", [300, 5000, 60000])  # one pinned copy each way; the same with a hand-over list; arrays one by one
@pytest.mark.parametrize("what", ["none", "block", "hipGetLastError", "hipMalloc", "hipMemcpyAsync"])
def test_a_call_leaves_nothing_queued(fake, n, what):
    """Also where it fails after it has queued copies: the next call may take its buffers."""
    child(fake, r"""
what, n = sys.argv[3], int(sys.argv[4])
seen = 0
for k in range(1, 12):  # (each call of the function in turn, until none is left to fail)
    kw = {"kernel": api.KERNEL_BLOCK, "mode": api.MODE_FAST} if what == "block" else {}
    if what.startswith("hip"):
        if what == "hipMalloc":  # the pools keep what they have: grow them
            n += 1000 if n > 50000 else 0
        fake.fake_fail(what.encode(), k)
    rc, pending, same = call(net, n, 0x1000 * k, **kw)
    fake.fake_fail(what.encode(), 0)
    assert pending == 0, (what, k, pending)
    assert same
    assert rc == 0 or what != "none"
    seen += rc != 0
assert (seen > 0) == (what != "none")
""", what, n)


def test_tile_kernel_matrices_leave_room_for_its_own_lds(fake):
    """The dense fallback's matrices go to LDS only where they fit beside what the kernel declares itself."""
    child(fake, r"""
import os
N, nc, own = 100, 10, 600  # katz96_t20; a kernel's declared LDS
need = 4 * (5 * N + 12 + 2 * N * N) + own
p = C.CDLL(os.path.join(api._HERE, "lib", "gen", "katz96_t20", "libwind_net.so"))


class Desc(C.Structure):
    _fields_ = [("abi", C.c_int), ("N", C.c_int), ("nconst", C.c_int), ("nreactions", C.c_int), ("name", C.c_char_p),
                ("flops_rhs", C.c_longlong), ("flops_jac", C.c_longlong), ("launch", C.c_void_p),
                ("lockstep", C.c_void_p),
                ("scratch", C.CFUNCTYPE(C.c_int, C.c_int, C.c_int, C.c_int, C.c_int, C.c_int, C.c_float, C.c_int,
                                        C.POINTER(C.c_size_t)))]


p.wind_plugin_get.restype = C.POINTER(Desc)
d = p.wind_plugin_get().contents
assert (d.N, d.nconst) == (N, nc)
for limit in (need - own + 256, need - 1, need, need + 1000):
    fake.fake_lds(limit, b"gen_tile_integrate", own)
    b = C.c_size_t()
    assert d.scratch(80, api.SIE, api.MODE_EXACT, api.KERNEL_AUTO, 256, 0.0, 0, C.byref(b)) == 0
    assert (b.value == 0) == (limit >= need), (limit, need, b.value)
""")


@pytest.mark.parametrize("N,R,form", [(32, 716, (2, 8)), (32, 2018, (2, 3)), (64, 734, (4, 6)), (64, 1586, (4, 3))])
def test_dense_forms_reach_the_networks_that_their_lds_allows(fake, N, R, form):
    """The largest networks that the register solver takes with its full number of workgroups per CU, and at all."""
    child(fake, r"""
import re
N, R, form = int(sys.argv[3]), int(sys.argv[4]), sys.argv[5]
net = api.Network.mass_action(N, *W.mass_action_network(N, 5, R=R))
y, c = W.mass_action_systems(3000, N, 1)
fake.fake_launched.restype = C.c_char_p
fake.fake_launched()
api.integrate(net, 0.0, 1.0, 1, c, y, 3000, 1e-3, 1e-3, mode=api.MODE_FAST, controller=api.CTRL_ADAPTIVE)
names = fake.fake_launched().decode()
assert "ma_dense_reg_integrateILi%sELi%sE" % tuple(form.split(",")) in names, names
""", N, R, "%d,%d" % form)


def test_network_tables_go_up_in_one_allocation(fake):
    """A mass-action network's tables: the only allocation failing is an error of the call, and a later one works."""
    child(fake, r"""
for N, R in ((1, 0), (9, 0), (3, 12), (64, 256), (170, 680)):
    rx, k = W.mass_action_network(N, 5, R=R)
    for what, fails in (("hipMalloc", 1), ("hipMalloc", 2)):
        fake.fake_fail(what.encode(), fails)
        try:
            api.Network.mass_action(N, rx, k).close()
            assert fails == 2, (N, R)
        except api.WindError:
            assert fails == 1, (N, R)
        fake.fake_fail(what.encode(), 0)
""")
