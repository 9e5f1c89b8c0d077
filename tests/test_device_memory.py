"""The solver's optional device memory (the ring of preconditioned residuals),
on a HIP runtime without a device that counts allocations (fake_hip.c): it is
bounded, and no call of any context fails because a ring holds the memory that
the call needs."""

import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys, threading, time
F = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
F.fake_used.restype = ctypes.c_size_t
F.fake_capacity.argtypes = [ctypes.c_size_t]
import numpy as np
from simcoflow3d_amd import configs
from tests import helpers as H
BIG = 1 << 40
SIZE = (40, 32, 24)
N = SIZE[0] * SIZE[1] * SIZE[2]
c = H.case(0, size=SIZE)
out = {n: np.zeros(c.halo_shape, order="F") for n in ("p", "u", "v", "w")}

def projector(memory=None, **kw):
    P = H.projector(c, max_iter=4, **kw)
    if memory is not None:
        P.set_solver_memory(memory)
    return P

def solve(P):  # "device" arrays: no kernel runs
    P.project_dev(H.fields(c), c.bc_flag, c.dt, out)

def geometry(P):
    P.grid_preprocess(configs.geometry_case(SIZE, "bodies", seed=1, stretch=True))

def host(P):
    P.project(H.fields(c), c.bc_flag, c.dt)

def use(*calls, **kw):
    before = F.fake_used()
    P = projector(**kw)
    for f in calls:
        f(P)
    n = F.fake_used() - before
    P.close()
    assert F.fake_used() == before and F.fake_bad_frees() == 0
    return n
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-w", "-o", so,
                    os.path.join(HERE, "fake_hip.c"), "-lpthread"], check=True)

    def run(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE + body, so], cwd=os.path.dirname(HERE),
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


@pytest.mark.parametrize("prec", (0, 1))
def test_ring_is_bounded(fake, prec):
    """15 buffers of 4 or 8 bytes a cell at most, what sp_set_solver_memory
    allows, and a sixteenth of the free memory."""
    fake(f"""
prec = {prec}
F.fake_capacity(BIG)
z = N * (4 if prec else 8) + 512
base = use(solve, precision=prec, memory=0)
assert 14 * (z - 512) < use(solve, precision=prec) - base <= 15 * z + 512
assert 2 * (z - 512) < use(solve, precision=prec, memory=4 * z) - base <= 4 * z
assert use(solve, precision=prec, memory=1) == base
for room in (16 * 40 * z, 16 * 4 * z, 8 * z):
    F.fake_capacity(base + room)
    assert 0 <= use(solve, precision=prec) - base <= room // 16
""")


@pytest.mark.parametrize("prec", (0, 1))
@pytest.mark.parametrize("call", ("geometry", "host"))
def test_a_later_call_finds_its_memory(fake, prec, call):
    """On a device that holds a projection and then the call, and no more."""
    fake(f"""
F.fake_capacity(BIG)
F.fake_capacity(use(solve, {call}, precision={prec}, memory=0))
use(solve, {call}, precision={prec})
F.fake_capacity(BIG)
need = use(solve, {call}, precision={prec}, memory=0)
P = projector(precision={prec})
solve(P)
F.fake_capacity(need)  # the ring is held, and the rest of the device is in use
{call}(P)
solve(P)
P.close()
assert F.fake_used() == 0 and F.fake_bad_frees() == 0
""")


@pytest.mark.parametrize("prec", (0, 1))
def test_another_context_finds_its_memory(fake, prec):
    """Two contexts where two fit without rings; one that is refused for good
    leaves the first as it was, and able to solve."""
    fake(f"""
F.fake_capacity(BIG)
base = use(solve, precision={prec}, memory=0)
P = projector(precision={prec})
solve(P)
assert F.fake_used() > base
F.fake_capacity(2 * base)
Q = projector(precision={prec})
solve(Q)
assert F.fake_used() <= 2 * base
solve(P)
P.set_params(div_tol=1e-9)
solve(P)
R = None
try:
    R = projector(precision={prec})
    solve(R)
except Exception as e:
    assert "memory" in str(e), e
else:
    raise AssertionError("a third context fitted")
if R is not None:
    R.close()
solve(P)
P.close()
Q.close()
assert F.fake_used() == 0 and F.fake_bad_frees() == 0
""")


def test_a_ring_in_use_is_waited_for(fake):
    """A solve under way keeps its ring; the context that needs the memory gets
    it when the solve is over."""
    fake("""
F.fake_capacity(BIG)
base = use(solve, memory=0)
P = projector()
solve(P)
F.fake_hold(1)
a = threading.Thread(target=solve, args=(P,))
a.start()
while not F.fake_held():
    time.sleep(0.001)
F.fake_capacity(2 * base)
Q = projector()
got = []
b = threading.Thread(target=lambda: (solve(Q), got.append(1)))
b.start()
time.sleep(0.3)
held = F.fake_used()
assert not got and F.fake_held()
F.fake_hold(0)
a.join()
b.join()
assert got and held > F.fake_used() - base and F.fake_used() <= 2 * base
P.close()
Q.close()
assert F.fake_used() == 0 and F.fake_bad_frees() == 0
""")
