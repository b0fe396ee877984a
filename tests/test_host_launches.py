"""The library's host side against a recording HIP runtime (mock_hip.cpp), in
a process of its own per test: which kernels a call launches, how many threads
and in which memory.  Nothing runs on a GPU."""
import json
import os
import subprocess
import sys
import tempfile

import pytest

from conftest import ROOT

_mock = []

PRELUDE = """
import ctypes, json, os, sys
c = ctypes
mock = c.CDLL(sys.argv[1], mode=c.RTLD_GLOBAL)   # before the library: its runtime calls come here
from specfab_amd import _lib
lib = _lib.lib()
mock.mock_name.restype, mock.mock_threads.restype = c.c_char_p, c.c_longlong
mock.mock_cost.argtypes = [c.c_char_p, c.c_double, c.c_double]
nvar = lambda L, prec=0: lib._ZN3sfg13fast_variantsEii(L, prec)   # generated variants; then the small-batch stepper

def ctx(variant=None):
    os.environ.pop("SFG_VARIANT", None)
    if variant is not None:
        os.environ["SFG_VARIANT"] = str(variant)
    return _lib.Context(0)

def desc(L, P, nsteps=1, scheme=_lib.SFG_RK4, prec=_lib.SFG_FP64):
    d = _lib.EvolveDesc()
    d.L, d.P, d.procs, d.scheme, d.precision, d.nsteps, d.dt = L, P, 11, scheme, prec, nsteps, 0.5
    d.iota = 1.0
    d.ugrad_dev = d.x_dev = 1 << 20   # not read
    d.gam0_dev = 1 << 20
    return d

def run(fn, cx, *a, **kw):
    mock.mock_reset()
    rc = fn(cx.handle, c.byref(desc(*a, **kw)), None)
    return rc, [mock.mock_name(i).decode() for i in range(mock.mock_count())]
"""


def host(code):
    """Run code after PRELUDE in a process with the recording runtime; its last
    line prints what it found as JSON."""
    from specfab_amd import _lib
    if not os.path.exists(_lib.LIBPATH):
        pytest.skip("library not built")
    if not _mock:
        out = os.path.join(tempfile.gettempdir(), "sfg_mock_hip_%d.so" % os.getpid())
        subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-w", "-I",
                               os.path.join(ROOT, "specfab_amd", "csrc"), os.path.join(ROOT, "tests", "mock_hip.cpp"),
                               "-o", out])
        _mock.append(out)
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, _mock[0]], cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.strip().split("\n")[-1])


def test_no_allocation_calls_of_the_small_batch_stepper():
    """sfg_evolve_noalloc with the small-batch stepper forced launches what
    sfg_evolve does and writes no parameters into the static workspace, whose
    size the batch no longer has to fit; a stepper that keeps its parameters
    there gets only batches that fit."""
    out = host("""
fold, gen = ctx(nvar(12)), ctx(2)
res = {}
for cx, tag in ((fold, "fold"), (gen, "gen")):
    _lib.check(lib.sfg_evolve(cx.handle, c.byref(desc(12, 0)), None))   # the tables of L = 12
    for P in (1, 4099, 300000, 400000, 1 << 20):
        rc, names = run(lib.sfg_evolve_noalloc, cx, 12, P)
        ok = all(mock.mock_params_in_bounds(i) for i, n in enumerate(names) if "params_kernel" in n)
        res["%s %d" % (tag, P)] = [rc, ok, names, run(lib.sfg_evolve, cx, 12, P)[1]]
print(json.dumps(res))
""")
    for key, (rc, in_bounds, names, plain) in out.items():
        assert in_bounds, key
        if key.startswith("fold"):
            assert rc == 0 and names == plain and len(names) == 1 and "fold_kernel" in names[0], (key, names)
        elif int(key.split()[1]) <= 300000:
            assert rc == 0 and names == plain and "params_kernel" in names[0], (key, names)
        else:
            assert rc != 0 and not names, key


# (L, 2^32 / threads per workgroup): one parcel per workgroup of the small-batch
# stepper, and HIP refuses 2^32 work-items or more in a launch
@pytest.mark.parametrize("L,line", [(4, 1 << 26), (12, 1 << 24), (16, 1 << 23)])
def test_small_batch_stepper_past_one_launch(L, line):
    """Batches at and past the launch limit step in several launches that
    cover every parcel once."""
    out = host("""
L, line = %d, %d
cx = ctx(nvar(L))
res = []
for P in (1, line - 8, line - 1, line, line + 1, 2 * line + 5):
    rc, names = run(lib.sfg_evolve, cx, L, P)
    spans = []
    for i in range(len(names)):
        p0, n = c.c_longlong(), c.c_longlong()
        mock.mock_fold_span(i, c.byref(p0), c.byref(n))
        spans.append([p0.value, n.value, mock.mock_threads(i)])
    res.append([P, rc, mock.mock_failed(), spans])
print(json.dumps(res))
""" % (L, line))
    for P, rc, failed, spans in out:
        assert rc == 0 and failed == 0, (P, rc, failed)
        at = 0
        for p0, n, threads in spans:
            assert p0 == at and n > 0 and threads < 1 << 32
            at += n
        assert at == P and len(spans) == (P + line - 9) // (line - 8), (P, spans)


def test_tuned_choice_holds_for_its_batch_sizes():
    """What sfg_autotune keeps: tuned on few parcels, nothing for batches beyond
    FAST_SMALL, and the small-batch stepper where its win (or loss) at the tuned
    size and steps carries over to; tuned on a field, its stepper for all."""
    out = host("""
SMALL, L = 64 * 256, 12
names = {}
for v in range(nvar(L) + 1):
    names[run(lib.sfg_evolve, ctx(v), L, 100)[1][-1]] = v
F = nvar(L)
def kind(cx, P, nsteps=2):
    return names[run(lib.sfg_evolve, cx, L, P, nsteps)[1][-1]]
best = c.c_int()
def tune(cx, P, steps=2):
    _lib.check(lib.sfg_autotune(cx.handle, L, 0, P, steps, None, c.byref(best), None, 0))
    return best.value
plain = ctx()
line = lib._ZN3sfg10fold_limitEiil(L, 0, 8)   # two RK4 steps
P = [1, 200, 1000, 3000, line, line + 1, 9000, SMALL, SMALL + 1, 200000, 1 << 20]
res = {"F": F, "untuned": [kind(plain, p) for p in P]}
# the small-batch stepper 1 us per parcel, the others 3 ms and 0.8 us per parcel;
# variant 1 the fastest of them
mock.mock_cost(b"fold_kernel", 0.0, 1e-3)
mock.mock_cost(b"evolve_fast", 3.0, 0.05)
mock.mock_cost(b"f64_v1E", 2.9, 0.05)
cx = ctx(); res["small"] = [tune(cx, 1000), [kind(cx, p) for p in P]]
cx = ctx(); res["wins"] = [tune(cx, 9000), [kind(cx, p) for p in P], kind(cx, 9000, 1)]
cx = ctx(); res["large"] = [tune(cx, 200000), [kind(cx, p) for p in P]]
res["both"] = [tune(cx, 1000), [kind(cx, p) for p in P]]
mock.mock_cost(b"fold_kernel", 0.0, 5.0)   # and where it loses
cx = ctx(); res["loses"] = [tune(cx, 1000), [kind(cx, p) for p in P], kind(cx, 1000, 3)]
print(json.dumps(res))
""")
    F, u = out["F"], out["untuned"]
    assert u[:5] == [F] * 5 and F not in u[5:] and u[7] != u[8]
    # tuned on few parcels: a large field keeps its own choice, and the line stays
    assert out["small"][0] == F and out["small"][1] == u[:5] + [1, 1, 1] + u[8:]
    # a win at 9,000 parcels moves the line there, for as many steps or more
    assert out["wins"][0] == F and out["wins"][1] == [F] * 7 + [1] + u[8:] and out["wins"][2] != F
    # tuned on a field: its stepper for every batch, until tuned on few parcels too
    assert out["large"][0] == 1 and out["large"][1] == [1] * len(u)
    assert out["both"][0] == F and out["both"][1] == u[:5] + [1] * 6
    # a loss at 1,000 parcels and two steps says nothing of fewer parcels or more steps
    assert out["loses"][0] == 1 and out["loses"][1] == [F, F] + [1] * 6 + u[8:] and out["loses"][2] == F


def test_velocity_launches_fill_their_lanes():
    """Elastic velocities of few parcels in many directions: the launch has
    about as many threads as (parcel, direction) pairs, whatever the number of
    parcels."""
    out = host("""
import math
cx = ctx()
lame = (c.c_double * 5)(7.15e9, 3.455e9, 0.8, 0.9, 1.1)
res = []
for P, nd in ((1, 1), (1, 20000), (16, 2000), (64, 2000), (96, 500), (127, 50), (128, 50), (129, 50), (20011, 36)):
    th = (c.c_double * nd)(*[0.1 + 1e-4 * i for i in range(nd)])
    mock.mock_reset()
    rc = lib.sfg_Vi_elastic_tranisotropic_batch(cx.handle, 4, P, 1 << 20, 0.5, lame, 917.0, nd, th, th, 1 << 20, 1 << 20, None)
    res.append([P, nd, rc, [mock.mock_threads(i) for i in range(mock.mock_count())]])
print(json.dumps(res))
""")
    for P, nd, rc, threads in out:
        assert rc == 0 and len(threads) == 1
        assert P * nd <= threads[0] <= 4 * P * nd / 3 + 128, (P, nd, threads)


@pytest.mark.parametrize("P,nd", [(1 << 20, 4095), (1 << 20, 4096), (1 << 20, 8192), ((1 << 20) + 1, 8192), (4 * 129 * 16384, 1000)])
def test_velocities_past_one_launch(P, nd):
    """2^25 workgroups and more (2^32 work-items): the launch stays below the
    runtime's limit and its kernel loops."""
    rc, n, threads = host("""
P, nd = %d, %d
cx = ctx()
lame = (c.c_double * 5)(7.15e9, 3.455e9, 0.8, 0.9, 1.1)
th = (c.c_double * nd)(*[0.1 + 1e-4 * i for i in range(nd)])
rc = lib.sfg_Vi_elastic_tranisotropic_batch(cx.handle, 4, P, 1 << 20, 0.5, lame, 917.0, nd, th, th, 1 << 20, 1 << 20, None)
print(json.dumps([rc, mock.mock_count(), mock.mock_threads(0) if mock.mock_count() else 0]))
""" % (P, nd))
    assert rc == 0 and n == 1 and threads == min(-(-P // 128) * nd * 128, 1 << 31)


# (L, precision, scheme, steps, parcels, us with the small-batch stepper, us with
# the generated one): measured on both sides of the line
MEASURED = [(4, 0, 0, 1, 2000, 12.4, 13.2), (4, 0, 0, 1, 5000, 21.5, 13.3), (4, 0, 1, 1, 6000, 26.8, 16.6),
            (4, 1, 0, 1, 2000, 17.5, 12.3), (4, 1, 1, 30, 4000, 85.4, 98.6), (6, 1, 1, 3, 6000, 51.4, 27.9),
            (8, 0, 1, 1, 7000, 43.0, 25.5), (8, 0, 1, 10, 9500, 148.0, 132.5), (12, 0, 1, 1, 5000, 56.4, 38.9),
            (12, 0, 1, 30, 8000, 737.6, 768.3), (12, 1, 1, 1, 4000, 49.2, 30.4), (20, 0, 0, 1, 1000, 27.7, 32.1),
            (20, 0, 1, 30, 7000, 1806.6, 1949.0), (20, 1, 1, 3, 4000, 152.1, 117.6)]


def test_choice_of_stepper_follows_the_times():
    out = host("""
cx = ctx()
print(json.dumps(["fold" in run(lib.sfg_evolve, cx, L, P, n, scheme, prec)[1][-1]
                  for L, prec, scheme, n, P, f, g in %r]))
""" % (MEASURED,))
    for (L, prec, scheme, n, P, f, g), fold in zip(MEASURED, out):
        assert fold == (f < g), (L, prec, scheme, n, P)


def test_tables_of_a_second_context():
    """A context's first step at L = 20 uploads tables; they are laid out once
    per process, so that a second context is ready in a fraction of the time."""
    t = host("""
import time
t = []
for k in range(4):
    cx = ctx()
    t0 = time.perf_counter()
    _lib.check(lib.sfg_evolve(cx.handle, c.byref(desc(20, 1)), None))
    t.append(time.perf_counter() - t0)
print(json.dumps(t))
""")
    assert min(t[1:]) < 0.2 * t[0], t


def test_trajectory_of_no_parcels():
    """No parcels need no buffers, as for sfg_evolve; parcels need theirs."""
    out = host("""
cx = ctx()
rc = lambda P, traj: lib.sfg_evolve_trajectory(cx.handle, c.byref(desc(8, P, 3, 0)), traj, None)
print(json.dumps([rc(0, None), rc(1, None), rc(1, 1 << 20), mock.mock_count()]))
""")
    assert out[0] == 0 and out[1] != 0 and out[2] == 0 and out[3] == 1
