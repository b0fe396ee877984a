"""The small-batch stepper (one workgroup per parcel, csrc/sfg_fold.hip): on
the CPU through the emulation of its kernel and layout against the oracle, on
the GPU against the generated steppers and at the batch sizes where the choice
between them changes."""
import ctypes
import os
import subprocess
import tempfile

import numpy as np
import pytest

from conftest import ROOT, relerr
from test_emul_kernels import GEN, PROCS, to_nlm, to_state

CSRC = os.path.join(ROOT, "specfab_amd", "csrc")
_lib = []


def fold_lib():
    if not os.path.exists(os.path.join(GEN, "gaunt_L20.inc")):
        pytest.skip("generated tables not present (run the build)")
    if not _lib:
        out = os.path.join(tempfile.gettempdir(), "sfg_emul_fold_%d.so" % os.getpid())
        subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-DSFG_HOST_EMUL", "-pthread", "-w", "-I", CSRC,
                               "-x", "c++", os.path.join(ROOT, "tests", "emul_fold.cpp"),
                               os.path.join(CSRC, "sfg_fold_host.cpp"), os.path.join(CSRC, "sfg_basis.cpp"), "-o", out])
        _lib.append(ctypes.CDLL(out))
    return _lib[0]


def emul(L, prec, scheme, procs, steps, dt, nlm0, ug, tau, g0, lam, counts=None, dec=0, given=False, traj=False, split=0):
    P = len(nlm0)
    x, st = to_state(nlm0, L), np.zeros(P, np.int32)
    out = np.zeros((steps + 1, P, nlm0.shape[1], 2), np.float32) if traj else None
    ptr = lambda a: None if a is None else a.ctypes.data_as(ctypes.c_void_p)
    c = ctypes
    fold_lib().emul_fold(L, c.c_int64(P), 0 if prec == "fp64" else 1, sum(PROCS[p] for p in procs),
                         1 if scheme == "rk4" else 0, steps, c.c_double(dt), ptr(ug), ptr(tau), ptr(g0), ptr(lam), ptr(x),
                         ptr(counts), dec, ptr(st), int(given), ptr(out), c.c_int64(split))
    return to_nlm(x, L), st, out


def inputs(L, P, seed):
    from specfab_amd import workloads as W
    rng = np.random.default_rng(seed)
    nlm0 = W.perturbed_isotropic(rng, P, L, sigma=1e-2)
    ug = np.ascontiguousarray(W.traceless_gradients(rng, P))
    return nlm0, ug, 10.0 ** rng.uniform(-4, -2, P), 10.0 ** rng.uniform(-4, -3, P)


def forced(variant):
    """A context that steps every batch with this variant."""
    from specfab_amd import _lib as SL
    os.environ["SFG_VARIANT"] = str(variant)
    try:
        return SL.Context(0)
    finally:
        del os.environ["SFG_VARIANT"]


# every layout (threads, slots) of the truncations, both schemes and process
# sets with and without <D>; the sums differ from the oracle's by their order
@pytest.mark.parametrize("L", [4, 6, 8, 10, 12, 14, 16, 18, 20])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32c", 2e-6)])
def test_emulated_fold_vs_oracle(oracle, L, prec, tol):
    P = 3
    nlm0, ug, g0, lam = inputs(L, P, L)
    for scheme, procs, given in (("rk4", ("LROT", "REG", "DDRX", "CDRX"), L % 4 == 0), ("euler", ("LROT", "REG"), False)):
        ref = oracle.evolve(L, nlm0, ug, g0, lam, 3, 0.5, scheme, procs)
        out, st, _ = emul(L, prec, scheme, procs, 3, 0.5, nlm0, ug, None, g0, lam, given=given)
        assert relerr(out, ref) < tol, (scheme, relerr(out, ref))
        assert not st.any()


def test_emulated_fold_step_counts_and_trajectory(oracle):
    """Per-parcel and remaining step counts (0 among them) and the trajectory
    in single precision, the state rounded after every step."""
    L, P = 8, 11
    nlm0, ug, g0, lam = inputs(L, P, 5)
    procs = ("LROT", "REG", "DDRX")
    counts = np.array([0, 1, 2, 3, 4, 5, 0, 7, 1, 2, 3], np.int32)
    out, st, _ = emul(L, "fp64", "rk4", procs, 9, 0.5, nlm0, ug, None, g0, lam, counts=counts.copy())
    left = counts.copy()
    out2, _, _ = emul(L, "fp64", "rk4", procs, 3, 0.5, nlm0, ug, None, g0, lam, counts=left, dec=1, given=True)
    assert (left == np.maximum(counts - 3, 0)).all()
    for p in range(P):
        for got, k in ((out, counts[p]), (out2, min(counts[p], 3))):
            ref = oracle.evolve(L, nlm0[p:p + 1], ug[p:p + 1], g0[p:p + 1], lam[p:p + 1], int(k), 0.5, "rk4", procs)
            assert relerr(got[p:p + 1], ref) < 1e-12
    _, _, tr = emul(L, "fp64", "euler", procs, 4, 0.5, nlm0, ug, None, g0, lam, traj=True)
    y = nlm0
    for k in range(1, 5):
        y = oracle.evolve(L, y, ug, g0, lam, 1, 0.5, "euler", procs).astype(np.complex64).astype(np.complex128)
        z = tr[k, :, :, 0] + 1j * tr[k, :, :, 1]
        # one rounding to single precision may fall the other way
        assert np.abs(z - y).max() <= 2 ** -23 * np.abs(y).max()


@pytest.mark.parametrize("P,split", [(2, 1), (19, 8), (19, 18)])
def test_emulated_fold_in_two_launches(P, split):
    """A batch stepped as two spans of parcels, as beyond a launch's limit."""
    nlm0, ug, g0, lam = inputs(4, P, P)
    counts = np.arange(P, dtype=np.int32) % 4
    args = (4, "fp64", "rk4", ("LROT", "REG", "DDRX"), 3, 0.5, nlm0, ug, None, g0, lam)
    for given in (False, True):
        one, st1, tr1 = emul(*args, traj=True, given=given)
        two, st2, tr2 = emul(*args, traj=True, given=given, split=split)
        assert (one == two).all() and (st1 == st2).all() and (tr1 == tr2).all()
        one, _, _ = emul(*args, counts=counts.copy(), given=given)
        two, _, _ = emul(*args, counts=counts.copy(), given=given, split=split)
        assert (one == two).all()


@pytest.mark.parametrize("L", [4, 8, 12])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_emulated_fold_of_coefficients_that_are_not_finite(L, bad):
    """One Euler step leaves the coefficients finite that the bad one does not
    couple to (l up to 4 and m up to 4 apart; l up to 2 without DDRX, whose
    zero weights count as couplings)."""
    nlm0, ug, g0, lam = inputs(L, 1, 3)
    lm = [(l, m) for l in range(0, L + 1, 2) for m in range(l + 1)]
    pos = {(l, m): l * (l - 1) // 2 + l + m for l, m in lm}   # complex index
    for procs in (("LROT", "REG"), ("LROT", "REG", "DDRX")):
        for l, m in [(0, 0), (2, 1), (L, 0), (L, L)]:
            x = nlm0.copy()
            x[0, pos[l, m]] = bad
            out, st, _ = emul(L, "fp64", "euler", procs, 1, 0.5, x, ug, None, g0, lam)
            assert st[0] == 1
            hit = {q for q in lm if not np.isfinite(out[0, pos[q]])}
            # <D> couples everything to the coefficients with l <= 4
            near = {(k, n) for k, n in lm if abs(k - l) <= 4 and (abs(n - m) <= 4 or n + m <= 4)}
            assert (l, m) in hit and hit <= (set(lm) if "DDRX" in procs and l <= 4 else near), (procs, l, m, hit - near)


@pytest.mark.gpu
def test_small_batch_stepper_past_one_launch(gpu_ctx):
    """L = 16 past 2^32 work-items (2^23 parcels of 512 threads): every parcel
    as in a small batch, bit for bit."""
    import torch
    from specfab_amd import _lib as SL
    from specfab_amd.batch import FabricBatch
    L, P, k = 16, (1 << 23) + 64, 64
    ctx = forced(SL.lib()._ZN3sfg13fast_variantsEii(L, 0))   # the index after the generated steppers
    nlm0, ug, g0, lam = inputs(L, k, 2)
    small = FabricBatch(L, nlm=nlm0, ugrad=ug, gam0=g0, ctx=ctx)
    big = FabricBatch(L, P=P, ugrad=small.ugrad.repeat(P // k, 1, 1), gam0=small.gam0.repeat(P // k), ctx=ctx)
    big.x.view(big.n, P // k, k).copy_(small.x[:, None, :].expand(-1, P // k, -1))
    for b in (small, big):
        b.evolve(1, 0.5, scheme="euler", procs=("LROT", "REG", "DDRX"))
    assert not big.status.any()
    for r in range(big.n):
        assert (big.x[r].view(P // k, k) == small.x[r]).all(), r
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("L,P", [(4, 1), (8, 7), (8, 64), (12, 1001), (20, 65)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32c", 2e-6)])
def test_fold_against_generated_steppers(gpu_ctx, L, P, precision, tol):
    """Every entry route of a small batch (stresses, per-parcel steps, DDRX off
    and on, Euler and RK4) against the row-sharing steppers."""
    import torch
    from specfab_amd import _lib as SL
    from specfab_amd.batch import FabricBatch
    nlm0, ug, g0, lam = inputs(L, P, 10 * L + P)
    tau = np.ascontiguousarray(ug + ug.transpose(0, 2, 1))[:, ::-1, ::-1].copy() + 0.1 * np.eye(3)
    prec = SL.SFG_FP64 if precision == "fp64" else SL.SFG_FP32C
    fold, other = forced(SL.lib()._ZN3sfg13fast_variantsEii(L, prec)), forced(0)
    for scheme, procs, t, steps in (("rk4", ("LROT", "REG", "DDRX", "CDRX"), tau, None), ("euler", ("LROT", "REG"), None, None),
                                    ("rk4", ("LROT", "DDRX"), None, np.arange(P) % 5)):
        outs = []
        for ctx in (fold, other):
            b = FabricBatch(L, nlm=nlm0, ugrad=ug, tau=t, gam0=g0, lam=lam, steps=steps, ctx=ctx)
            b.evolve(4, 0.5, scheme=scheme, procs=procs, precision=precision)
            assert not b.status.any()
            outs.append(b.nlm().cpu().numpy())
        assert relerr(outs[0], outs[1]) < tol, (scheme, relerr(outs[0], outs[1]))
    fold.close()
    other.close()


@pytest.mark.gpu
@pytest.mark.parametrize("L", [8, 12])
def test_choice_of_stepper_by_batch_size(gpu_ctx, L):
    """On an untuned context the parcels of batches on both sides of each line
    of the choice (the small-batch stepper's limit, one 64-parcel group per CU)
    come out bit for bit as with the stepper that belongs there forced, and
    both steppers agree."""
    from specfab_amd import _lib as SL
    from specfab_amd.batch import FabricBatch
    lib = SL.lib()
    line = lib._ZN3sfg10fold_limitEiil(L, 0, ctypes.c_int64(8))   # two RK4 steps
    assert 1 < line < 16384
    nlm0, ug, g0, lam = inputs(L, 16385, L)
    fold = lib._ZN3sfg13fast_variantsEii(L, 0)   # the index after the generated steppers

    def step(P, ctx):
        b = FabricBatch(L, nlm=nlm0[:P], ugrad=ug[:P], gam0=g0[:P], ctx=ctx)
        b.evolve(2, 0.5, procs=("LROT", "REG", "DDRX"))
        assert not b.status.any()
        return b.nlm().cpu().numpy()
    untuned = SL.Context(0)
    for P in (1, line, line + 1, 16384, 16385):
        gen = step(P, forced(lib._ZN3sfg12fast_defaultEiil(L, 0, ctypes.c_int64(P))))
        small = step(P, forced(fold))
        out = step(P, untuned)
        assert (out == (small if P <= line else gen)).all(), P
        assert relerr(small, gen) < 1e-13, P
        assert P == 1 or not (small == gen).all(), P   # else the line above says nothing


@pytest.mark.gpu
@pytest.mark.parametrize("L,P,scheme", [(4, 1, "euler"), (8, 5, "euler"), (12, 1, "rk4"), (20, 2, "euler")])
def test_trajectory_against_single_steps(gpu_ctx, L, P, scheme):
    """One launch with the state rounded after every step gives the states of
    single-step calls with the rounding between them, bit for bit."""
    import torch
    from specfab_amd.batch import FabricBatch
    nlm0, ug, g0, lam = inputs(L, P, 3 * L)
    kw = dict(scheme=scheme, procs=("LROT", "REG", "DDRX", "CDRX"))
    a = FabricBatch(L, nlm=nlm0, ugrad=ug, gam0=g0, lam=lam)
    b = FabricBatch(L, nlm=nlm0, ugrad=ug, gam0=g0, lam=lam)
    tr = a.trajectory(6, 0.5, **kw)
    for k in range(6):
        b.evolve(1, 0.5, **kw)
        z = b.nlm().to(torch.complex64)
        assert torch.equal(tr[k], z), k
        b.set_nlm(z)
    assert torch.equal(a.x, b.x) and not a.status.any()
