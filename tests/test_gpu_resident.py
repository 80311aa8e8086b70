"""Resident conjugate gradients (many iterations in one launch, the blocks
meeting through device-wide sums) against the segment kernels (three launches
per iteration on the same segments): the same bits, iteration counts and
residuals.  A profiled solve takes the segment kernels."""
import ctypes as C
import json
import os
import subprocess
import sys
import threading

import numpy as np
import pytest
import scipy.sparse

from insilico_amd import abi, problems as P
import test_zz_no_alloc as noalloc

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _banded(n, half, seed):
    """symmetric, diagonally dominant CSR with up to 2 * half + 1 entries a
    row at scattered offsets"""
    r = np.random.RandomState(seed)
    off = np.unique(np.concatenate([[1], r.randint(1, max(2, n // 2), half)]))[:half]
    off = off[off < n]
    row, col, val = [np.arange(n)], [np.arange(n)], [np.full(n, 2.0 * half + 2.0)]
    for d in off:
        v = -r.uniform(0.2, 1.0, n - d)
        i = np.arange(n - d)
        row += [i, i + d]
        col += [i + d, i]
        val += [v, v]
    row, col, val = np.concatenate(row), np.concatenate(col), np.concatenate(val)
    o = np.lexsort((col, row))
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(row, minlength=n), out=rp[1:])
    return rp, col[o].astype(np.int32), val[o], r.standard_normal(n)


# rows about the edges of slices, of segments (1024 rows for short rows, 512,
# 256) and of what all segments hold (256 of 1024 rows); row lengths for 4, 8 and 16 lanes,
# register passes and streamed rows
CSR = [(1, 1), (2, 1), (63, 2), (64, 2), (65, 2), (1023, 3), (1024, 3), (1025, 3), (4097, 4),
       (511, 9), (513, 9), (5000, 13), (70001, 13), (140000, 10), (700, 30), (4096, 40),
       (262144, 2), (262145, 2)]


@pytest.mark.parametrize("n,half", CSR)
def test_csr_resident_equals_segment_kernels(oracle, n, half):
    print("case", n, half, flush=True)
    rp, ci, val, b = _banded(n, half, n + half)
    with abi.Context(0) as c:
        c.set_csr(rp, ci, val)
        c.set_rhs(b)
        for mode in (abi.SOLVE_FP64, abi.SOLVE_MIXED):
            got = []
            for prof in (0, 1, 0):
                c.set_profiling(prof)
                it, rel, _ = c.solve(mode, abi.FMT_CSR, 1e-9)
                got.append((it, rel, c.get_solution()))
            for g in got[1:]:
                assert g[:2] == got[0][:2]
                assert np.array_equal(g[2], got[0][2])
            # the residual is FP64 and of this matrix: what rounding allows
            r = b - oracle.spmv(rp, ci, val, got[0][2])
            assert np.linalg.norm(r) <= 1.001e-9 * np.linalg.norm(b) + 1e-13


def _sheet_2d(n):
    """2-D elasticity: node blocks of 2 components"""
    xyz, conn = P.unit_cube(2, n)
    return P.linear_elastic_fundsol(xyz, conn, 2)


def _half_clamped(n):
    """neo-Hooke at u = 0 with partly prescribed nodes: full slices"""
    p = P.neohooke3d(n)
    p.g[p.meta["right_x"] * 3] = 0.01
    return p


def _poisson_2d(n):
    p = P.poisson2d(n)
    p.coef = np.exp(0.5 * P.normal(n, p.conn.shape[0]))[:, None]
    return p


def _q2_2d(n):
    """2-D degree-2 field with a coefficient per element"""
    p = P.poisson2d_q2(n)
    p.coef = np.exp(0.5 * P.normal(n, p.conn.shape[0]))[:, None]
    return p


# storage forms of SELL solves at the edges of their segments: scalar
# symmetric slices (3-D, 2-D) of one wave's and more slices per wave, node
# blocks shared out over 8, 4, 3, 2 and 1 waves per slice and several slices
# per wave, full slices in registers and streamed
SELL = [(P.diffusion3d, n) for n in (2, 3, 8, 15, 24, 41, 66, 80, 85)]
SELL += [(_poisson_2d, n) for n in (3, 10, 40, 130, 270, 700)]
SELL += [(P.elasticity3d, n) for n in (2, 3, 5, 13, 20, 25, 30, 41, 44, 56, 66)]
SELL += [(_sheet_2d, n) for n in (3, 17, 60, 200, 300, 600)]
SELL += [(_half_clamped, n) for n in (2, 7, 16, 40, 46)]
SELL += [(P.diffusion3d_q2, n) for n in (2, 7, 20, 33)] + [(_q2_2d, n) for n in (4, 50)]


@pytest.mark.parametrize("make,n", SELL, ids=lambda v: str(getattr(v, "__name__", v)))
def test_sell_resident_equals_segment_kernels(make, n):
    prob = make(n)
    print("case", make.__name__, n, prob.n_active, flush=True)
    with abi.Context(0) as c:
        c.load_problem(prob)
        c.prepare(abi.SOLVE_MIXED, abi.FMT_SELL)
        c.assemble(abi.FP64)
        for mode in (abi.SOLVE_MIXED, abi.SOLVE_FP64):
            got = []
            for prof in (0, 1, 0):
                c.set_profiling(prof)
                # (large systems: enough iterations for a few replacements)
                it, rel, st = c.solve(mode, abi.FMT_SELL, 1e-8, max_it=400, check=False)
                assert st in (abi.INS_OK, abi.ERRORS_INV["NOCONV"])
                got.append((it, rel, st, c.get_solution()))
            assert got[0][2] == abi.INS_OK or got[0][0] == 400
            for g in got[1:]:
                assert g[:3] == got[0][:3]
                assert np.array_equal(g[3], got[0][3])


def test_csr_iteration_limit_and_breakdown():
    rp, ci, val, b = _banded(3000, 4, 5)
    with abi.Context(0) as c:
        c.set_csr(rp, ci, val)
        c.set_rhs(b)
        for mode in (abi.SOLVE_FP64, abi.SOLVE_MIXED):
            x = []
            for prof in (0, 1):
                c.set_profiling(prof)
                it, rel, st = c.solve(mode, abi.FMT_CSR, 1e-14, max_it=3, check=False)
                assert it == 3 and st == abi.ERRORS_INV["NOCONV"]
                x.append(c.get_solution())
            assert np.array_equal(x[0], x[1])
        c.set_profiling(0)
        c.set_rhs(np.zeros(3000))
        it, rel, st = c.solve(abi.SOLVE_FP64, abi.FMT_CSR, 1e-9)
        assert it == 0 and rel == 0.0 and not c.get_solution().any()
        c.set_csr(rp, ci, -val)
        c.set_rhs(b)
        it, rel, st = c.solve(abi.SOLVE_FP64, abi.FMT_CSR, 1e-9, check=False)
        assert st == abi.ERRORS_INV["BREAKDOWN"]


RUN = r"""
import hashlib, json
from insilico_amd import abi, problems as P
out = {}
with abi.Context(0) as c:
    c.load_problem(P.diffusion3d(20, seed=3))
    c.assemble(abi.FP64)
    for name, mode, fmt in (("fp64 csr", 0, 0), ("mixed csr", 1, 0), ("fp64 sell", 0, 1),
                            ("mixed sell", 1, 1)):
        it, rr, _ = c.solve(mode, fmt, 1e-9)
        out[name] = [it, rr, hashlib.sha256(c.get_solution().tobytes()).hexdigest()]
print(json.dumps(out), flush=True)
"""


def test_a_wait_that_is_given_up_falls_back():
    """with a bound of no polls a block gives up at once; the solve is then
    repeated by the segment kernels, with the same result"""
    got = []
    for polls in ("500000", "0"):
        env = dict(os.environ, INS_RESIDENT_POLLS=polls)
        r = subprocess.run([sys.executable, "-c", RUN], cwd=ROOT, env=env, capture_output=True,
                           text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        got.append(json.loads(r.stdout.strip().splitlines()[-1]))
    assert got[0] == got[1]


SCALAR = r"""
import hashlib, json
from insilico_amd import abi, problems as P
out = {}
cases = [("3d %d %d" % (n, s), P.diffusion3d(n, seed=s))
         for n, seeds in ((5, 2), (16, 12), (31, 3), (41, 1), (66, 1)) for s in range(seeds)]
cases += [("2d %d" % n, P.poisson2d(n)) for n in (7, 40, 130)]
for name, prob in cases:
    with abi.Context(0) as c:
        c.load_problem(prob)
        c.prepare(abi.SOLVE_MIXED, abi.FMT_SELL)
        c.assemble(abi.FP64)
        it, rr, _ = c.solve(abi.SOLVE_MIXED, abi.FMT_SELL, 1e-8)
        out[name] = [it, hashlib.sha256(c.get_solution().tobytes()).hexdigest()]
print(json.dumps(out), flush=True)
"""


def test_mixed_scalar_solves_take_the_steps_of_the_plain_kernels():
    """A mixed solve of scalar symmetric slices rounds every FP32 step as the
    three kernels on whole vectors do (INS_RESIDENT=0), so it has their
    iterates: where it stops, and how far from the solution, hangs on rounding.
    (The FP64 sums are added in another order; no step of these systems feels
    their last bits.)"""
    got = []
    for on in ("1", "0"):
        env = dict(os.environ, INS_RESIDENT=on)
        r = subprocess.run([sys.executable, "-c", SCALAR], cwd=ROOT, env=env, capture_output=True,
                           text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        got.append(json.loads(r.stdout.strip().splitlines()[-1]))
    assert got[0] == got[1]


def _fresh(prob, mode):
    with abi.Context(0) as c:
        c.load_problem(prob)
        c.assemble(abi.FP64)
        it, rel, _ = c.solve(mode, abi.FMT_SELL, 1e-9)
        return it, rel, c.get_solution()


@pytest.mark.parametrize("make", [P.diffusion3d, P.elasticity3d], ids=["scalar", "blocks"])
def test_a_cancelled_launch_that_gave_up_leaves_nothing_behind(make, monkeypatch):
    """A request whose launch gave up leaves before anyone looks at it; the
    next solves of its context, other systems, must not meet its words"""
    n = 14
    first, second, third = (make(n, seed=s) for s in (3, 4, 5))
    with abi.Context(0) as c, abi.Server(0, 2) as srv:
        for prob in (second, third):
            c.load_problem(first)
            c.assemble(abi.FP64)
            monkeypatch.setenv("INS_RESIDENT_POLLS", "0")
            slot = srv.attach(c, 1e-9)
            srv.step(4)
            assert srv.poll(slot)[0] == abi.SLOT_RUNNING
            srv.detach(slot)
            monkeypatch.delenv("INS_RESIDENT_POLLS")
            c.load_problem(prob)
            c.assemble(abi.FP64)
            for mode in (abi.SOLVE_FP64, abi.SOLVE_MIXED):
                it, rel, _ = c.solve(mode, abi.FMT_SELL, 1e-9)
                want = _fresh(prob, mode)
                assert (it, rel) == want[:2]
                assert np.array_equal(c.get_solution(), want[2])


def test_solves_after_a_give_up_keep_their_bits(monkeypatch):
    """the pause after a launch that gave up, and the return to resident ones"""
    prob = P.diffusion3d(14, seed=6)
    with abi.Context(0) as c:
        c.load_problem(prob)
        c.assemble(abi.FP64)
        want = None
        for polls in ["0"] + [None] * 18 + ["0"] + [None] * 2:
            if polls:
                monkeypatch.setenv("INS_RESIDENT_POLLS", polls)
            else:
                monkeypatch.delenv("INS_RESIDENT_POLLS", raising=False)
            for mode in (abi.SOLVE_FP64, abi.SOLVE_MIXED):
                c.solve(mode, abi.FMT_SELL, 1e-9)
            got = c.get_solution()
            want = got if want is None else want
            assert np.array_equal(got, want)


# one request of every storage form: scalar slices, node blocks in 3-D and 2-D,
# full slices (partly prescribed nodes, degree 2), and one too large for segments
BATCH = [(P.diffusion3d, 17), (P.elasticity3d, 9), (_sheet_2d, 30), (_half_clamped, 8),
         (P.diffusion3d_q2, 7), (_poisson_2d, 50), (P.diffusion3d, 75), (P.elasticity3d, 50)]


@pytest.mark.parametrize("batch", [BATCH[:-1], BATCH], ids=["segments", "whole"])
@pytest.mark.parametrize("polls", [None, "0"], ids=["resident", "given up"])
def test_batch_of_all_forms_has_the_bits_of_its_solves(polls, batch, monkeypatch):
    """resident launches, or, beside the last request, which is too large for
    segments, the batched segment kernels on the second stream; with a bound of
    no polls resident requests start again on those"""
    cs, alone = [], []
    for make, n in batch:
        c = abi.Context(0)
        c.load_problem(make(n))
        c.prepare(abi.SOLVE_MIXED, abi.FMT_SELL)
        c.assemble(abi.FP64)
        it, rel, _ = c.solve(abi.SOLVE_MIXED, abi.FMT_SELL, 1e-8)
        alone.append((it, rel, c.get_solution()))
        cs.append(c)
    if polls:
        monkeypatch.setenv("INS_RESIDENT_POLLS", polls)
    with abi.Server(0, len(cs)) as srv:
        for _ in range(2):
            slots = [srv.attach(c, 1e-8) for c in cs]
            srv.run_until_done()
            for (make, n), c, slot, want in zip(batch, cs, slots, alone):
                state, status, it, rel = srv.poll(slot)
                assert (state, status) == (abi.SLOT_FINISHED, abi.INS_OK)
                srv.detach(slot)
                assert it == want[0], (make.__name__, n)
                assert np.array_equal(c.get_solution(), want[2]), (make.__name__, n)
    for c in cs:
        c.close()


@pytest.mark.parametrize("make,n,polls", [(P.elasticity3d, 28, None), (P.diffusion3d, 44, None),
                                          (P.elasticity3d, 28, "0")],
                         ids=["blocks", "scalar", "given up"])
def test_running_requests_move_to_the_segment_kernels(make, n, polls, monkeypatch):
    """two requests run resident for some steps; four more arrive, and the
    launches of six would take longer than the batched segment kernels: all
    move there and end with the bits of their solves, also where a launch gave
    up just before"""
    cs, alone = [], []
    for k in range(6):
        c = abi.Context(0)
        c.load_problem(make(n, seed=k))
        c.prepare(abi.SOLVE_MIXED, abi.FMT_SELL)
        c.assemble(abi.FP64)
        it, rel, _ = c.solve(abi.SOLVE_MIXED, abi.FMT_SELL, 1e-8)
        alone.append((it, c.get_solution()))
        cs.append(c)
    with abi.Server(0, 6) as srv:
        slots = [srv.attach(c, 1e-8) for c in cs[:2]]
        for _ in range(4):
            srv.step(7)
        if polls:
            monkeypatch.setenv("INS_RESIDENT_POLLS", polls)
            slots += [srv.attach(cs[2], 1e-8)]   # (a new table: the bound goes with it)
            srv.step(7)
        slots += [srv.attach(c, 1e-8) for c in cs[len(slots):]]
        srv.run_until_done()
        for c, slot, want in zip(cs, slots, alone):
            state, status, it, _ = srv.poll(slot)
            assert (state, status) == (abi.SLOT_FINISHED, abi.INS_OK)
            srv.detach(slot)
            assert it == want[0]
            assert np.array_equal(c.get_solution(), want[1])
    for c in cs:
        c.close()


def test_two_threads_solve_at_once():
    """launches that wait for one another take turns on the device"""
    probs = [P.diffusion3d(24, seed=1), P.elasticity3d(12, seed=2), P.diffusion3d(13, seed=3)]
    want = [_fresh(p, m) for p in probs for m in (abi.SOLVE_FP64, abi.SOLVE_MIXED)]
    got = [[] for _ in probs]

    def work(k):
        try:
            for _ in range(3):
                got[k].append([_fresh(probs[k], m) for m in (abi.SOLVE_FP64, abi.SOLVE_MIXED)])
        except Exception as e:   # (the main thread reports it)
            got[k].append(e)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(probs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    for k in range(len(probs)):
        assert len(got[k]) == 3
        for round_ in got[k]:
            for g, w in zip(round_, want[2 * k:2 * k + 2]):
                assert g[:2] == w[:2] and np.array_equal(g[2], w[2])


# (problem, storage form): the residual that the oracle's own FP64 assembly and
# product give for the solutions of both kinds of kernels
ORACLE = [(P.diffusion3d, 15), (_poisson_2d, 40), (P.elasticity3d, 9), (_sheet_2d, 17),
          (_half_clamped, 7), (P.diffusion3d_q2, 6)]


@pytest.mark.parametrize("make,n", ORACLE, ids=lambda v: str(getattr(v, "__name__", v)))
def test_solutions_against_the_oracle(oracle, make, n):
    prob = make(n)
    orp, oci, oval, ob, _ = oracle.assemble(prob)
    with abi.Context(0) as c:
        c.load_problem(prob)
        c.prepare(abi.SOLVE_MIXED, abi.FMT_SELL)
        c.assemble(abi.FP64)
        for fmt in (abi.FMT_SELL, abi.FMT_CSR):
            for mode in (abi.SOLVE_MIXED, abi.SOLVE_FP64):
                for prof in (0, 1):
                    c.set_profiling(prof)
                    c.solve(mode, fmt, 1e-8)
                    r = ob - oracle.spmv(orp, oci, oval, c.get_solution())
                    # the device's matrix is the oracle's to 1e-12 of its largest entry
                    assert np.linalg.norm(r) <= 1.001e-8 * np.linalg.norm(ob) + 1e-10


# rows longer than the registers hold, at both sides of what is streamed (FP64
# up to 39,000 rows of 79, FP32 up to 66,000), and a single long row among short
# ones; the allocation-free solve has the bits of the FP64 solve on either side
@pytest.mark.parametrize("n,half,long_row", [(30000, 39, 0), (48000, 39, 0), (72000, 39, 0),
                                             (60000, 13, 200), (130000, 13, 200)])
def test_long_rows(oracle, n, half, long_row):
    rp, ci, val, b = _banded(n, half, n)
    if long_row:
        i = np.unique(np.linspace(1, n - 1, long_row).astype(int))
        a = scipy.sparse.csr_matrix((val, ci, rp), (n, n)) + scipy.sparse.coo_matrix(
            (np.full(2 * len(i), -1e-3), (np.r_[np.zeros(len(i), int), i],
                                          np.r_[i, np.zeros(len(i), int)])), (n, n)).tocsr()
        a.sort_indices()
        rp, ci, val = a.indptr.astype(np.int32), a.indices.astype(np.int32), a.data
    with abi.Context(0) as c:
        c.set_csr(rp, ci, val)
        c.set_rhs(b)
        for mode in (abi.SOLVE_MIXED, abi.SOLVE_FP64):
            got = []
            for prof in (0, 1):
                c.set_profiling(prof)
                it, rel, _ = c.solve(mode, abi.FMT_CSR, 1e-9)
                got.append((it, rel, c.get_solution()))
            assert got[0][:2] == got[1][:2]
            assert np.array_equal(got[0][2], got[1][2])
            r = b - oracle.spmv(rp, ci, val, got[0][2])
            assert np.linalg.norm(r) <= 1.001e-9 * np.linalg.norm(b) + 1e-13
    f, hip = noalloc._noalloc(), noalloc._Hip()
    try:
        x = hip.put(np.zeros(n))
        it, rel = C.c_int(), C.c_double()
        assert f(0, None, n, len(ci), *(hip.put(v) for v in (rp, ci, val, b)), x, 1e-9, 10000,
                 C.byref(it), C.byref(rel)) == abi.INS_OK
        assert (it.value, rel.value) == got[0][:2]
        assert np.array_equal(hip.get(x, n, np.float64), got[0][2])
    finally:
        hip.free()
