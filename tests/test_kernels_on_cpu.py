"""What the waves of the solvers' kernels may do to each other, on the CPU: the kernels' own text is
compiled for the CPU (tests/emulate) and run under a scheduler that takes the waves in any order and
leaves some aside for long times.  The results must not depend on it."""
import ctypes as C
import os
import platform
import re
import shutil
import subprocess

import numpy as np
import pytest

import part_model as P
from freecappuccino_amd import mesh as M
from oracle import oracle as O

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))
CSRC = os.path.join(ROOT, "freecappuccino_amd", "csrc")
EMULATE = os.path.join(ROOT, "tests", "emulate")
CLANG = shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"
MARK = {8: 0x7FF4DEADBEEF0001, 4: 0x7FA0BEEF}


def _cut(name, start, end):
    with open(os.path.join(CSRC, name)) as f:
        text = f.read()
    i = text.index(start)
    return text[i:text.index(end, i)]


def _cuts():
    yield "cut_syncfree.inc", (_cut("fcap_linalg.h", "constexpr int kSfTickets", "// zeroed state") +
                               _cut("fcap_syncfree.h", "// A wait is bounded", "}  // namespace fcap"))
    # (the compiler barrier that keeps a wave's LDS accesses in order is a meeting of its lanes here)
    yield "cut_parts.inc", re.sub(r'__asm__ volatile\("" ::: "memory"\);', "emu::meet(emu::kPoint);",
                                  _cut("fcap_parts.hip", "constexpr int kBlock", "// " + "-" * 65 + " analysis"))
    yield "cut_rows.inc", _cut("fcap_linalg.hip", "// " + "-" * 43 + " dependency-driven sweeps",
                               "// The pivot recurrences")
    yield "cut_slices.inc", (_cut("fcap_linalg.h", "struct SliceView", "SliceView slices_for") +
                             _cut("fcap_slices.hip", "constexpr unsigned kPad", "template <class T, int MODE>\nvoid sliced"))
    yield "cut_solver.inc", _cut("fcap_solvers.hip", "// the end of an iteration with", "// " + "-" * 65 + " helpers")


class Run(C.Structure):
    _fields_ = [("grid", C.c_int), ("seed", C.c_int), ("resident", C.c_int), ("freeze_steps", C.c_int),
                ("freeze", C.c_double), ("freeze_store", C.c_double), ("wait_ticks", C.c_longlong), ("max_steps", C.c_longlong),
                ("order", C.c_void_p)]


def _run(grid, seed=1, freeze=0.0, freeze_store=0.0, freeze_steps=1, resident=0, wait_ticks=10**9, max_steps=3 * 10**6, order=None):
    return Run(grid, seed, resident, freeze_steps, freeze, freeze_store, wait_ticks, max_steps,
               None if order is None else order.ctypes.data)


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    if not os.path.exists(CLANG) or platform.machine() != "x86_64":
        pytest.skip("needs clang++ and x86-64")
    d = str(tmp_path_factory.mktemp("emulate"))
    for name, text in _cuts():
        with open(os.path.join(d, name), "w") as f:
            f.write(text)
    lib = os.path.join(d, "kernels.so")
    p = subprocess.run([CLANG, "-std=c++17", "-O1", "-fPIC", "-shared", "-ffp-contract=off", "-w", "-I", d, "-I",
                        EMULATE, "-I", CSRC, "-I", os.path.join(ROOT, "include"),
                        os.path.join(EMULATE, "kernels.cpp"), "-o", lib], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr[-4000:]
    return C.CDLL(lib)


def _matrix(ioffset, ja, diag, seed):
    """The structure as the oracle takes it, symmetric values and a right-hand side."""
    csr = O.CSR(ioffset, ja, diag, np.zeros(0, np.int32), np.zeros(0, np.int32))
    rng = np.random.default_rng(seed)
    n = len(diag)
    row = np.repeat(np.arange(n), np.diff(ioffset))
    key = np.minimum(row, ja - 1) * n + np.maximum(row, ja - 1)
    a = -rng.uniform(0.5, 1.0, key.size)[np.unique(key, return_inverse=True)[1]]
    a[diag - 1] = 20.0 + rng.uniform(0, 1, n)
    return csr, a, rng.standard_normal(n)


def _mesh(m):
    csr = O.csr_build(m.n_cells, m.owner[:m.n_inner] + 1, m.neighbour + 1)
    return csr.ioffset, csr.ja, csr.diag


def _ptr(x):
    return x.ctypes.data_as(C.c_void_p)


def _part_sweeps(emu, s, width, a, d, r, small, dtype, run):
    """Both sweeps of the schedule s; (result, forward's and backward's outputs after it, return codes)."""
    mark = np.uint64(MARK[8]) if dtype == np.float64 else np.uint32(MARK[4])
    marks = lambda: np.full(s.npk, mark).view(dtype)  # noqa: E731
    tmp, zp, z = marks(), np.zeros(s.npk, dtype), np.zeros(len(r), dtype)
    rhs, rc = r.astype(dtype), []
    for upper, (src, out, mk) in enumerate(((rhs, tmp, zp), (tmp, zp, tmp))):
        codes = P.packed(s.codes(bool(upper), width, emu.emu_ring()))
        vals = P.packed(s.values(bool(upper), width, a, d, dtype))
        rc.append(emu.emu_parts(C.byref(run), dtype == np.float32, width, upper, s.nparts, s.npk, _ptr(codes),
                                _ptr(s.step), _ptr(s.win), _ptr(vals), _ptr(src), C.c_double(small), _ptr(out),
                                _ptr(mk), _ptr(z)))
    return z, tmp, mark, rc


def _cases():
    yield "pencils", _mesh(M.hex_box(70, 13, 7)), 3, P.pencil_parts
    yield "runs", _mesh(M.tet_box(8)), 4, lambda *zero: P.run_parts(*zero, 2100)
    yield "wide", P.stencil((6, 6, 65), P.STEPS8), 8, lambda *zero: P.run_parts(*zero, 1900)


@pytest.mark.parametrize("name,structure,width,parts", list(_cases()), ids=lambda v: v if isinstance(v, str) else "")
def test_part_sweeps_whatever_the_waves_do(emu, name, structure, width, parts):
    """Feeders, pollers and the chain wave left aside at any point of theirs, above all behind a flag
    they set, in one workgroup for all parts or one for each: the oracle's sweeps bit for bit, and the forward sweep's output marked again.  (Read from
    the ring behind its flag, a feeder's result was that of a window sixteen further on.)"""
    csr, a, r = _matrix(*structure, 3)
    zero = csr.ioffset - 1, csr.ja - 1, csr.diag - 1
    s = P.Schedule(*zero, *parts(*zero))
    assert s.nparts > 1 and np.diff(s.win).max() > 32
    d = O.dic_pivots(csr, a)
    ref = O.lu_apply(csr, a, d, r)
    for seed in range(8):
        run = _run(grid=1 + seed % 3, seed=seed, freeze=0.003, freeze_store=0.03, freeze_steps=3000)
        z, tmp, mark, rc = _part_sweeps(emu, s, width, a, d, r, 1e-20, np.float64, run)
        assert rc == [0, 0], rc
        np.testing.assert_array_equal(z, ref, err_msg=f"seed {seed}")
        assert np.all(tmp.view(mark.dtype) == mark)


@pytest.mark.parametrize("late", [0.7, 0.9])
def test_the_limit_is_that_of_one_wait(emu, late):
    """A part whose first window's inputs come late, and its second's as late after that: each wait is
    within the limit, so the sweep ends well -- the second's is not charged with the time in which the
    part had not begun.  One wait past the limit ends the sweep with an error."""
    limit, windows = 20000, 6
    n = 64 * windows
    rows = np.arange(n)
    codes = np.full((4, n + 128), emu.emu_ring(), np.int32)
    codes[3, :n] = rows                                   # every row reads one value of another part,
    outside = n + np.arange(n) % 64 + 64 * (rows >= 64)   # first window's and the others' of their own
    codes[0, :n] = (outside | 0x80000000).astype(np.uint32).view(np.int32)
    vals = np.ones((4, n + 128))
    step, win = np.zeros(n + 128, np.uint8), np.array([0, windows], np.int32)
    rng = np.random.default_rng(1)
    rhs, fed = rng.standard_normal(n + 128), rng.standard_normal(128)
    for second, rc in ((late, 0), (1.2, 1)):
        out = np.full(n + 128, np.uint64(MARK[8])).view(np.float64)
        when = np.repeat([int(late * limit), int((late + second) * limit)], 64).astype(np.int64)
        at = (n + np.arange(128)).astype(np.int32)
        run = _run(1, wait_ticks=limit)
        assert emu.emu_parts_fed(C.byref(run), n + 128, _ptr(P.packed(codes)), _ptr(step), _ptr(win),
                                 _ptr(P.packed(vals)), _ptr(rhs), _ptr(out), _ptr(np.zeros(n + 128)), 128, _ptr(at),
                                 _ptr(fed), _ptr(when)) == rc
        if rc == 0:
            np.testing.assert_array_equal(out[:n], rhs[:n] - fed[outside - n])


def _levels(csr, upper):
    """Rows by (level, row) and each one's entries, as the row-wise sweeps have them packed."""
    ptr, ja, diag = csr.ioffset - 1, csr.ja - 1, csr.diag - 1
    n = len(diag)
    lev = np.zeros(n, int)
    rng = range(n - 1, -1, -1) if upper else range(n)
    part = lambda i: slice(diag[i] + 1, ptr[i + 1]) if upper else slice(ptr[i], diag[i])  # noqa: E731
    for i in rng:
        lev[i] = lev[ja[part(i)]].max(initial=-1) + 1
    return np.lexsort((np.arange(n), lev)), part


def _row_sweeps(emu, csr, a, d, r, width, run):
    n, small, arrays = len(r), 1e-20, []
    for upper in (False, True):
        rows, part = _levels(csr, upper)
        cnt, col, val = np.zeros(n, np.int32), np.zeros((width, n), np.int32), np.zeros((width, n))
        for p, i in enumerate(rows):
            c = part(i).stop - part(i).start
            cnt[p], col[:c, p], val[:c, p] = c, csr.ja[part(i)] - 1, a[part(i)]
        arrays.append((rows.astype(np.int32), cnt, col, val, d[rows]))
    two = lambda k: (C.c_void_p * 2)(arrays[0][k].ctypes.data, arrays[1][k].ctypes.data)  # noqa: E731
    tmp = np.full(n, np.uint64(MARK[8])).view(np.float64)
    w = np.zeros(n)
    rc = emu.emu_rows(C.byref(run), width, n, two(0), two(1), two(2), two(3), two(4), _ptr(r), C.c_double(small),
                      _ptr(tmp), _ptr(w))
    return rc, w, tmp


@pytest.mark.parametrize("grid,resident,reverse", [(16, 3, False), (40, 5, True), (16, 1, False), (9, 0, False),
                                                   (8, 8, True), (7, 0, False), (2, 1, True), (1, 0, False)])
@pytest.mark.parametrize("name,structure,width", [("box", _mesh(M.hex_box(14, 9, 8)), 3),
                                                  ("wide", P.stencil((9, 8, 9), P.STEPS8), 8)],
                         ids=lambda v: v if isinstance(v, str) else "")
def test_row_sweeps_need_no_workgroup_but_the_running_ones(emu, name, structure, width, grid, resident, reverse):
    """Workgroups that start when others have ended, fewer at once than there are block counters, the
    first ones last: whichever run compute every row they wait for themselves (the oracle's sweeps bit
    for bit), and the forward sweep's output is marked again."""
    csr, a, r = _matrix(*structure, 5)
    d = O.dic_pivots(csr, a)
    ref = O.lu_apply(csr, a, d, r)
    order = np.arange(grid, dtype=np.uint32)[::-1 if reverse else 1].copy()
    for seed in range(3):
        run = _run(grid, seed=seed, freeze=0.003 * seed, freeze_steps=2000, resident=resident, wait_ticks=10**6,
                   order=order)
        rc, w, tmp = _row_sweeps(emu, csr, a, d, r, width, run)
        assert rc == 0, "a wait ran past its limit" if rc == 1 else "no end"
        np.testing.assert_array_equal(w, ref, err_msg=f"seed {seed}")
        assert np.all(tmp.view(np.uint64) == np.uint64(MARK[8]))


@pytest.mark.parametrize("bicg", [0, 1])
@pytest.mark.parametrize("converged", [True, False])
def test_every_block_ends_the_solve_alike(emu, bicg, converged):
    """The kernel that begins an iteration tests for convergence in every block, and one block sets
    `done`, which all of them read first.  Whatever waves are late, the direction is whole: as it was
    where the solve ends (the refinement cycles carry it on), every entry new where it goes on."""
    n, grid, nv = 2000, 4, 40
    rng = np.random.default_rng(2)
    p0, z = rng.standard_normal((2, n)).astype(np.float32)
    want, done = None, C.c_int()
    for seed in range(60):
        p = p0.copy()
        run = _run(grid, seed=seed, freeze=0.0 if seed == 0 else 0.05, freeze_steps=400)
        assert emu.emu_begin(C.byref(run), bicg, n, _ptr(p), _ptr(z), C.c_double(1e-6 if converged else 1.0),
                             C.c_double(1.0), C.c_double(1e-3), nv, C.byref(done)) == 0
        assert done.value == converged
        if seed == 0:
            want = p0 if converged else p.copy()
            assert converged or np.all(p != p0)
        np.testing.assert_array_equal(p, want, err_msg=f"seed {seed}")


@pytest.mark.parametrize("n,spread,longest", [(1, 1, 1), (64, 5, 4), (65, 40, 5), (255, 9, 7), (700, 300, 8),
                                              (70001, 70000, 5), (3000, 200, 7)])
def test_single_precision_products_in_slices(emu, n, spread, longest):
    """FP32 products, their partials and damped-Jacobi steps over slices: the row's entries one by one
    in order, in the precision of the CSR kernels, bit for bit.  Columns within 16 bits of each other
    and, with 70,001 rows, beyond (wide slices); ragged rows and last slices."""
    rng = np.random.default_rng(n)
    cnt = rng.integers(1, longest + 1, n)
    ptr = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32)
    row = np.repeat(np.arange(n), cnt)
    ja = np.clip(row + rng.integers(-spread, spread + 1, row.size), 0, n - 1).astype(np.int32)
    a = rng.standard_normal(row.size)
    x, b = rng.standard_normal((2, n)).astype(np.float32)
    d = (1.0 + rng.random(n)).astype(np.float32)
    a32 = a.astype(np.float32)
    grid = -(-n // 256)
    for mode in (2, 3, 4):
        y, pa, pb = np.zeros(n, np.float32), np.zeros(grid), np.zeros(grid)
        wide = emu.emu_sliced32(mode, n, max(4, longest), _ptr(ptr), _ptr(ja), _ptr(a), _ptr(x), _ptr(b), _ptr(d),
                                _ptr(y), _ptr(pa), _ptr(pb))
        assert (wide > 0) == (spread > 65535)
        acc = b.copy() if mode == 4 else np.zeros(n, np.float32)
        for k in range(longest):
            has = k < cnt
            p = a32[ptr[:-1][has] + k] * x[ja[ptr[:-1][has] + k]]
            acc[has] = acc[has] - p if mode == 4 else acc[has] + p
        want = x + np.float32(0.7) * (acc / d) if mode == 4 else acc
        np.testing.assert_array_equal(y, want, err_msg=f"mode {mode}")
        if mode != 4:
            starts = np.arange(0, n, 256)
            np.testing.assert_allclose(pa, np.add.reduceat(acc.astype(float) * b, starts), rtol=0, atol=1e-11 * n)
        if mode == 3:
            np.testing.assert_allclose(pb, np.add.reduceat(acc.astype(float) ** 2, starts), rtol=1e-13)
