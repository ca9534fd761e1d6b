"""cs_solve_bsr_noalloc (the solve that allocates nothing) against cs_solve, through the C-ABI.

Two calls in a row on one GPU, the second on a smaller system, each on the system a context
assembled (hang33, then hang17, four steps in): the result is within what cs_solve's own
tolerance allows (positions x = x0 + dt (v + dv) within 1e-5 m of cs_solve's, so |dv| within
1e-5 / dt), meets the 1e-5 residual in FP64 on the host, and takes the same iteration count
within two (the same algorithm; only the summation order differs).  The device buffers are
made by the test (hipMalloc through the library's own HIP runtime); the entry point itself
allocates nothing.
"""
import ctypes as C

import numpy as np
import pytest

from clothsimulator_amd import Simulator, load_library, scenes
from clothsimulator_amd._cabi import CS_E_ARG, CS_E_CAPACITY, CS_OK, LaunchFault

pytestmark = pytest.mark.gpu

MAX_NODES = 65536  # CS_NOALLOC_MAX_NODES


def _hip():
    """The HIP runtime the library itself runs on (already loaded by it)."""
    H = C.CDLL("libamdhip64.so.7")
    H.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    H.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    H.hipFree.argtypes = [C.c_void_p]
    return H


class DeviceArray:
    """A device copy of a host array, made and freed by the test (hipMalloc / hipMemcpy)."""

    def __init__(self, host):
        self.H = _hip()
        self.host = np.ascontiguousarray(host)
        self.ptr = C.c_void_p()
        assert self.H.hipMalloc(C.byref(self.ptr), max(self.host.nbytes, 4)) == 0
        assert self.H.hipMemcpy(self.ptr, self.host.ctypes.data, self.host.nbytes, 1) == 0  # host to device

    def get(self):
        out = np.empty_like(self.host)
        assert self.H.hipMemcpy(out.ctypes.data, self.ptr, out.nbytes, 2) == 0  # device to host
        return out

    def __del__(self):
        self.H.hipFree(self.ptr)


def _noalloc(rp, ci, vals, b, tol=1e-5, maxit=4000, entry="cs_solve_bsr_noalloc", more=()):
    """(status, x, iterations, residual)"""
    solve = getattr(load_library(), entry)
    drp, dci = DeviceArray(rp.astype(np.int32)), DeviceArray(ci.astype(np.int32))
    dvals, db = DeviceArray(vals.reshape(-1).astype(np.float32)), DeviceArray(b.astype(np.float32))
    dx = DeviceArray(np.full(len(b), np.nan, np.float32))
    it, rel = C.c_int(-1), C.c_float(-1.0)
    st = solve(None, len(rp) - 1, drp.ptr, dci.ptr, dvals.ptr, db.ptr, dx.ptr, tol, maxit, C.byref(it), C.byref(rel),
               *more)
    return st, dx.get(), it.value, rel.value


def _noalloc_launches(rp, ci, vals, b, **fault):
    """(status, x, iterations, residual, launches that held the iterations); fault: how the launch fails."""
    launches = C.c_int(-1)
    out = _noalloc(rp, ci, vals, b, entry="cs_solve_bsr_noalloc_test",
                   more=(C.byref(LaunchFault(**fault)), C.byref(launches)))
    return *out, launches.value


def test_noalloc_solve_matches_cs_solve_on_two_calls():
    import scipy.sparse as sp
    for n in (33, 17):  # the second call on a smaller system
        spec = scenes.hang(n)
        sim = Simulator(spec)
        s, _ = sim.run(4)
        assert s == CS_OK
        rp, ci, vals, b = sim.assemble(0)
        dv, st = sim.solve(0)
        status, x, iters, rel = _noalloc(rp, ci, vals, b)
        A = sp.bsr_matrix((vals.astype(np.float64), ci, rp), shape=(len(b), len(b)))
        res = np.linalg.norm(b.astype(np.float64) - A @ x.astype(np.float64)) / np.linalg.norm(b)
        dt = spec.params.dt
        dx = dt * float(np.abs(x - dv).max())
        print("hang%d: cs_solve %d iterations, no-alloc %d (status %d, recursive %.3g, FP64 %.3g); "
              "positions differ by %.3g m" % (n, st.pcg_iters, iters, status, rel, res, dx))
        assert status == CS_OK
        assert np.isfinite(x).all()
        assert res <= 2e-5 and rel <= 1e-5
        # cs_solve confirms its stop on the true residual and, when that misses, continues a little
        # below the tolerance; the no-alloc solve stops on its recursive residual
        assert iters <= st.pcg_iters + 2 and st.pcg_iters <= max(iters + 2, 1.1 * iters)
        assert dx <= 1e-5
        sim.close()


def test_noalloc_rejects_oversize_and_malformed_systems():
    L = load_library()
    it = C.c_int()
    # beyond the fixed scratch: rejected before any pointer is read
    assert L.cs_solve_bsr_noalloc(None, MAX_NODES + 1, None, None, None, None, None, 1e-5, 10, C.byref(it),
                                  None) == CS_E_CAPACITY
    assert L.cs_solve_bsr_noalloc(None, 0, None, None, None, None, None, 1e-5, 10, None, None) == CS_E_ARG
    # a row without its diagonal block, and a column out of range
    rp = np.array([0, 1, 2], np.int32)
    b = np.ones(6, np.float32)
    vals = np.tile(np.eye(3, dtype=np.float32).reshape(1, 9), (2, 1))
    for ci in (np.array([1, 0], np.int32), np.array([0, 5], np.int32)):
        status, _, _, _ = _noalloc(rp, ci, vals, b)
        assert status == CS_E_ARG
    # the same arrays with valid columns solve (identity system: one iteration)
    status, x, iters, _ = _noalloc(rp, np.array([0, 1], np.int32), vals, b)
    assert status == CS_OK and iters == 1 and np.allclose(x, 1.0)


def _band(n, reach):
    """A symmetric, diagonally dominant system with rows of up to 2 reach + 1 blocks."""
    rng = np.random.default_rng(n + reach)
    rp, ci, vals = [0], [], []
    off = rng.uniform(-0.5, 0.5, (n, reach + 1))  # symmetric couplings i, i + k
    for i in range(n):
        for j in range(max(0, i - reach), min(n, i + reach + 1)):
            ci.append(j)
            vals.append(np.eye(3) * (2.0 + reach) if i == j else np.eye(3) * off[min(i, j), abs(i - j)])
        rp.append(len(ci))
    rp, ci = np.array(rp, np.int32), np.array(ci, np.int32)
    vals = np.array(vals, np.float32)
    b = rng.standard_normal(3 * n).astype(np.float32)
    return rp, ci, vals, b


@pytest.mark.parametrize("n,reach", [(1, 0), (2, 1), (255, 3), (256, 6), (257, 7), (1000, 20), (65536, 1)])
def test_noalloc_sizes_and_row_lengths(n, reach):
    """One workgroup to all 256 of them; rows of up to 2 reach + 1 blocks, 14 of which are in
    registers.  The stop is on the true residual (FP64 row sums), so in FP64 it holds up to the
    rounding of the squared norms: 1e-5 (1 + 1e-4)."""
    import scipy.sparse as sp
    rp, ci, vals, b = _band(n, reach)
    status, x, iters, rel, launches = _noalloc_launches(rp, ci, vals, b)
    assert launches >= 1
    A = sp.bsr_matrix((vals.astype(np.float64), ci, rp), shape=(3 * n, 3 * n))
    res = np.linalg.norm(b - A @ x.astype(np.float64)) / np.linalg.norm(b)
    print("%d rows, reach %d: status %d, %d iterations, residual %.3g, in FP64 %.3g" % (n, reach, status, iters, rel, res))
    assert status == CS_OK
    assert res <= 1e-5 * (1 + 1e-4) and abs(res - rel) <= 1e-4 * rel + 1e-9
    # the iteration budget is kept, and spending it is reported
    if iters > 2:
        status, x, iters, rel = _noalloc(rp, ci, vals, b, maxit=2)
        assert status != CS_OK and iters == 2 and np.isfinite(x).all()


def test_noalloc_launch_that_fails_is_repeated_separately():
    """A refused launch, and a workgroup that gives up at any meeting of the 2 i of i iterations (its peers'
    next wait runs out, 5 ms here; after the last there is none): the separate launches' result, bit for
    bit that of the one launch.  The calls after it take separate launches too, one after a refusal and 255
    after a wait that ran out, then the launch is tried again."""
    small = _band(2, 1)
    rp, ci, vals, b = _band(1000, 20)  # four workgroups, rows of more blocks than the registers hold
    status, ref, iters, rel, launches = _noalloc_launches(rp, ci, vals, b)
    assert status == CS_OK and launches == 1
    for fault in [{"refuse": 1}] + [{"lose_wg": 1, "lose_at": at, "wait_s": 5e-3}
                                    for at in (1, 2, 2 * iters - 1, 2 * iters, 2 * iters + 1)]:
        s, x, i, r, launches = _noalloc_launches(rp, ci, vals, b, **fault)
        assert launches == (1 if fault.get("lose_at") == 2 * iters + 1 else 0), fault
        assert (s, i, r) == (status, iters, rel) and np.array_equal(x, ref), fault
        pause = 0 if launches else 1 if "refuse" in fault else 255
        assert all(_noalloc_launches(*small)[4] == 0 for _ in range(pause)), fault
        assert _noalloc_launches(*small)[4] >= 1, fault


@pytest.mark.parametrize("n,launched", [(256, False), (257, True)])
def test_noalloc_rows_too_wide_for_one_launch(n, launched):
    """One row and column full (n blocks in row 0): up to 256 blocks in one launch, more in separate ones;
    the same bits either way."""
    rng = np.random.default_rng(n)
    rows = [sorted({0, i} | ({i - 1} if i > 1 else set()) | ({i + 1} if 0 < i < n - 1 else set())) for i in range(n)]
    rows[0] = list(range(n))
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    ci = np.concatenate(rows).astype(np.int32)
    diag = ci == np.repeat(np.arange(n), np.diff(rp))
    # couplings of -0.02: row 0's sum to 0.02 n < 16, the others' to 0.06 < 4 (positive definite)
    vals = np.where(diag[:, None], 4.0, -0.02) * np.eye(3).reshape(1, 9)
    vals[0] *= 4.0
    b = rng.standard_normal(3 * n).astype(np.float32)
    status, x, iters, rel, launches = _noalloc_launches(rp, ci, vals.astype(np.float32), b)
    assert status == CS_OK and (launches == 0) == launched
    other = _noalloc_launches(rp, ci, vals.astype(np.float32), b, refuse=1)
    assert other[4] == 0 and other[0] == status and other[2:4] == (iters, rel) and np.array_equal(other[1], x)
    assert _noalloc_launches(*_band(2, 1))[4] == 0 and _noalloc_launches(*_band(2, 1))[4] >= 1  # the pause after it
