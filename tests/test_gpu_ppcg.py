"""PCG inside one launch (cs_ppcg.hip) against the separately launched iterations
(CS_FLAG_TIME_KERNELS keeps those), on the same assembled systems, at the sizes where the kernel's
workgroups, registers and launches begin and end."""
import numpy as np
import pytest

from clothsimulator_amd import CS_MESH_CLOTH, Simulator, scenes
from clothsimulator_amd._cabi import (CS_FLAG_FIXED_TUNING, CS_FLAG_INSTANCES, CS_FLAG_TIME_KERNELS, CS_PRECOND_AMG,
                                      CS_PRECOND_AMG_LEARNED, CS_PRECOND_BLOCK_JACOBI, CS_PRECOND_LEARNED, MeshArrays,
                                      default_params, material_struct)

pytestmark = pytest.mark.gpu


def _state(spec, seed=0, amp=2e-3, vel=0.2):
    rng = np.random.default_rng(seed)
    x = spec.cloths[0].mesh.x.astype(np.float64)
    return (np.float32(x + rng.normal(0, amp / np.sqrt(len(x)), x.shape)), np.float32(rng.normal(0, vel, x.shape)))


def _solve(spec, flags, x, v, launches, **params):
    """(solution, stats, assembled system); launches: the cooperative launches the solve must take."""
    p = default_params(dt=spec.params.dt, gravity=tuple(spec.params.gravity))
    p.flags = spec.params.flags | flags
    for k, val in params.items():
        setattr(p, k, val)
    sim = Simulator(spec, params=p)
    sim.set_state(CS_MESH_CLOTH, 0, x, x, v)
    rp, ci, vals, b = sim.assemble(0)
    dv, st = sim.solve(0)
    assert sim.solve_launches() == launches
    return dv.astype(np.float64), st, (rp, ci, vals.astype(np.float64), b.astype(np.float64))


def _residual(system, dv):
    rp, ci, vals, b = system
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    y = np.zeros((len(rp) - 1, 3))
    np.add.at(y, rows, np.einsum("kij,kj->ki", vals, dv.reshape(-1, 3)[ci]))
    return np.linalg.norm(b - y.ravel()) / np.linalg.norm(b)


def _compare(spec, x, v, launches=1, **params):
    """The solve in one launch forms the same sums in the same order: the same bits."""
    a, sa, system = _solve(spec, 0, x, v, launches, **params)
    l, sl, _ = _solve(spec, CS_FLAG_TIME_KERNELS, x, v, 0, **params)
    assert sa.pcg_converged and sl.pcg_converged and sa.pcg_iters == sl.pcg_iters
    assert np.array_equal(a, l)
    # 1e-5 |b|, in FP64 up to the rounding of the assembled values that are read back (static and
    # contact blocks merged in FP32: 1e-7 of |A| |dv| each way)
    assert _residual(system, a) <= 1.2e-5


# one workgroup through LDS up to 512 rows (22: 484, 23: 529), 256-row workgroups: one XCD up to 8 of
# them (45: 2,025, 46: 2,116), up to 24,576 rows (156: 24,336, 157: 24,649), then 512-row ones
@pytest.mark.parametrize("n", [2, 3, 16, 22, 23, 45, 46, 156, 157])
def test_solve_equals_launched(n):
    spec = scenes.hang(n)
    _compare(spec, *_state(spec))


# 9: the smallest hierarchy; 45, 46 and 156, 157 as above; 65: workgroups without rows share the
# multigrid's dense operator; with the learned smoother only cloths without a hierarchy (8).
@pytest.mark.parametrize("precond,n", [(CS_PRECOND_LEARNED, n) for n in (2, 16, 46, 157)] +
                         [(CS_PRECOND_AMG, n) for n in (8, 9, 23, 45, 65, 129, 157)] +
                         [(CS_PRECOND_AMG_LEARNED, n) for n in (8, 9, 33)])
def test_preconditioned_solve_equals_launched(precond, n):
    spec = scenes.crumple(n, height=0.01, sigma=0.05 / n)
    x, v = _state(spec, amp=0.0)
    _compare(spec, x, v, launches=0 if precond == CS_PRECOND_AMG_LEARNED and n > 8 else 1, precond=precond)


@pytest.mark.parametrize("precond", [CS_PRECOND_LEARNED, CS_PRECOND_AMG])
def test_preconditioned_contacts_equal_launched(precond):
    spec = scenes.fold(49, gap=9e-4, noise=5e-5)
    x = spec.cloths[0].mesh.x
    _compare(spec, x, np.zeros_like(x), precond=precond)


def test_multigrid_batch_matches_launched():
    """Sides 5 to 33 in one launch each for the cloths with and without a hierarchy, against the
    launched batch; the coarsest levels are solved the same way."""
    out = []
    for flags, launches in ((0, 2), (CS_FLAG_TIME_KERNELS, 0)):
        spec = scenes.instances(count=6, seed=3, side_lo=5, side_hi=33, gap=8e-4)
        sides = sorted(int(round(np.sqrt(c.mesh.n_nodes))) for c in spec.cloths)
        assert sides[0] <= 8 and sides[-1] > 22
        spec.params.precond = CS_PRECOND_AMG
        spec.params.flags |= flags | CS_FLAG_FIXED_TUNING
        sim = Simulator(spec)
        s, st = sim.physics_step()
        assert s == 0 and st.pcg_rel_residual <= 1e-5 and sim.solve_launches() == launches
        out.append((st.pcg_iters, [sim.state(CS_MESH_CLOTH, k)[0] for k in range(6)]))
    assert abs(out[0][0] - out[1][0]) <= 6
    assert max(np.abs(a - b).max() for a, b in zip(out[0][1], out[1][1])) <= 1e-5


@pytest.mark.parametrize("n,launches", [(362, 1), (363, 0)])
def test_solve_at_the_register_capacity(n, launches):
    """131,044 rows are solved in the launch, 131,769 are not; both meet the tolerance."""
    spec = scenes.crumple(n)
    x, v = _state(spec)
    dv, st, system = _solve(spec, 0, x, v, launches)
    assert st.pcg_converged and _residual(system, dv) <= 1.2e-5


def test_contacts_equal_launched():
    spec = scenes.fold(49, gap=9e-4, noise=5e-5)
    x = spec.cloths[0].mesh.x
    _compare(spec, x, np.zeros_like(x))


@pytest.mark.parametrize("precond", [CS_PRECOND_BLOCK_JACOBI, CS_PRECOND_LEARNED])
def test_rows_wider_than_the_registers(precond):
    """A fan of 40 triangles: its hub's row has 41 blocks, the rim's rows 6 or fewer."""
    k = 40
    a = 2 * np.pi * np.arange(k) / k
    xy = np.concatenate([[[0.0, 0.0]], 0.1 * np.stack([np.cos(a), np.sin(a)], 1)])
    faces = np.array([[0, 1 + i, 1 + (i + 1) % k] for i in range(k)], np.int32)
    mesh = MeshArrays(np.column_stack([xy, np.zeros(k + 1)]), faces)
    spec = scenes.SceneSpec("fan", default_params(), [scenes.ClothSpec(mesh, material_struct())], [], 1)
    _compare(spec, *_state(spec, amp=1e-3), precond=precond)


def test_columns_too_far_for_16_bits_are_solved_by_launches():
    """A 190 x 190 sheet with shuffled nodes: columns further than 32,767 from their row."""
    spec = scenes.hang(190)
    m = spec.cloths[0].mesh
    perm = np.random.default_rng(0).permutation(m.n_nodes)
    inv = np.argsort(perm)
    spec.cloths[0].mesh = MeshArrays(m.x[perm], inv[m.faces].astype(np.int32))
    spec.cloths[0].handles = [int(inv[h]) for h in spec.cloths[0].handles]
    x, v = _state(spec)
    dv, st, system = _solve(spec, 0, x, v, 0)
    assert st.pcg_converged and _residual(system, dv) <= 1.2e-5


@pytest.mark.parametrize("n", [17, 33])
def test_iteration_budget_and_zero_right_hand_side(n):
    spec = scenes.hang(n)
    x, v = _state(spec)
    a, sa, _ = _solve(spec, 0, x, v, 1, pcg_max_iters=7)
    l, sl, _ = _solve(spec, CS_FLAG_TIME_KERNELS, x, v, 0, pcg_max_iters=7)
    assert sa.pcg_iters == sl.pcg_iters == 7 and not sa.pcg_converged and not sl.pcg_converged
    assert np.array_equal(a, l)
    a, sa, _ = _solve(spec, 0, x, v, 1, pcg_max_iters=0)
    assert sa.pcg_iters == 0 and not sa.pcg_converged and not a.any()
    still = scenes.hang(n)
    still.params = default_params(gravity=(0.0, 0.0, 0.0))
    m = still.cloths[0].mesh
    a, sa, _ = _solve(still, 0, m.x, np.zeros_like(m.x), 1)
    assert sa.pcg_iters == 0 and sa.pcg_converged and not a.any()


# one launch; two launches (about 150,000 rows); more than two, which the separate kernels solve
@pytest.mark.parametrize("count,lo,hi,launches", [(5, 9, 40, 1), (3, 17, 22, 1), (24, 70, 90, 2), (48, 100, 129, 0)])
def test_batches_match_separate_runs(count, lo, hi, launches):
    spec = scenes.instances(count=count, seed=2, side_lo=lo, side_hi=hi, gap=8e-4)
    assert spec.params.flags & CS_FLAG_INSTANCES
    batch = Simulator(spec)
    s, st = batch.physics_step()
    assert s == 0 and st.pcg_rel_residual <= 1e-5 and batch.solve_launches() == launches
    for k in sorted({0, count // 2, count - 1}):
        one = Simulator(scenes.SceneSpec("one", default_params(dt=spec.params.dt), [spec.cloths[k]],
                                         [spec.obstacles[k]], 1))
        s, _ = one.physics_step()
        assert s == 0
        a, b = one.state()[0], batch.state(CS_MESH_CLOTH, k)[0]
        if launches:  # in one launch or alone: the same bits
            assert np.array_equal(a, b), (k, np.abs(a - b).max())
        assert np.abs(a - b).max() <= 1e-5


def test_two_runs_give_the_same_bits():
    spec = scenes.drape(65)
    x, v = _state(spec)
    a, _, _ = _solve(spec, 0, x, v, 1)
    b, _, _ = _solve(spec, 0, x, v, 1)
    assert np.array_equal(a, b)


def test_contexts_on_several_threads_solve_at_once():
    """Four contexts stepped at once by four threads (their launches need the whole chip, or share it with
    the others' kernels) give the steps each gives alone, and every solve stays in one launch."""
    import threading
    specs = [scenes.drape(65), scenes.hang(33), scenes.crumple(129, height=0.01, sigma=0.05 / 129), scenes.hang(17)]
    specs[0].params.precond = CS_PRECOND_AMG
    specs[1].params.precond = CS_PRECOND_LEARNED

    def steps(k, out):
        sim = Simulator(specs[k])
        launches = []
        for _ in range(6):
            s, _ = sim.step()
            launches.append((s, sim.solve_launches()))
        out[k] = (sim.state()[0], sim.state()[2], launches)

    alone, together = {}, {}
    for k in range(4):
        steps(k, alone)
    threads = [threading.Thread(target=steps, args=(k, together)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(4):
        assert together[k][2] == [(0, 1)] * 6
        assert np.array_equal(alone[k][0], together[k][0]) and np.array_equal(alone[k][1], together[k][1])


def _fault_case(case):
    """(spec, two states) of a system in the one-launch range with several workgroups."""
    if case == "batch":
        spec = scenes.instances(count=3, seed=3, side_lo=23, side_hi=40)
        spec.params.flags |= CS_FLAG_FIXED_TUNING
        return spec
    spec = scenes.crumple(33, height=0.01, sigma=0.05 / 33)
    spec.params.precond = {"jacobi": CS_PRECOND_BLOCK_JACOBI, "learned": CS_PRECOND_LEARNED, "amg": CS_PRECOND_AMG}[case]
    return spec


def _solve_after_another(case, flags=0, **fault):
    """A solve right after one of another system on the same context (what it leaves in the buffers is
    no solution here): (solution, iterations, launches)."""
    spec = _fault_case(case)
    spec.params.flags |= flags
    sim = Simulator(spec)
    for seed in (1, 2):
        rng = np.random.default_rng(seed)
        for k in range(sim.n_cloths):
            x = sim.state(CS_MESH_CLOTH, k)[0]
            sim.set_state(CS_MESH_CLOTH, k, x, x, np.float32(rng.normal(0, 0.2, x.shape)))
        if seed == 2:
            assert sim.solve_launches() == (0 if flags else 1)
            sim.set_launch_fault(**fault)
        if case == "batch":
            s, st = sim.physics_step()
            assert s == 0
            dv = np.concatenate([sim.state(CS_MESH_CLOTH, k)[2].ravel() for k in range(sim.n_cloths)])
        else:
            sim.assemble(0)
            dv, st = sim.solve(0)
        assert st.pcg_converged
    return dv, st.pcg_iters, sim.solve_launches()


@pytest.mark.parametrize("case", ["jacobi", "learned", "amg", "batch"])
def test_a_refused_launch_falls_back(case):
    dv, it, launches = _solve_after_another(case, refuse=1)
    ref, rit, _ = _solve_after_another(case, CS_FLAG_TIME_KERNELS)
    assert launches == 0 and it == rit and np.array_equal(dv, ref)


@pytest.mark.parametrize("case", ["jacobi", "learned", "amg", "batch"])
@pytest.mark.parametrize("at", [1, 2, 7, 30])
def test_a_workgroup_that_gives_up_falls_back(case, at):
    """Its peers' next wait runs out (bounded to 5 ms here); the solve is repeated in separate launches."""
    dv, it, launches = _solve_after_another(case, lose_wg=1, lose_at=at, wait_s=5e-3)
    ref, rit, _ = _solve_after_another(case, CS_FLAG_TIME_KERNELS)
    assert launches == 0 and it == rit and np.array_equal(dv, ref)


@pytest.mark.parametrize("fault,pauses", [({"refuse": 1}, (1, 3)), ({"lose_wg": 1, "lose_at": 3, "wait_s": 2e-3}, (255,))])
def test_one_launch_is_tried_again_after_a_pause(fault, pauses):
    """A refusal passes: the solves after it take separate launches (1, then 3, ... while it is refused
    again), then the launch is tried again.  A wait that ran out pauses it for 255 solves."""
    sim = Simulator(scenes.hang(23))  # three workgroups
    sim.assemble(0)

    def launches():
        sim.solve(0)
        return sim.solve_launches()

    assert launches() == 1
    for n in pauses:
        sim.set_launch_fault(**fault)
        assert launches() == 0
        if n == pauses[-1]:
            sim.set_launch_fault()
        assert [launches() for _ in range(n)] == [0] * n
    assert [launches() for _ in range(3)] == [1] * 3
    sim.set_launch_fault(refuse=1)  # a success ends the doubling
    assert launches() == 0
    sim.set_launch_fault()
    assert [launches() for _ in range(2)] == [0, 1]


def test_a_workgroup_that_gives_up_at_the_last_meeting_is_noticed():
    """At the last meeting no peer waits for the lost workgroup again, and the record is complete: only
    the lost workgroup's own word tells.  A block-Jacobi solve of i iterations meets 2 i + 3 times, and
    three times more per continuation from the true residual."""
    ref, it, _ = _solve_after_another("jacobi", CS_FLAG_TIME_KERNELS)
    ran = []
    for at in [2 * it + 3 + 3 * k for k in range(5)] + [2 * it + 4 + 3 * k for k in range(5)]:
        dv, i, launches = _solve_after_another("jacobi", lose_wg=1, lose_at=at, wait_s=5e-3)
        assert i == it and np.array_equal(dv, ref), at
        ran.append((at, launches))
    last = max(at for at, launches in ran if launches == 0)
    assert (last + 1, 1) in ran  # one later is never reached: `last` was the last meeting
