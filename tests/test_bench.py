"""bench.py's line without a GPU: which runs its figures come from."""
import json
import sys

import bench


def test_reported_figures_come_from_runs_without_kernel_sampling(monkeypatch, capsys):
    """Sampling kernels keeps solves out of the one launch that users get, so every reported rate is of a
    run without it, and the sampled run gives the roofline alone."""
    from clothsimulator_amd import scenes
    calls = []

    def run(workload, precond, steps, warmup, timed, extra_flags=0):
        calls.append((precond, timed))
        seconds = 7.0 if timed else {"jacobi": 2.0, "amg": 1.0}[precond]
        spec = scenes.by_name(workload)
        r = {"spec": spec, "elapsed": seconds, "iters": [3] * steps, "contacts": [0] * steps, "failed": 0,
             "failures": [], "one_launch": 0 if timed else steps, "value": spec.n_cloth_nodes * steps / seconds,
             "ms_per_step": 1e3 * seconds / steps, "span": steps, "timed": steps}
        if timed:
            r.update(spmv=(1.0, 10), pair=(0.5, 10))
        return r

    monkeypatch.setattr(bench, "run", run)
    monkeypatch.setattr(sys, "argv", ["bench.py", "--workload", "hang33", "--steps", "4", "--precond", "amg",
                                      "--compare", "jacobi,amg", "--no-cpu"])
    bench.main()
    out = json.loads(capsys.readouterr().out.strip().splitlines()[-1])
    assert sorted(calls) == [("amg", False), ("amg", True), ("jacobi", False)]
    assert out["ms_per_step"] == 250.0 and out["block_jacobi"]["ms_per_step"] == 500.0
    assert out["speedup_vs_jacobi"] == 2.0
    assert out["steps_solved_in_one_launch"] == 4
    assert out["roofline"]["launches_sampled"] == 10 and abs(out["roofline"]["avg_us"] - 50.0) < 1e-9
