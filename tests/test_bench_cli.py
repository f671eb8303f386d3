"""CPU tests of bench.py's command-line contract: more than one GPU is refused with a
message (this build runs on one GPU), before anything touches a GPU."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_multi_gpu_is_refused():
    p = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2", "--steps", "1", "--warmup", "0"],
                       capture_output=True, text=True, timeout=300, cwd=ROOT)
    assert p.returncode == 2
    assert "one GPU" in p.stderr and "--gpus 2" in p.stderr


def test_world_size_env_is_refused():
    env = dict(os.environ, WORLD_SIZE="4")
    p = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py")], capture_output=True, text=True, timeout=300,
                       cwd=ROOT, env=env)
    assert p.returncode == 2


def test_timed_region_runs_without_a_stage_recorder():
    """The timed forwards are what a user runs (a recorder takes a layer to its separate
    launches); every EVENT_EVERY-th of the forwards behind them is sampled."""
    import bench
    from kmoe import ops

    seen = []
    step = lambda: seen.append(ops.stage_timing())
    assert bench.time_forwards(step, 7, lambda: seen.append("sync")) > 0
    assert seen == ["sync"] + [False] * 7 + ["sync"]
    seen.clear()
    bench.sample_gate_up(step, 11, lambda: None)
    assert [i for i, on in enumerate(seen) if on] == [0, bench.EVENT_EVERY, 2 * bench.EVENT_EVERY]
    assert not ops.stage_timing()
