"""bench.py's command line without a GPU: the help lists every workload and
the observables switch, and a request for more than one GPU ends with a
message and exit status 2 before anything touches a device."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(*args):
    return subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), *args], capture_output=True, text=True,
                          timeout=120, cwd=ROOT)


def test_help_lists_workloads_and_observables():
    out = _run("--help")
    assert out.returncode == 0
    for word in ("config2", "config3", "config4", "--observables", "--converge", "--saturate"):
        assert word in out.stdout


def test_more_than_one_gpu_is_refused():
    out = _run("--gpus", "2")
    assert out.returncode == 2
    assert "one GPU" in out.stderr


@pytest.mark.parametrize("args,kernel,lanes", [
    ([], "k_sweep_tree<Ising>", 16), (["--observables", "1"], "k_sweep_tree<Ising>", 16),
    (["--observables", "2"], "k_sweep_tree<Ising>", 16), (["--sweep-kernel", "3"], "k_sweep_tuned<Ising>", 1),
    (["--producers", "3"], "k_sweep_tuned<Ising>", 1), (["--sweep-kernel", "1"], "k_sweep_fast<Ising>", 1),
    (["--workload", "config3", "--observables", "2"], "k_sweep_tree<AT>", 16),
    (["--workload", "config4"], "k_sweep_field_tree<AT>", 16),
    (["--workload", "config4", "--observables", "1"], "k_sweep_field<AT>", 1),
    (["--workload", "config4", "--observables", "2"], "k_sweep<AT>", 1)])
def test_the_line_names_the_kernel_that_runs(monkeypatch, args, kernel, lanes):
    monkeypatch.syspath_prepend(ROOT)
    import bench
    monkeypatch.setattr(sys, "argv", ["bench.py", *args])
    name, n = bench.sweep_kernel_of(bench.parse())
    assert name.startswith(kernel) and n == lanes
