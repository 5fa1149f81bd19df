"""What the batched 2D form launches, in which order, when calls fail or settings
change: the library's own objects on a runtime without a device
(cpp/host_sequence.cpp), which prints launches and captures."""
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def run(cwa, tmp_path_factory):
    from coupledwateranimation_amd import build

    objs = [build.OUT / (Path(s).stem + ".o") for s in build.SOURCES]
    if not all(o.exists() for o in objs):
        build.build()
    exe = tmp_path_factory.mktemp("host") / "host_sequence"
    rocm = Path(build.hipcc()).resolve().parents[1]
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I",
                    str(rocm / "include"), str(HERE / "cpp" / "host_sequence.cpp"),
                    *map(str, objs), "-o", str(exe)], check=True)

    def f(*args):
        r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr
        calls, lines = [], []
        for line in r.stdout.splitlines():
            if line.startswith("returned"):
                calls.append((int(line.split()[1]), lines))
                lines = []
            else:
                lines.append(line)
        assert not lines
        return calls

    return f


def _launches(lines, kernel):
    return sum(x.startswith(f"launch {kernel} ") for x in lines)


def test_a_failed_step_leaves_no_keys_behind(run):
    """Whichever launch of a call of three steps fails, the next call clears the
    counts and run lists before it hashes; the one after that need not."""
    (rc, lines), _, _ = run("step_fails", 0)
    n = len(lines)
    assert rc == 0 and _launches(lines, "k2_wave") == 3 and _launches(lines, "k2_hash") == 1
    for nth in range(1, n + 1):
        (rc, lines), (rc1, after), (rc2, later) = run("step_fails", nth)
        assert rc < 0 and sum(x.startswith("failed ") for x in lines) == 1
        assert rc1 == 0 and rc2 == 0
        assert after[0].startswith("launch k_clear_cells "), (nth, after[:3])
        assert after[1].startswith("launch k2_hash ")
        assert _launches(after + later, "k_clear_cells") == 1


@pytest.mark.parametrize("nth", [1, 2, 3])
def test_a_failed_capture_runs_nothing(run, nth):
    """A call from graphs captures all that it needs before the first of them runs."""
    (rc, lines), (rc1, after) = run("graph_fails", nth)
    assert rc < 0 and lines[-1] == "failed instantiation"
    assert not any(x.startswith(("replay", "launch")) for x in lines)
    assert rc1 == 0 and _launches(after, "k2_wave") == 20 and _launches(after, "k2_hash") == 1


def test_settings_read_are_the_settings_that_run(run):
    """The wave pass's block as get_tuning reports it, before and after another
    setting is written back with it."""
    _, (_, first), _, (_, second) = run("tuning")
    name, threads = first[0].split()
    assert name == "wave_block"
    for lines in (first, second):
        assert [x.split()[2] for x in lines if x.startswith("launch k2_wave ")] == [threads]


def test_the_tuner_times_replays_alone(run):
    """No graph is captured between the events that time the chosen setting."""
    ((rc, lines),) = run("tune")
    assert rc == 0
    first, last = [k for k, x in enumerate(lines) if x == "event"][-2:]
    timed = lines[first + 1:last]
    assert _launches(timed, "k2_wave") == 3
    assert "replay" in timed and "capture" not in timed


@pytest.mark.parametrize("substeps", [1, 2, 4, 5, 8, 16, 32, 64])
def test_the_first_call_from_graphs_captures_little(run, substeps):
    """Graphs of several steps are for steps of few launches: a call captures no more
    than 200 launches a graph, or three steps (a first one, one of the middle
    and a last one)."""
    ((rc, lines),) = run("graph_first", substeps)
    launches = sum(x.startswith("launch ") for x in lines)
    captured = [int(x.split()[1]) for x in lines if x.startswith("captured ")]
    assert rc == 0 and _launches(lines, "k2_wave") == 6
    per_step = launches / 6
    assert max(captured) <= max(200, per_step + 1)
    assert sum(captured) <= max(launches, 3 * per_step + 1)
    if substeps >= 32:
        assert sum(captured) <= 3 * per_step + 1
