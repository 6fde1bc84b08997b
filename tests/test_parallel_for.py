"""parallel_for of the host side: every index runs once on any number of
threads, the exception of the lowest throwing index comes back, and an
allocation that fails (of the thread list, of a thread) ends in an exception
or in fewer threads, never in the end of the process."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("probe") / "parallel_probe")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-o", exe,
                    os.path.join(HERE, "native", "parallel_probe.cpp")], check=True)

    def run(n, grain, bad=-1, fail=0):
        p = subprocess.run([exe, str(n), str(grain), str(bad), str(fail)], capture_output=True, text=True, timeout=60)
        assert p.returncode == 0, (p.returncode, p.stderr)
        *end, lo, hi = p.stdout.split()
        return " ".join(end), int(lo), int(hi)
    return run


@pytest.mark.parametrize("n,grain", [(0, 1), (1, 1), (2, 1), (15, 4), (16, 1), (17, 1), (1000, 16), (1000, 0)])
def test_every_index_once(probe, n, grain):
    assert probe(n, grain) == ("done", 1, 1)


@pytest.mark.parametrize("bad", [0, 1, 499, 999])
def test_the_lowest_exception_comes_back(probe, bad):
    assert probe(1000, 16, bad=bad)[0] == f"threw {bad}"


@pytest.mark.parametrize("fail", range(1, 24))
def test_failing_allocations(probe, fail):
    end, lo, hi = probe(1000, 16, fail=fail)
    assert (end, lo, hi) == ("done", 1, 1) or (end == "bad_alloc" and hi <= 1)
