"""CPU: what call patterns capture and launch (tests/runs_check.cpp over the library's own run
cutting).  A shot holds a bounded number of graphs and gives none back while it steps, and once a
pattern has come up a few times its steps are replayed in long runs: an advance is whole blocks,
and before and after them at most one run each, of its own or of five power-of-two parts."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rc") / "runs_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", os.path.join(ROOT, "tests", "runs_check.cpp"),
                    f"-I{os.path.join(ROOT, 'ela3d_amd', 'csrc')}", "-o", exe], check=True)
    return exe


def count(exe, every, n, calls=400):
    out = subprocess.run([exe, str(every), str(n), str(calls)], check=True, stdout=subprocess.PIPE, text=True).stdout
    f = out.split()
    return {k: int(v) for k, v in zip(f[::2], f[1::2])}


def blocks(every):
    """Steps of a block of whole energy cycles."""
    return 16 if every <= 0 else 16 // every * every


@pytest.mark.parametrize("every", [*range(0, 26), 33, 50, 64, 100, 250, 321])
def test_patterns(checker, every):
    # cadences and call lengths whose runs differ from call to call among them: 7, 9, 11, 13, 17
    # and 25 with 50 steps, 20 with 21
    for n in (1, 2, 5, 10, 16, 20, 21, 25, 50, 64, 300, 0):
        r = count(checker, every, n)
        assert r["wrong"] == 0 and r["held"] <= 32 + 28, (n, r)
        if n:
            assert r["covered"] == 200 * n
            full = n // 16 + n // every + 1 if every > 16 else n // blocks(every) + 1
            assert r["launches"] <= 200 * (full + 10), (n, r)


def test_server_rounds(checker):
    """Rounds of 50 steps without energy sums: three runs of 16 and one of 2."""
    assert count(checker, 0, 50)["launches"] == 4 * 200
    assert count(checker, 10, 100)["launches"] == 10 * 200
    assert count(checker, 1, 16)["launches"] == 200
    assert count(checker, 17, 50)["launches"] <= 200 * 5
