"""Which size classes a launch of spring chains uses (csrc/de_spring_classes.h): the
set follows the lanes that the ensemble's sizes fill, not the number of systems.
Each ensemble below was timed on the device with every set; the rule must take the
fastest one or one within 10% of it."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def run(lines):
    cpp = os.path.join(HERE, "cpp")
    subprocess.check_call(["make", "-s", "-C", cpp, "_build/spring_classes"])
    out = subprocess.run([os.path.join(cpp, "_build", "spring_classes")], input="\n".join(lines),
                         capture_output=True, text=True, timeout=60, check=True)
    return [line.split() for line in out.stdout.splitlines()]


def line(dopri5, sizes):
    v, c = np.unique(np.asarray(sizes, dtype=np.int64), return_counts=True)
    return " ".join(["1" if dopri5 else "0"] + ["%d %d" % vc for vc in zip(v, c)])


def classes_of(dopri5, sizes):
    return run([line(dopri5, sizes)])[0][0]


def draw(kind, n):
    rng = np.random.default_rng(n)
    log = lambda k: np.clip(np.floor(np.exp(rng.uniform(np.log(4), np.log(257), k))), 4, 256)  # noqa: E731
    if kind == "log-uniform":
        return log(n)
    if kind == "small":  # 4 to 8 masses, 1% of them larger
        return np.concatenate([log(n // 100), rng.integers(4, 9, n - n // 100)])
    if kind == "four":
        return np.concatenate([[8, 16, 24, 32], np.full(n - 4, 4)])
    if kind == "three":  # 17 to 24 masses fill three per lane
        return np.concatenate([[4, 8, 16, 32, 64], rng.integers(17, 25, n - 5)])
    if kind == "large":
        return np.concatenate([[4, 8, 16, 32, 64], rng.integers(129, 257, n - 5)])
    return np.clip(rng.geometric(1.0 / 12.0, n), 1, 256)  # "geometric"


# Milliseconds with few / mid / all classes (few / all for the other methods).
TIMED = [
    (True, "log-uniform", 1024, 0.95, 1.28, 1.65), (True, "log-uniform", 2048, 1.01, 1.29, 1.69),
    (True, "log-uniform", 8192, 1.94, 1.78, 2.00), (True, "log-uniform", 16384, 3.48, 2.70, 2.58),
    (True, "log-uniform", 32768, 6.49, 4.78, 4.10), (True, "log-uniform", 65536, 12.54, 8.93, 7.24),
    (True, "small", 2048, 1.03, 1.06, 1.07), (True, "small", 8192, 1.82, 1.34, 1.56),
    (True, "small", 32768, 4.50, 2.16, 2.04), (True, "small", 65536, 8.09, 3.30, 2.77),
    (True, "four", 1024, 0.52, 0.65, 0.77), (True, "four", 6144, 1.08, 0.75, 0.77),
    (True, "four", 16384, 2.16, 1.07, 0.88), (True, "four", 32768, 3.87, 1.54, 0.98),
    (True, "three", 4096, 1.56, 0.69, 0.82), (True, "three", 16384, 4.47, 1.60, 1.14),
    (True, "three", 65536, 16.31, 4.67, 2.90),
    (True, "large", 2048, 1.15, 1.27, 1.28), (True, "large", 16384, 4.87, 5.05, 5.03),
    (True, "geometric", 2048, 0.74, 1.26, 1.44), (True, "geometric", 8192, 1.60, 1.30, 1.56),
    (True, "geometric", 32768, 5.01, 2.51, 2.00),
    (False, "log-uniform", 2048, 0.48, None, 0.57), (False, "log-uniform", 16384, 1.48, None, 1.20),
    (False, "geometric", 1024, 0.27, None, 0.43), (False, "geometric", 8192, 0.61, None, 0.50),
    (False, "geometric", 12288, 0.81, None, 0.55)]


def test_the_fastest_set_of_classes_is_used():
    got = run([line(d, draw(kind, n)) for d, kind, n, *_ in TIMED])
    for (dopri5, kind, n, *ms), (pick,) in zip(TIMED, got):
        t = dict(zip(("few", "mid", "all"), ms))
        assert t[pick] <= 1.10 * min(v for v in ms if v), (dopri5, kind, n, pick)


@pytest.mark.parametrize("sizes", [[4], [256], [4, 16, 60, 200], [1, 2, 3, 4], [17, 20, 24]])
def test_no_more_classes_than_queues_use_their_own(sizes):
    for n in (1, 100, 100000):
        assert [r[0] for r in run([line(d, np.repeat(sizes, n)) for d in (True, False)])] == \
            ["all", "all"]


def test_a_callers_group_size_is_taken():
    # Every chain of at least as many masses as lanes and at most four per lane gets the
    # lanes asked for; the others a shape that holds them.
    asked = [(n, g) for n in range(1, 257) for g in (1, 2, 4, 8, 16, 32, 64)]
    got = [tuple(map(int, r)) for r in run(["shape %d %d" % a for a in asked])]
    for (n, lanes), (g, c) in zip(asked, got):
        assert g * c >= n and c in (1, 2, 3, 4) and g <= 64
        if lanes <= n <= 4 * lanes:
            assert g == lanes, (n, lanes, g, c)
