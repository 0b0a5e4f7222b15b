"""Quadratures of many samples start no more threads than the process may run on:
ranks that share a node are confined to their cores."""
import os
import subprocess
import sys

import pytest

CHILD = """
import os, threading
os.sched_setaffinity(0, {cores})
import numpy as np
from qsi_subspace_ed_amd import ftlm
a = np.random.default_rng(0).standard_normal((96, 300))
b = 0.5 + np.random.default_rng(1).random((96, 300))
ftlm.quadrature(a[:1], b[:1])
count = lambda: len(os.listdir("/proc/self/task"))
most, stop = [0], threading.Event()
def watch():
    while not stop.is_set():
        most[0] = max(most[0], count())
t = threading.Thread(target=watch)
t.start()
before = count()
ftlm.quadrature(a, b)
stop.set()
t.join()
print("more", most[0] - before)
"""


@pytest.mark.parametrize("cores", [1, 2])
def test_threads(cores):
    have = sorted(os.sched_getaffinity(0))
    if len(have) < 3:
        pytest.skip("needs three cores")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", CHILD.format(cores=set(have[:cores]))],
                         cwd=root, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr
    # this thread and cores - 1 more
    assert int(out.stdout.split()[-1]) <= cores - 1, out.stdout
