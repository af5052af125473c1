"""Plans are built where the system grants fewer threads than asked for: a child process
whose threads take 8 GiB of address space each, with room for a few, builds each kind
of plan (dry run) and gets the plan that it gets with all its threads."""
import os
import resource
import subprocess
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import resource, sys
sys.path[:0] = ["tests", "tests/golden"]
from conftest import load_dkt
dkt = load_dkt()
dkt.load()
tree = dkt.balance_tree(dkt.sphere_tree(3, 30, 2, 6, (0.5, 0.5, 0.5), 0.3), 1)
das = [dkt.DA(tree, order) for order in (1, 2)]
limit = int(sys.argv[1])
if limit:
    now = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
    resource.setrlimit(resource.RLIMIT_AS, (now + limit, now + limit))
for da in das:
    for conforming in (False, True):
        print(da.order, conforming, sorted(dkt.Plan(da, conforming=conforming, dry_run=True).info().items()), flush=True)
"""


def _info(limit, stack):
    def child_limits():
        if stack:
            resource.setrlimit(resource.RLIMIT_STACK, (stack, resource.getrlimit(resource.RLIMIT_STACK)[1]))
    return subprocess.run([sys.executable, "-c", CHILD, str(limit)], cwd=REPO,
                          env=dict(os.environ, OMP_NUM_THREADS="1"), preexec_fn=child_limits, capture_output=True,
                          text=True, timeout=120)


def test_plans_with_few_threads():
    hard = resource.getrlimit(resource.RLIMIT_STACK)[1]
    if hard not in (resource.RLIM_INFINITY, -1) and hard < 8 << 30:
        pytest.skip("stack limit cannot be raised")
    want = _info(0, 0)
    assert want.returncode == 0 and len(want.stdout.splitlines()) == 4, want.stderr
    for room in (4 << 30, 20 << 30):  # none, two
        got = _info(room, 8 << 30)
        assert got.returncode == 0, (room, got.stdout, got.stderr[-300:])
        assert got.stdout == want.stdout
