"""The device engine's host paths without a GPU: the library runs on a HIP
runtime whose memory is the host's and whose launches do nothing
(fakehip.c), in a process of its own. What is checked is what the host asked
for, not answers."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

PRELUDE = """
import ctypes, sys
hip = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
hip.fake_used.restype = ctypes.c_size_t
hip.fake_limit.argtypes = [ctypes.c_size_t]
hip.fake_clears.argtypes = [ctypes.c_size_t]
sys.path.insert(0, sys.argv[2])
import numpy as np
import fastcon as fc
def raises(f):
    try:
        f()
    except fc.FastconError as e:
        return e.status
    return 0
s = np.arange(40, dtype=np.int32)
t = s + 50
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fakehip") / "libfakehip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", so,
                    os.path.join(ROOT, "tests", "fakehip.c")], check=True)

    def go(body):
        p = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), so, os.path.join(ROOT, "fast-con_amd")],
                           capture_output=True, text=True, timeout=120)
        assert p.returncode == 0, p.stdout + p.stderr

    return go


def test_a_failed_clear_leaves_no_workspace_behind(run):
    """The teams' words must be zero before their first run: when their clear
    fails, the next call clears anew."""
    run("""
    hg = fc.gen_er(3000, 12.0, 1)
    g = fc.Graph(hg)
    for k in (1, 5, 8):  # one of the eight machines' clears
        held = hip.fake_used()
        done = hip.fake_clears(8 * hg.V)
        hip.fake_fail_clear(k)
        assert raises(lambda: g.stcon_many(s, t)) == fc.ERR_HIP
        assert hip.fake_used() == held
        g.stcon_many(s, t)
        assert hip.fake_clears(8 * hg.V) == done + (k - 1) + 8, k
        g.close()
        g = fc.Graph(hg)
    hip.fake_fail_clear(1)
    held = hip.fake_used()
    assert raises(lambda: g.stcon_batch(s, t)) == fc.ERR_HIP
    assert hip.fake_used() == held
    """)


def test_team_workspaces_make_room(run):
    """Allocations that fit without the teams' workspaces succeed beside them,
    on the same graph and on another, and the workspaces come back later."""
    run("""
    hg = fc.gen_er(100000, 12.0, 1)
    g = fc.Graph(hg)
    held = hip.fake_used()
    g.stcon_many(s, t)
    teams = hip.fake_used() - held
    assert teams >= 8 * 24 * hg.V
    other = fc.Graph(hg)  # its size, for the limit
    size = hip.fake_used() - held - teams
    other.close()
    assert size < teams
    hip.fake_limit(held + teams + size // 2)
    other = fc.Graph(hg)  # needs what the first graph's teams hold
    assert hip.fake_used() == held + size
    hip.fake_limit(held + size + 64 * teams)
    g.stcon_many(s, t)
    assert hip.fake_used() == held + size + teams
    other.close()
    hip.fake_limit(hip.fake_used() + 1000)
    status = raises(lambda: g.sched_trace(s, t))  # a wave machine of its own and its copy (launches do nothing here)
    assert status == fc.ERR_CAPACITY, status
    assert hip.fake_used() > held
    """)


def test_team_workspaces_leave_room(run):
    """At most a quarter of what is free."""
    run("""
    hg = fc.gen_er(3000, 12.0, 1)
    g = fc.Graph(hg)
    held = hip.fake_used()
    g.stcon_many(s, t)
    teams = hip.fake_used() - held
    g.close()
    hip.fake_limit(held + 4 * (teams - (1 << 17)) - 4096)  # (what a run uploads and reads back takes 2^17)
    g = fc.Graph(hg)
    status = raises(lambda: g.stcon_many(s, t))  # by launches, which do nothing here
    assert status == fc.ERR_CAPACITY, status
    assert hip.fake_used() == held, (hip.fake_used(), held, teams)
    """)
