"""A captured step is replayed for the counts it was captured for: the ordered
FP64 sums have 16 or 32 targets a work-group by the count at the call's start, and
a graph of the other form is not kept.  The results are the same, so the kernels
that ran are read from torch's profiler, in a process of its own."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCRIPT = """
import torch
from torch.profiler import profile, ProfilerActivity
from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64
from vortex_amd.state import uniform_wake
pan = geo.circle(64, 0.5)
c = Case(make_params(pan, precision=VX_PREC_F64, dt=0.005, nu=1e-3, birth_offset_rel=0.5), pan)
c.build_matrix()
c.reserve(12000)
for n in (3800, 6000, 3800):
    c.set_state(*uniform_wake(n, seed=1, max_ve_g=1e-4))
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        c.run_steps_graph(3, (1.0, 0.0))
        torch.cuda.synchronize()
    names = [e.name for e in p.events() if "_ordered<" in e.name]
    print("RAN", n, len(names), sum("_ordered<16" in k for k in names), flush=True)
c.close()
"""


def test_captured_form_follows_the_count():
    r = subprocess.run([sys.executable, "-c", SCRIPT], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    ran = [tuple(map(int, q.split()[1:])) for q in r.stdout.splitlines() if q.startswith("RAN")]
    assert ran == [(3800, 6, 6), (6000, 6, 0), (3800, 6, 6)]
