"""koral_hip_implicit_batch_noalloc takes no device memory: neither by an
allocation nor as the scratch memory that the runtime sets aside when a queue
first runs a kernel that spills.  A process of its own, whose queues have run
nothing that needs scratch before, watches the free memory around first calls
on the default and on new streams, for the sizes of both of its schedules."""
import ctypes
import os
import re
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r'''
import ctypes, sys
sys.path.insert(0, sys.argv[1])
import torch
from koral_amd import params as KP, problems as PR, cell
from koral_amd._lib import lib, check
f, v = lib().koral_hip_implicit_batch_noalloc, ctypes.c_void_p
f.argtypes = [v, ctypes.c_long, v, v, v, v, v, ctypes.c_double, v, v, v]
P = KP.params_implicit_batch()
P.mag, P.nv = int(sys.argv[2]), 10 + 3 * int(sys.argv[2])

def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]

for n in (1000, 40000):
    Q = KP.params_implicit_batch()
    pp, g20, G20, dt = PR.implicit_batch_states(Q, n, seed=1)
    if not P.mag:
        pp = pp[:, [0, 1, 2, 3, 4, 5, 9, 10, 11, 12]]
    p, g, G = (cell.to_dev(x) for x in (pp, g20, G20))
    d, u = torch.from_numpy(dt).cuda(), cell.p2u(P, p, g, G)
    fl, info = (torch.zeros((k, n), dtype=torch.int32, device="cuda") for k in (7, 6))
    for s in (torch.cuda.current_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(s):
            fl.zero_()  # the stream has its queue
        before = free()
        check(f(ctypes.byref(P), n, *(v(t.data_ptr()) for t in (u, p, g, G, d)), 0., v(fl.data_ptr()),
                v(info.data_ptr()), v(s.cuda_stream)), "noalloc")
        print("taken %d" % (before - free()), "solved %d" % int((info[1] >= 0).sum()), flush=True)
'''


@pytest.mark.parametrize("mag", [0, 1])
def test_first_calls_take_no_memory(mag):
    r = subprocess.run([sys.executable, "-c", CHILD, ROOT, str(mag)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    print(r.stdout, flush=True)
    taken = [int(x) for x in re.findall(r"taken (-?\d+)", r.stdout)]
    assert len(taken) == 4 and "solved 0" not in r.stdout
    # a queue's own bookkeeping is 2 MiB; twelve bytes of scratch a lane take 8
    assert max(taken) <= 4 << 20, taken


LAST_WAVE = 3 << 12  # IMP_WAVE_CELLS_NOSCRATCH


def test_calls_in_a_row_match_allocating_entry():
    """The sizes around the line between the two schedules, larger and smaller
    batches by turns on the shared lists: identical to koral_hip_implicit_batch."""
    import torch
    from koral_amd import params as KP, problems as PR, cell
    from koral_amd._lib import lib, check
    f, v = lib().koral_hip_implicit_batch_noalloc, ctypes.c_void_p
    f.argtypes = [v, ctypes.c_long, v, v, v, v, v, ctypes.c_double, v, v, v]
    P = KP.params_implicit_batch()
    runs = []
    for n in (40000, LAST_WAVE + 1, 1, 20011, LAST_WAVE, 65):
        pp, g20, G20, dt = PR.implicit_batch_states(P, n, seed=n)
        p, g, G = (cell.to_dev(x) for x in (pp, g20, G20))
        d = torch.from_numpy(dt).cuda()
        u = cell.p2u(P, p, g, G)
        q, w = p.clone(), u.clone()
        fl, info = (torch.zeros((k, n), dtype=torch.int32, device="cuda") for k in (7, 6))
        check(f(ctypes.byref(P), n, *(v(t.data_ptr()) for t in (w, q, g, G, d)), 0., v(fl.data_ptr()),
                v(info.data_ptr()), v(torch.cuda.current_stream().cuda_stream)), "noalloc")
        runs.append((n, (p, u, g, G, d), (q, w, fl, info)))
    for n, (p, u, g, G, d), got in runs:
        fl, info = cell.implicit(P, u, p, g, G, d)
        for a, b in zip(got, (p, u, fl, info)):
            assert np.array_equal(a.cpu().numpy(), b.cpu().numpy(), equal_nan=True), n
