"""Where an upload's host time is reported (GPU): the plans of a deep factor belong
to the schedule, not to the copies."""
import time

import numpy as np
import pytest

import rchol_amd
from rchol_amd import factor as F
from rchol_amd.solver import OPT_CHUNKED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["chunked", "merged"])
def test_plans_are_schedule_time(form):
    """Making the chunked plan of a 64^3 factor takes longer than copying the
    factor's rows, the merge plan of a 24^3 one longer than copying its rows."""
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    m, leaves = (64, 16) if form == "chunked" else (24, 1)
    A = F.laplace_3d(m)
    if leaves == 1:
        Gs, _, _ = F.factor(A, None, [A.shape[0]], "static", 1)
    else:
        perm, blocks = F.nd_grid(m, m, m, int(np.log2(leaves)) + 1)
        Gs, _, _ = F.factor(A, perm, blocks, "static", 1)
    print(f"case setup times {form}", flush=True)
    with rchol_amd.Solver() as s:
        if form == "chunked":
            s.set_option(OPT_CHUNKED, 1)
        s.upload_G(Gs)
        t = time.perf_counter()
        s.upload_G(Gs)
        wall = 1e3 * (time.perf_counter() - t)
        st = s.stats()
        assert st["chunked"] == (form == "chunked")
        analysis, schedule, copies = st["setup_ms"][1:]
        print(analysis, schedule, copies, wall)
        assert schedule > copies > 0 and analysis + schedule + copies <= wall
