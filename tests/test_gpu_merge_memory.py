"""An upload when the device has room for the factor but not for its merged
rows (GPU): the factor runs on its plain levels or in chunks, and merges again
once there is room."""
import numpy as np
import pytest

import rchol_amd
from rchol_amd import factor as F
from rchol_amd.solver import OPT_CHUNKED, OPT_MERGE, merge_apply_host
from oracle import oracle as O

pytestmark = pytest.mark.gpu

ROOM = 128 << 20


@pytest.mark.parametrize("mode", [-1, 0])
def test_no_room_for_the_merged_rows(mode):
    import torch
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    A = F.grid_laplacian(28, 28, 28, np.ones(F.grid_edges(28, 28, 28)[0].size), 1e-2)
    n = A.shape[0]
    Gs, _, _ = F.factor(A, None, [n], "static", 1)
    r = np.random.default_rng(4).uniform(-1.0, 1.0, n)
    zo = O.precond(Gs, r)
    _, _, ents, _ = merge_apply_host(Gs, r)
    # 12 bytes an entry: more than the room, and the factor's own less
    assert 12 * sum(ents) > 1.5 * ROOM and 3 * 24 * int(Gs[0][-1]) < ROOM // 2
    print(f"case no room, chunk mode {mode}", flush=True)

    def applied(s):
        assert np.linalg.norm(s.precond(r) - zo) <= 1e-12 * np.linalg.norm(zo)
        st = s.stats()
        return st["chunked"], st["fwd_tasks"], st["bwd_tasks"]

    with rchol_amd.Solver(A) as s:
        s.set_option(OPT_CHUNKED, mode)
        s.set_option(OPT_MERGE, 0)
        s.upload_G(Gs)
        plain = applied(s)
        s.set_option(OPT_MERGE, 1)
        s.upload_G(Gs)
        merged = applied(s)
        assert merged != plain and merged[0] == 0
        s.set_option(OPT_MERGE, 0)
        s.upload_G(Gs)  # the merged rows are given back
        torch.cuda.empty_cache()
        held = []
        try:
            free = torch.cuda.mem_get_info()[0]
            while free > ROOM:
                held.append(torch.empty(min(free - ROOM // 2, 64 << 30), dtype=torch.uint8,
                                        device="cuda"))
                now = torch.cuda.mem_get_info()[0]
                if now >= free:
                    break
                free = now
            assert free <= ROOM
            s.set_option(OPT_MERGE, 1)
            s.upload_G(Gs)
            assert applied(s) == plain
            x, rr, it = s.pcg(A @ np.ones(n), 1e-10, 500)
            assert np.linalg.norm(x - 1.0) <= 1e-7 * np.sqrt(n)
        finally:
            held.clear()
            torch.cuda.empty_cache()
        s.upload_G(Gs)
        assert applied(s) == merged
