"""A run whose bin buffers have to grow: the same results, and stage times that are times."""
import numpy as np
import pytest

from conftest import compare_results, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("overlap", [0, 1])
@pytest.mark.parametrize("stencil", [False, True])
def test_stage_times_of_a_regrown_run(gv, orc, overlap, stencil):
    v, f = gv.icosphere(5, 0.4, (0.5, 0.5, 0.5), 0.02, seed=31)
    soup = gv.flatten(v, f)
    bmin, bmax, mms = gv.mesh_bbox(v)
    with gv.Context() as c:
        c.set_tune(l2_overlap=overlap)
        say(f"regrow, overlap {overlap}, stencil {stencil}")
        want = None
        for cap in (0, 100):
            g = c.voxelize(soup, bmin, bmax, mms, 96, 4, initial_capacity=cap, l1_stencil=stencil)
            i, got = g.info(), g.download()
            g.release()
            assert (i["regrows"] > 0) == (cap > 0)
            assert all(0.0 <= t <= i["ms_total"] for t in i["ms_stage"]), i["ms_stage"]
            if want is not None:
                compare_results("regrown", got, want, 4)
            want = got
        if not stencil:
            compare_results("regrown", want, orc.voxelize(soup, orc.grid_setup(bmin, bmax, mms, 96, 4), orc.ORC_FAST), 4)
