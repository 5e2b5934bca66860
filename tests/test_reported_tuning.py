"""What a render reports of its tuning is what ran, without a GPU (tests/fake_hip.cpp lists the kernels)."""
import sys

import pytest

from test_memory_limits import Child, fake_hip, run_in_child  # noqa: F401  (fixture)

QUEUES = ("trace_block", "persistent_blocks", "sort_materials", "use_graph")


def whole_paths_report_no_queue_tuning(c):
    """A wavefront render small enough to run as whole paths launches no queue kernel and no graph; its path
    order has bands of 8 rows, its passes the samples asked for. With an option it runs as queues."""
    c.load(64, 48)
    for kw, form in ((dict(), "paths"), (dict(spp_per_pass=3), "paths"), (dict(sort_materials=1), "queues"), (dict(tile_rows=4), "queues")):
        c.forms()
        st = c.ctx.render(8, 3, 2, 1, integrator=1, **kw)[2]
        assert c.forms() == form, kw
        assert st["spp_per_pass"] == kw.get("spp_per_pass", 8) and st["tile_rows"] == kw.get("tile_rows", 8)
        if form == "paths":
            assert [st[k] for k in QUEUES] == [0, 0, 0, 0], kw
        else:
            assert [st[k] for k in QUEUES] == [256, 2048, 1, 1], kw
    assert [c.ctx.render(8, 3, 2, 1, integrator=0)[2][k] for k in QUEUES + ("tile_rows", "spp_per_pass")] == [0] * 6


SCENARIOS = [whole_paths_report_no_queue_tuning]


@pytest.mark.parametrize("scenario", [s.__name__ for s in SCENARIOS])
def test_reported_tuning(fake_hip, tmp_path, scenario):  # noqa: F811
    run_in_child(fake_hip, tmp_path, __file__, scenario)


if __name__ == "__main__":
    globals()[sys.argv[2]](Child(sys.argv[1]))
