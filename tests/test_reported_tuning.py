"""What a render reports of its tuning is what ran, without a GPU (tests/fake_hip.cpp lists the kernels)."""
import os
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


def passes(launched):
    """(grid, block) of each pass's first trace launch."""
    out = []
    for line in launched.decode().splitlines():
        name, *size = line.split(" ")
        if "k_wf_generate" in name:
            out.append(None)
        elif "k_wf_trace" in name and out[-1] is None:
            out[-1] = tuple(int(x) for x in size)
    return out


def the_autotuner_times_grids_that_differ(c):
    """A trace launch holds at most the workgroups resident at once (1536 of 256 threads), so grids above that
    are one candidate; the choice names the grid that ran. Every pass here takes longer than the one
    before it, so the first tuning stays."""
    c.load(64, 48)
    c.fake.fake_hip_launched()
    st = c.ctx.render(4, 3, 2, 1, integrator=1, autotune=1)[2]
    got = passes(c.fake.fake_hip_launched())
    # a warm-up and a timed pass each: the start, two block sizes, the two grids that differ from 1536, then at
    # the start's block and grid the sort, three band heights, the half pass (three passes) and the render
    assert got[:10] == [x for x in ((1536, 256), (2048, 64), (2048, 128), (512, 256), (1024, 256)) for _ in (0, 1)]
    assert got[10:] == [(1536, 256)] * (2 * (1 + 3) + 3 + 1)
    assert (st["trace_block"], st["persistent_blocks"]) == (256, 1536)
    with open(os.environ["LTS_TUNE_CACHE"]) as f:
        assert f.read().split()[1:3] == ["256", "1536"]


SCENARIOS = [the_autotuner_times_grids_that_differ, whole_paths_report_no_queue_tuning]


@pytest.mark.parametrize("scenario", [s.__name__ for s in SCENARIOS])
def test_reported_tuning(fake_hip, tmp_path, monkeypatch, scenario):  # noqa: F811
    monkeypatch.setenv("LTS_TUNE_CACHE", str(tmp_path / "tune"))
    run_in_child(fake_hip, tmp_path, __file__, scenario)


if __name__ == "__main__":
    globals()[sys.argv[2]](Child(sys.argv[1]))
