"""The autotuner's table: a run without --all-knobs settles depth and log and
keeps the knobs that were timed with the launches of a default batch."""
import json

from c2a_amd import autotune as A


def test_rerun_keeps_the_default_launch_knobs():
    table = json.load(open(A.DEFAULT_TABLE))["buckets"]
    rows = [dict(r, spec_depth=4, replay_log=64, miss_depth=1, ext_levels=7) for r in table]
    rows.append({"max_ntri": 7, "spec_depth": 3, "replay_log": 2048, "miss_depth": 2,
                 "ext_levels": 0})   # a bucket the table does not have
    for r, old in zip(A.keep_knobs(rows, table), table + rows[-1:]):
        assert (r["miss_depth"], r["ext_levels"]) == (old["miss_depth"], old["ext_levels"])
    assert all(r["spec_depth"] == 4 for r in A.keep_knobs(rows, table)[:-1])
