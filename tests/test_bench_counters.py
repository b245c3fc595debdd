"""bench.py reports counters only of the walk kernel that it times."""
import json
import os
import shutil

import bench

CSRC = os.path.join(bench.ROOT, "pepc_amd", "csrc")


def _record(tmp_path, **kw):
    p = tmp_path / "counters.json"
    p.write_text(json.dumps({"hbm_bytes_per_launch": 1.5e9, "sq_insts_valu_per_launch": 4.0e9,
                             "workload": "w", **kw}))
    return str(p)


def test_only_the_same_sources_and_workload(tmp_path):
    sha = bench.walk_sources_sha16()
    assert bench.walk_counters(_record(tmp_path, walk_sources_sha16=sha), sha, "w") == (1.5e9, 4.0e9)
    assert bench.walk_counters(_record(tmp_path, walk_sources_sha16="0" * 16), sha, "w") == (None, None)
    right = _record(tmp_path, walk_sources_sha16=sha)
    assert bench.walk_counters(right, sha, "other") == (None, None)
    assert bench.walk_counters(_record(tmp_path), sha, "w") == (None, None)
    assert bench.walk_counters(str(tmp_path / "none.json"), sha, "w") == (None, None)
    (tmp_path / "bad.json").write_text("[1,")
    assert bench.walk_counters(str(tmp_path / "bad.json"), sha, "w") == (None, None)


def test_sources_hash(tmp_path):
    """Comments do not count, code does."""
    for name in ("walk.hip", "common.h", "kernels.h"):
        shutil.copy(os.path.join(CSRC, name), tmp_path / name)
    sha = bench.walk_sources_sha16(str(tmp_path))
    assert sha == bench.walk_sources_sha16()
    with open(tmp_path / "common.h", "a") as f:
        f.write("\n// a comment\n/* and\nanother */\n")
    assert bench.walk_sources_sha16(str(tmp_path)) == sha
    with open(tmp_path / "common.h", "a") as f:
        f.write("constexpr int kMore = 1;\n")
    assert bench.walk_sources_sha16(str(tmp_path)) != sha
