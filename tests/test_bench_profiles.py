"""bench.py's profile summaries know the kernels that are there: every batched-build kernel has a stage, the timed render
instance is told from the others, and counters of another version of the render kernel are not reported.
"""
import json
import re
import sqlite3

import bench

CSRC = bench.ROOT / "ptgpu_pc_amd" / "csrc"


def test_batch_build_kernels_have_a_stage(tmp_path, monkeypatch):
    kernels = set(re.findall(r"\bvoid (kb_\w+)\(", (CSRC / "lbvh_batch.hip").read_text()))
    assert kernels == set(bench.BATCH_STAGE)
    db = tmp_path / "kt_results.db"
    con = sqlite3.connect(str(db))
    con.execute("create table top_kernels (name text, total_calls integer, average real)")
    con.executemany("insert into top_kernels values (?, ?, ?)",
                    [(f"void ptgpu::{k}<true>(ptgpu::BuildSeg const*, int const*, int)", 4, 50.0) for k in sorted(kernels)])
    con.commit()
    con.close()
    monkeypatch.setattr(bench, "batch_workload", lambda: [{"shapes": range(1000)}])
    out = tmp_path / "out.md"
    bench.batch_build_summary(db, ["python3 bench.py --batch"], out)
    text = out.read_text()
    assert "kb_mtree" in text and "| traversal_tree | 0.100 |" in text


def test_timed_render_instance():
    name = "void ptgpu::k_render_lanes<{}>(ptgpu::RenderParams)"
    for args, timed in (("36, false, true, false, true, false", True), ("32, false, true, false, true, true", True),
                        ("24, false, false, false, false, false", True), ("36, true, true, false, true, false", False),
                        ("48, false, true, true, true, false", False)):
        assert bool(bench.RENDER_INSTANCE_RE.search(name.format(args))) == timed
    # the template's parameters are as many as the expression expects
    decl = re.search(r"template <([^>]*)>\n__global__ [^\n]*void k_render_lanes\(", (CSRC / "render.hip").read_text())
    assert len(decl.group(1).split(",")) == 6


def test_counters_of_another_version(tmp_path, monkeypatch):
    f = tmp_path / "traffic.json"
    monkeypatch.setattr(bench, "TRAFFIC_FILE", f)
    row = {"kernel": bench.RENDER_KERNEL, "workload": bench.WORKLOAD, "version": bench.render_version(), "traffic_bytes": 5.0}
    f.write_text(json.dumps(row))
    assert bench.measured_traffic() == 5
    for other in ({**row, "version": "0" * 16}, {k: v for k, v in row.items() if k != "version"}):
        f.write_text(json.dumps(other))
        assert bench.measured_counters() is None
