"""The timeline summary of a profiler database finds the transforms of the kernels that run now: from
the fold (or the clear) to the nodes, in either precision."""
import os
import sqlite3
import subprocess
import sys

TOOL = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "gpu-sfft_amd", "sfft_amd",
                    "rocpd_summary.py")


def _db(path, names):
    con = sqlite3.connect(path)
    con.execute("create table kernels (name text, start integer, end integer, grid_x integer, "
                "grid_y integer, workgroup_x integer, lds_size integer, vgpr_count integer)")
    for i, n in enumerate(names):
        con.execute("insert into kernels values (?, ?, ?, 64, 1, 64, 0, 8)",
                    (n, 10000 * i, 10000 * i + 6000))
    con.commit()
    con.close()


def test_timeline_finds_transforms(tmp_path):
    names = ["void sfft::fft_pass_kernel<double, 0, 0, 0>(sfft::PassArgs)",
             "void sfft::fold_slab_kernel<double, 24, 512>(sfft::SlabArgs)",
             "void sfft::sel_split_kernel<unsigned long long, sfft::SelOne>(sfft::SelOne)",
             "void sfft::nodes_kernel<double, 9, true, false>(sfft::NodeJob)",
             "sfft::hash_clear_kernel(unsigned int*)",
             "void sfft::sel_split_kernel<unsigned int, sfft::SelOne>(sfft::SelOne)",
             "sfft::hash_count_kernel(sfft::HashArgs)",
             "void sfft::nodes_kernel<float, 7, true, true>(sfft::NodeJob)"]
    path = str(tmp_path / "run.db")
    _db(path, names)
    out = subprocess.run([sys.executable, TOOL, "timeline", path], capture_output=True, text=True,
                         check=True).stdout.splitlines()
    rows = [ln.split() for ln in out if ln.startswith("fp") and ":" not in ln]
    assert rows == [["fp64", "26.0", "18.0", "8.0", "3"], ["fp32", "36.0", "24.0", "12.0", "4"]]
    assert sum("nodes_kernel" in ln for ln in out) == 2
