"""The counter summaries of walicxe3d_amd/profile_run.py: the memory
counters are scaled by the 1 GiB device copy that ends every profiled run.
The state upload is a copy dispatch of the same grid size, so the copy is
told apart by dispatch order (the last of the largest grid)."""
import csv
import os

from walicxe3d_amd import profile_run as PR


def _write(path, rows):
    cols = ["Dispatch_Id", "Grid_Size", "Kernel_Name", "Counter_Name", "Counter_Value"]
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, fieldnames=cols)
        w.writeheader()
        for r in rows:
            w.writerow(dict(zip(cols, r)))


def test_calibration_copy_is_the_last_large_copy(tmp_path):
    d = tmp_path / "run"
    d.mkdir()
    # upload of a 4.2 GiB state (dispatch 3), small copies, the stage
    # kernels, then the 1 GiB calibration copy (dispatch 22), same grid as
    # the upload
    _write(str(d / "run_counter_collection.csv"), [
        (1, 512, "__amd_rocclr_copyBuffer", "WRITE_SIZE", 0.78125),
        (3, 131072, "__amd_rocclr_copyBuffer", "WRITE_SIZE", 4409600.0),
        (4, 512, "__amd_rocclr_copyBuffer", "WRITE_SIZE", 0.0625),
        (9, 7000000, "void wx::k_stage<5, true, true, float, float, 4, -100>(wx::FusedArgs)", "WRITE_SIZE", 1.0e7),
        (22, 131072, "__amd_rocclr_copyBuffer", "WRITE_SIZE", 1048576.0),
    ])
    acc = PR._per_kernel(PR._read(str(d)), "WRITE_SIZE")
    assert PR._copy_reading(acc) == 1048576.0
    # the scale the summary applies: bytes per counter byte
    assert PR.COPY_BYTES / (1024.0 * PR._copy_reading(acc)) == 1.0


def test_second_stage_traffic_includes_the_end_of_the_step(tmp_path):
    """Where a kernel of its own ends the step, bench.py's second-stage time
    covers both, and so do the bytes per launch of the summary."""
    dirs = {}
    for name, copy, vals in (("FETCH_SIZE", 524288.0, (10.0, 20.0, 40.0)), ("WRITE_SIZE", 1048576.0, (1.0, 2.0, 4.0))):
        d = tmp_path / name
        d.mkdir()
        _write(str(d / "run_counter_collection.csv"), [
            (3, 256, "void wx::k_flow<5, false, float, float, 4, 1, false>(wx::FusedArgs)", name, vals[0]),
            (4, 256, "void wx::k_flow<5, true, float, float, 4, 1, false>(wx::FusedArgs)", name, vals[1]),
            (5, 256, "void wx::k_end<5, float, float, true, false, false>(wx::FusedArgs)", name, vals[2]),
            (9, 131072, "__amd_rocclr_copyBuffer", name, copy)])
        dirs[name] = str(d)
    out = str(tmp_path / "t.txt")
    assert PR.main(["summarize", "--fetch", dirs["FETCH_SIZE"], "--write", dirs["WRITE_SIZE"], "--workload", "sedov",
                    "--out", out]) == 0
    got = [line for line in open(out) if line.startswith("hbm_bytes_per_launch")]
    assert len(got) == 1 and got[0].split()[2] == "%.4e" % (1024.0 * (2 * 20 + 2 + 2 * 40 + 4))
