"""Device memory of plans, on the CPU (the engine's host code with a stand-in HIP
runtime that counts allocations against a limit): a plan that can be made in
less memory is made where its first choice does not fit.  Also which rows a plan
cuts in segments."""
from host_build import run_host

SOURCES = ["xc_engine.cpp", "xc_hostio.cpp"]


def test_lag_plans_hold_row_operands_in_bands(tmp_path):
    rc, out = run_host(tmp_path, "plan_memory.cpp", SOURCES + ["xc_tiled.cpp"], "lag")
    assert rc == 0, f"status {rc}: {out}"


def test_fft_plan_keeps_rows_whole_where_segments_do_not_fit(tmp_path):
    rc, out = run_host(tmp_path, "plan_memory.cpp", SOURCES + ["xc_tiled.cpp"], "fft")
    assert rc == 0, f"status {rc}: {out}"


def test_reversed_row_jobs_hold_one_period(tmp_path):
    rc, out = run_host(tmp_path, "reversed_job.cpp", SOURCES)
    assert rc == 0, f"status {rc}: {out}"


def test_small_jobs_keep_rows_whole_where_segments_are_slower(tmp_path):
    rc, out = run_host(tmp_path, "plan_memory.cpp", SOURCES + ["xc_tiled.cpp"], "rule")
    assert rc == 0, f"status {rc}: {out}"
