"""Failed launches in the serving loop, on the CPU (the engine's host code with a
stand-in HIP runtime): requests of a failed batch return the error, whichever
slot ran it and whether or not it had run a batch before.  Memory budgets of one
batch."""
from host_build import run_host


def test_failed_batches_return_the_error(tmp_path):
    rc, out = run_host(tmp_path, "serve_failure.cpp", ["xc_serve.cpp", "xc_engine.cpp", "xc_hostio.cpp"])
    assert rc == 0, f"status {rc}: {out}"


def test_budget_of_one_batch_makes_a_slot(tmp_path):
    rc, out = run_host(tmp_path, "serve_budget.cpp", ["xc_serve.cpp", "xc_engine.cpp", "xc_hostio.cpp"])
    assert rc == 0, f"status {rc}: {out}"


def test_server_without_room_for_warm_buffers(tmp_path):
    rc, out = run_host(tmp_path, "serve_host_memory.cpp", ["xc_serve.cpp", "xc_engine.cpp", "xc_hostio.cpp"])
    assert rc == 0, f"status {rc}: {out}"
