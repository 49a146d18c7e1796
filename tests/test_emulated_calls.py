"""What the kernels read and write, on the CPU: the sources built with the address sanitizer (``emulated.py``), every region
of the workspace with a guarded gap behind it, every result against the C checker."""

import pytest

from tests import emulated

pytestmark = pytest.mark.skipif(emulated.CXX is None, reason="no clang++")


@pytest.mark.parametrize("specs", [
    ["select:1500:3:uniform:::2", "select:1500:3:simplex:::3", "select:700:5:nan", "select:3001:3:grid:::2", "twopart:2500:5:shell"],
    ["select:4097:3:shell:::2", "select:9000:5:simplex:::2", "select:5000:2:layers", "rank:6001:5:uniform", "until:3000:5:inf"],
    ["select:33000:2:shell:::2", "select:33000:2:layers", "select:40001:3:simplex:::3"],
    ["batch:1100:3:shell:7", "batch:1500:5:simplex:5::2", "batch:300:3:uniform:9", "batch:5000:2:uniform:3"],
    ["batch:1100:2:shell:3::2", "batch:4000:2:layers:2", "batch:3001:2:equal:2", "batch:130:2:nan:5", "batch:2047:2:chain:2"],
    ["batch:300:3:uniform:2", "batch:500:3:grid:2", "batch:512:3:simplex:2", "batch:512:3:equal", "batch:257:3:nan:3", "batch:500:5:chain:2",
     "batch:400:5:inf:2", "batch:513:3:uniform", "batch:1000:5:grid", "batch:1024:3:shell", "batch:777:3:equal", "batch:900:5:nan"],
    ["select64:3000:3:uniform", "select64:9001:5:simplex", "crowd:1400:2:uniform", "crowd:5000:3:grid", "mask:20000:3:shell", "mask:70000:2:uniform"],
])
def test_every_access_lies_in_its_region(specs):
    out = emulated.run(specs)
    assert out.count("ok ") == len(specs)


def test_nothing_follows_an_order_whose_sort_ran_out_of_time():
    # (the ranks of more than 32 768 rows of two objectives are sorted by workgroups that wait for each other, on a control
    # block of the sort's own; the kernels behind it go by the call's: they took its order of -1 for rows)
    assert "ok " in emulated.run(["select:33000:2:uniform::::poisoned"], EMU_GIVE_UP="argsort_step_kernel")


@pytest.mark.parametrize("options,spec", [("mid_argsort=0", "select:17001:3:uniform::"), ("prefix_count_first=2 prefix_nearby=2", "select:33000:3:simplex::9000")])
def test_no_matrix_follows_orders_whose_sort_ran_out_of_time(options, spec):
    # (it is built from positions that nobody has written then)
    set_to = ["prefix_min_rows=16384", "order_stream=0"] + options.split()
    assert "ok " in emulated.run([a for o in set_to for a in ("-o", o)] + [spec + "::poisoned"], EMU_GIVE_UP="objective_order_kernel")


@pytest.mark.parametrize("options,spec,look", [
    ("", "select:33000:2:uniform", "argsort_step_kernel:1:2:1"),
    ("", "select:33000:2:uniform", "two_peel_kernel:1:4:1"),
    ("prefix_min_rows=16384 mid_argsort=0 order_stream=0", "select:17001:3:uniform", "objective_order_kernel:1:2:1"),
    ("peel_lds=0 peel_records=0", "select:1500:3:uniform", "peel_kernel:1:5:1"),
    ("peel_lds=0", "select:1500:3:uniform", "peel_records_kernel:1:5:1"),
    ("", "select:1500:3:uniform", "kernel:3:5:1"),  # peel_lds_kernel
    ("peel_lds=0", "select:1500:3:uniform", "crowd_runs_kernel:1:0:1"),
    ("", "select:1500:3:simplex", "crowd_gather_kernel:1:0:1"),
    ("", "select:1500:3:simplex", "crowd_gather_kernel:1:0:2"),  # crowd_sort_body, crowd_finish_body
    ("", "select:1500:3:simplex", "crowd_gather_kernel:1:0:3"),
])
def test_a_workgroup_leaves_as_a_whole(options, spec, look):
    # (another workgroup's wait runs out while this one starts: between the looks that two of its waves take at the error word)
    set_to = ["spin_limit=20000"] + options.split()
    out = emulated.run([a for o in set_to for a in ("-o", o)] + [spec + "::::poisoned"], EMU_ERROR_BEHIND=look)
    assert "ok " in out and "another workgroup gives up" in out


@pytest.mark.parametrize("spec,searched", [("crowd:1365:3:uniform", False), ("crowd:1366:3:uniform", True), ("crowd:1100:2:grid", False)])
def test_small_fronts_are_done_in_the_first_ordering_launch(spec, searched):
    # (1365 x 3 values fit the workgroups that order a small front whatever the mask selects: one launch, nothing behind it)
    out = emulated.run([spec], EMU_TRACE="1")
    assert ("crowd_terms_kernel" in out) == searched and "crowd_runs_kernel" in out and "ok " in out


def test_populations_of_a_launch_on_either_side_of_the_small_front():
    # (64 compute units for six populations: ten workgroups each order a last front of up to 320 rows together, larger ones go
    # through the sorted runs; uniform fitness stays below, rows around a sphere and on a plane lie above; every call meets
    # the word that the one before it has left)
    specs = ["batch:1300:5:uniform:6::2", "batch:1300:5:shell:6::2", "batch:1300:5:simplex:6::2", "batch:1300:5:uniform:6", "batch:1300:3:shell:6::2",
             "batch:1300:3:simplex:6::2", "batch:1300:3:uniform:6"]
    assert emulated.run(specs, EMU_CUS="64").count("ok ") == len(specs)


def test_populations_whose_peel_orders_their_last_fronts_take_one_launch_for_what_is_left():
    out = emulated.run(["batch:1300:5:uniform:3::2"], EMU_TRACE="1", EMU_CUS="256")
    first, second = out.split("rep 1")
    assert "crowd_terms_kernel" in first and "crowd_gather_kernel" not in first
    assert "crowd_terms_kernel" not in second and "crowd_gather_kernel" in second


def test_objective_orders_from_shares():
    # (smaller than the sizes at which they take this path by themselves; the shares of the last one do not fit)
    specs = ["-o", "prefix_min_rows=16384", "-o", "mid_argsort=0", "select:17001:3:grid", "select:17000:3:layers", "rank:17000:5:simplex",
             "-o", "order_stream_capacity=1000", "select:17003:5:shell"]
    out = emulated.run(specs, EMU_TRACE="1")
    assert out.count("ok ") == 4 and out.count("objective_shares_kernel") == 4


_COUNT_FIRST = ["-o", "prefix_count_first=2", "-o", "prefix_min_rows=16384"]


@pytest.mark.parametrize("m", [3, 5])
def test_totals_in_spatial_order(m):
    # (in the second call front 0 falls short: the matrix is built where the totals' scratch memory lay)
    specs = [f"select:{n}:{m}:{data}::{k}" for n, data, k in ((33000, "simplex", 9000), (33001, "shell", 6000), (33025, "equal", 100))]
    out = emulated.run(_COUNT_FIRST + ["-o", "prefix_nearby=2"] + specs, EMU_TRACE="1")
    assert out.count("ok ") == len(specs) and out.count("nearby_pairs_kernel") == len(specs)
    out = emulated.run(_COUNT_FIRST + ["-o", "prefix_nearby=0"] + specs[:1], EMU_TRACE="1")
    assert "ok " in out and "nearby" not in out


@pytest.mark.parametrize("n,spatial", [(57344, False), (65536, True)])
def test_totals_in_spatial_order_from_the_size_on_at_which_they_are_the_faster(n, spatial):
    out = emulated.run(["-o", "prefix_count_first=2", f"select:{n}:5:simplex::20000"], EMU_TRACE="1")
    assert "ok " in out and ("nearby_pairs_kernel" in out) == spatial
