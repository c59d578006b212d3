"""prof_summary's traffic of the degree-4 polynomial: its four launches are one entry with the bytes of all
four, COCG's z = M r or BiCGStab's on p and on s; launches past convergence do not count."""
import csv
import json

import pytest

PRE = "void dmri::(anonymous namespace)::"


def _csv(path, counter, launches):
    with open(path, "w", newline="") as fh:
        w = csv.DictWriter(fh, ["Dispatch_Id", "Kernel_Name", "Counter_Name", "Counter_Value"])
        w.writeheader()
        for i, (name, value) in enumerate(launches):
            w.writerow({"Dispatch_Id": i, "Kernel_Name": PRE + name + "(dmri::SolveArgs)", "Counter_Name": counter,
                        "Counter_Value": value})


@pytest.mark.parametrize("cocg", [True, False])
def test_four_steps_are_one_entry(tmp_path, cocg):
    import prof_summary as ps

    last = "poly_step_kernel<1, 1, double>" if cocg else "poly_step_kernel<1, 0, double>"
    step = "poly_step_kernel<1, 0, double>"
    one = [(step, 100.0), (step, 200.0), (step, 100.0), (last, 300.0)]
    none = [(step, 0.5)] * 3 + [(last, 0.5)]
    ops = ([("spmv_v_kernel<1, false, 4>", 400.0)] if cocg else
           [("spmv_v_kernel<1, false, 0>", 400.0), ("spmv_t_kernel<1, false, 2>", 410.0)])
    run = [("copy_kernel", 1.0), ("residual_kernel<1, false>", 5.0)] + 3 * ((one if cocg else one + one) + ops) + none
    for name, counter in (("f", "FETCH_SIZE"), ("w", "WRITE_SIZE")):
        _csv(tmp_path / name, counter, run)
    ps.traffic(tmp_path / "f", tmp_path / "w", 1024.0, tmp_path / "out", {}, 2)
    got = json.loads((tmp_path / "out").read_text())
    names = ("spmv_pre",) if cocg else ("spmv_v_pre", "spmv_t_pre")
    for key in ("traffic_per_launch_by_kernel", "traffic_per_launch_first_iteration_by_kernel"):
        for nm in names if key == "traffic_per_launch_by_kernel" or cocg else ():
            assert got[key][nm] == pytest.approx(2 * 700.0 * 1024)
    assert "poly_step" not in got["traffic_per_launch_by_kernel"]
    assert [got["launches_by_kernel"][nm] for nm in names] == [3] * len(names)
    assert got["traffic_per_launch_by_kernel"]["spmv_q" if cocg else "spmv_v"] == pytest.approx(2 * 400.0 * 1024)
    assert ps.iteration_kernel(PRE + "spmv_v_kernel<8, false, 12>(x)", 1) == "spmv_q"
