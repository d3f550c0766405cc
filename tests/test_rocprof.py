"""Reduction of profiler output to per-stage figures (nsp.rocprof), on the CPU."""
import csv
import json

import pytest

from nsp import rocprof


def trace(path, steps, groups, correctors):
    """A kernel trace of `steps` ensemble steps: each evaluation is the radial
    derivative, the transforms of two classes and the four sweep passes in
    `groups` launches each (1 us per launch; the first step is a warm-up of 9 us
    launches)."""
    t = 0
    with open(path, "w", newline="") as f:
        w = csv.writer(f)
        w.writerow(["Start_Timestamp", "End_Timestamp", "Kernel_Name"])
        for s in range(steps + 1):
            for e in range(1 + correctors):
                names = ["void nsp::dr3_kernel<1>(nsp::Geom)"]
                names += [f"void nsp::{k}<float, {c}>()" for k in ("theta_inv_ct", "zpass5_ct", "theta_fwd_ct")
                          for c in range(2)]
                names += [f"void nsp::sweep_kernel<{p}, {int(e == 0)}, 1, 0, 0, 0, 0>()" for p in range(4)
                          for _ in range(groups)]
                for n in names:
                    d = 1000 if s else 9000
                    w.writerow([t, t + d, n])
                    t += d + 100


@pytest.mark.parametrize("groups,correctors", [(1, 1), (2, 1), (2, 3)])
def test_ensemble_stages_count_evaluations_not_launches(tmp_path, groups, correctors):
    trace(tmp_path / "t.csv", 3, groups, correctors)
    rocprof.main(["ensemble", "--trace", str(tmp_path / "t.csv"), "--steps", "3", "--form", "mixed", "--command", "x",
                  "--out", str(tmp_path / "o.json")])
    got = json.load(open(tmp_path / "o.json"))["mixed"]["stages"]
    ev = 1 + correctors
    want = {"dr3_kernel": (ev, ev), "theta_inv_kernel": (2 * ev, ev), "zpass_kernel": (2 * ev, ev),
            "theta_fwd_kernel": (2 * ev, ev), "linear_sweep_kernel(predictor)": (4 * groups, 1),
            "linear_sweep_kernel(corrector)": (4 * groups * correctors, correctors)}
    assert got == {k: dict(us_per_step=float(us), launches_per_step=float(n)) for k, (us, n) in want.items()}
