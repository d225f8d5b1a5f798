"""bench.py's reading of a profile (no GPU needed)."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import bench


def test_a_launch_is_placed_behind_the_copy_of_the_inputs():
    """A profiled step dispatches the copy of its inputs, then each timed launch's kernels as often as
    it ran (a product eleven times)."""
    rows = [("LayerNorm", 0.1, 0.0, 1.0, "k_ln_fused", 1), ("MatMul", 0.2, 1.0, 1.0, "k_gemm_w+k_splitk_sum", 11),
            ("Loss", 0.3, 0.0, 1.0, "k_ce_rows_p", 1), ("Nothing", 0.0, 0.0, 0.0, "", 1)]
    step = ["k_fetch_inputs", "k_ln_fused"] + ["k_gemm_w", "k_splitk_sum"] * 11 + ["k_ce_rows_p"]
    for launch, kernels in (("LayerNorm", ["k_ln_fused"]), ("MatMul", ["k_gemm_w", "k_splitk_sum"]),
                            ("Loss", ["k_ce_rows_p"])):
        at = bench.dispatch_places(rows, launch)
        assert at["step_dispatches"] == len(step)
        assert step[at["first"]:at["first"] + at["count"]] == kernels
