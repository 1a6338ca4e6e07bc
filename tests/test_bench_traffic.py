"""bench.py reports the headline's HBM traffic from a committed counter summary, which has to be of the launches that the plan issues."""
import bench
from smallframework_amd import capi, models


def test_the_committed_traffic_is_of_the_plan_that_runs():
    ops, launches = models.mobilenet_v1().ops, 0
    for i, op in enumerate(ops):
        if op.kind in ("conv", "dense") and op.C % capi.CB == 0:
            after = ops[i + 1] if i + 1 < len(ops) else None
            launches += not (after is not None and after.kind == "dw" and models.HipExecutor._pointwise_dw_pays(op, after))
    traffic = bench.measured_traffic_bytes("mobilenet_v1", 64, "conv_mfma_f32_*", launches)
    assert traffic is not None and 40e6 < traffic < 80e6, launches
