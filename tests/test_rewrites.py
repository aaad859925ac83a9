"""The plan of a fast FP32 streaming launch takes the limiter as one operation, divides by a
common divisor once, and picks a reciprocal instead of computing another."""
from paraiso_amd import variants
from paraiso_amd.generator.hip.ir import lower_kernel
from paraiso_amd.generator.hip.lane import MINMOD, plan_lane
from paraiso_amd.generator.plan import translate
from paraiso_amd.om.arith import Op


def test_plan():
    mk, setup, _ = variants.VARIANTS["rewrites_f32"]
    om = translate(setup, mk()).om
    k = lower_kernel(om, 0, (True, True), exact=True)
    p = plan_lane(k, sorted(set(v for _, v in k.stores)), fast=True)
    ops = [v.payload[0] for v in p.values if v.op == "arith"]
    assert ops.count(MINMOD) == 2 and ops.count(Op.Inv) == 2 and Op.Div not in ops
    assert Op.LE not in ops and Op.Abs not in ops        # the limiter's own are gone
    slow = plan_lane(k, sorted(set(v for _, v in k.stores)))
    assert MINMOD not in [v.payload[0] for v in slow.values if v.op == "arith"]
