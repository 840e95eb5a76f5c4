"""DDADI sweeps on line lengths and line counts about the 8 steps and 32 lines of their
workgroups, bit for bit with the oracle, with operands whose quotients leave the range in which
the march divides by a reciprocal (zeros, huge and tiny increments)."""
import numpy as np
import pytest

from oracle.oracle_py import OracleBlock
from tests.parity import RES, SST_RES, assert_fields_equal, make_case

pytestmark = pytest.mark.gpu

DIMS = [(1, 2, 3), (7, 8, 9), (16, 1, 17), (33, 5, 8), (9, 40, 1), (8, 28, 24)]


@pytest.mark.parametrize("scale", ["ordinary", "zeros", "extreme"])
@pytest.mark.parametrize("iturb", [0, 6], ids=["laminar", "sst"])
@pytest.mark.parametrize("dims", DIMS)
def test_lines(hip_device, dims, iturb, scale):
    print(f"case DDADI lines {dims} iturb={iturb} {scale}", flush=True)
    from finflo_amd.ffhip import Context
    ckw = dict(kind="all", amp=0.02, seed=17)
    if iturb:
        ckw["turb"] = (1.0, 150.0)
    prm, blk = make_case(dims, dict(iturb=iturb, ddadi=1, cfl=3.0), ckw)
    a = blk.copy()
    oa = OracleBlock(prm, a)
    oa.save_old(); oa.state(); oa.turb(); oa.residual()
    names = SST_RES[:7] if iturb else RES
    rng = np.random.default_rng(3)
    for q, name in enumerate(names[:7 if iturb else 5]):
        if scale == "zeros" and q in (1, 3):
            a[name] = np.zeros(a.ntot)
        if scale == "extreme":
            x = a[name] * 10.0 ** rng.choice([-290, -150, 0, 0, 0, 150], a.ntot)
            a[name] = x
    g = a.copy()
    ctx = Context(prm)
    ctx.register(g)
    ctx.upload()
    with np.errstate(all="ignore"):
        oa.implicit()
    ctx.impsdi(); ctx.download()
    assert_fields_equal(g, a, ["DTL"] + names, interior=False, what="DDADI")
    ctx.close()
