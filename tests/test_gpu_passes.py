"""The passes that take several of the reference's loops in one launch: RESIKE's gradients with
ZEROZZ and EXTEND, the SEPS maximum with CROSKO's rounding, and STATIM with the OLD copies,
on thin and odd blocks, every cell of the slab."""
import numpy as np
import pytest

from finflo_amd.cases import make_hierarchy
from finflo_amd.layout import OLD, default_params
from oracle.oracle_py import OracleBlock
from tests.parity import assert_fields_equal

pytestmark = pytest.mark.gpu

GRAD = ["OHMI", "W12", "W13", "W23", "S11", "S12", "S13", "S22", "S23", "S33"]
DIMS = [(2, 2, 2), (6, 2, 10), (258, 4, 2), (10, 6, 1)]


def level(dims, iturb, m):
    from finflo_amd.ffhip import Context
    prm = default_params(iturb=iturb, cfll=3.0)
    fine = dims if m == 1 else (2 * dims[0], 2 * dims[1], 2 * dims[2] if dims[2] > 1 else 1)
    blocks = make_hierarchy(*fine, m, prm, distort=0.1, kind="all", amp=0.03, seed=29,
                            turb=(1.0, 150.0) if iturb else None)
    b = blocks[m - 1]
    rng = np.random.default_rng(31)
    for name in GRAD + OLD + ["FUN1", "SRK"]:
        b[name] = rng.uniform(-1, 1, b.ntot)
    if iturb:
        b["EPS2"] = 1.0 + rng.uniform(5.0, 50.0, b.ntot)
    a = b.copy()
    ctx = Context(prm)
    ctx.register_levels(blocks)
    ctx.upload(level=m)
    return ctx, b, a, OracleBlock(prm, a, level=m)


@pytest.mark.parametrize("m", [1, 2])
@pytest.mark.parametrize("dims", DIMS)
def test_gradients_and_floor(hip_device, dims, m):
    """OHMI, W12.. and SIJ in the interior, the ghost layers EXTEND or DERFUN fills and the
    zeros elsewhere; FUN1 with the floor that the SEPS maximum sets (the maximum is exact; the
    tanh upstream of FUN1 rounds differently, hence 1e-12)."""
    print(f"case gradients dims {dims} level {m}", flush=True)
    ctx, b, a, oa = level(dims, 6, m)
    oa.state(); ctx.statim(level=m)
    oa.residual(m2=2); ctx.residi(level=m, m2=2); ctx.download(level=m)
    assert_fields_equal(b, a, GRAD, interior=False, what="gradients")
    assert_fields_equal(b, a, ["STRAIN"], what="strain rate")
    assert_fields_equal(b, a, ["RK", "REPS"], interior=False, what="rounding")
    assert_fields_equal(b, a, ["SEPS", "FUN1", "SRK"], rtol=1e-12, what="source terms")
    ctx.close()


@pytest.mark.parametrize("iturb", [0, 6], ids=["laminar", "sst"])
@pytest.mark.parametrize("dims", DIMS)
def test_copies_of_a_cycle(hip_device, dims, iturb):
    """A cycle's OLD copies are the variables before it, ghost layers included."""
    print(f"case copies dims {dims} iturb={iturb}", flush=True)
    ctx, b, a, oa = level(dims, iturb, 1)
    before = {o: np.array(a[o[:-3] if o[:-3] in ("U", "V", "W", "RK") else
                            {"TOLD": "TEMP", "POLD": "PDIFF", "EPSOLD": "REPS"}[o]]) for o in OLD}
    ctx.cycle(ncycles=1); ctx.download(level=1)
    for o in OLD:
        assert np.array_equal(b[o], before[o]), o
    ctx.close()
