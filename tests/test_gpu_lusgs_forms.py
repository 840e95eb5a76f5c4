"""The staged LU-SGS sweeps on one block between the other forms: every form finds and leaves
the halo slots empty, and the staged corrector's runs of eight cells along I end right for
every remainder of IMAX (and for fewer than eight cells).  Bit for bit against the oracle."""
import pytest

from oracle.oracle_py import OracleBlock
from finflo_amd.cases import make_block
from finflo_amd.layout import default_params
from tests.parity import PRIM, RES, assert_fields_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("imax", [1, 7, 8, 9, 10, 19, 28])
def test_forms_share_the_halo_slots(hip_device, imax):
    from finflo_amd.ffhip import Context
    dims = (imax, 17, 10)
    print(f"case LU-SGS forms in turn dims={dims}", flush=True)
    prm = default_params(rmult=500.0)
    blk = make_block(*dims, prm, distort=0.1, seed=imax, amp=0.04, kind="all")
    a, g = blk.copy(), blk.copy()
    o = OracleBlock(prm, a)
    ctx = Context(prm)
    ctx.register(g)
    ctx.upload()
    for form in ("staged", "tiles", "staged", "staged1", "staged", "staged"):
        ctx.lusgs_mode(form)
        ctx.cycle()
        o.cycle()
        ctx.download()
        assert_fields_equal(g, a, PRIM, interior=False, what=form)
        assert_fields_equal(g, a, RES, what=form)
    ctx.close()
