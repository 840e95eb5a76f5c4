"""The residual's built-in tiles: one K-plane per workgroup, or two on blocks of more than
3072 one-plane workgroups (32x8 tiles), against the oracle.  The slim blocks lie on either
side of that line (2 x KMAX workgroups), with ragged I and J and an odd KMAX; laminar Roe,
van Leer and FULLNS bit for bit, k-omega to the parity bar of 1e-12."""
import numpy as np
import pytest

from oracle.oracle_py import OracleBlock
from finflo_amd.cases import make_block
from finflo_amd.layout import default_params
from tests.parity import RES, SST_RES, assert_fields_equal

pytestmark = pytest.mark.gpu

FORMS = {"roe": {}, "vanleer": dict(iflux=0), "roe_ns": dict(fullns=1, rmult=500.0),
         "vanleer_ns": dict(fullns=1, iflux=0, rmult=500.0), "sst": dict(iturb=6),
         "sst_ns": dict(iturb=6, fullns=1)}


@pytest.mark.parametrize("kmax", [1536, 1537], ids=["one_plane", "two_planes"])
@pytest.mark.parametrize("form", FORMS)
def test_tile_planes(hip_device, form, kmax):
    from finflo_amd.ffhip import Context
    print(f"case residual tiles {form} kmax={kmax}", flush=True)
    prm = default_params(**FORMS[form])
    kw = prm.iturb == 6
    blk = make_block(5, 9, kmax, prm, lengths=(1.0, 1.0, 150.0), seed=3, amp=0.04, kind="all",
                     turb=(1.0, 80.0) if kw else None)
    a, g = blk.copy(), blk.copy()
    o = OracleBlock(prm, a)
    ctx = Context(prm)
    ctx.register(g)
    ctx.upload()
    o.state(); ctx.statim()
    o.turb(); ctx.turbdi()
    ro, rg = o.residual(), ctx.residi()
    ctx.download()
    ctx.close()
    assert_fields_equal(g, a, SST_RES if kw else RES, rtol=1e-12 if kw else 0.0, what=form)
    np.testing.assert_allclose(rg[:5], ro[:5], rtol=1e-10 if kw else 1e-13)
