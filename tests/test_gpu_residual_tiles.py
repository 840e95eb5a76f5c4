"""The residual's built-in tiles: one K-plane per workgroup, or two on blocks of more than
3072 one-plane workgroups (32x8 tiles), against the oracle.  The slim blocks lie on either
side of that line (2 x KMAX workgroups), with ragged I and J and an odd KMAX; laminar Roe,
van Leer and FULLNS bit for bit, k-omega to the parity bar of 1e-12.  The same for the tiles of
blocks with few J rows (64x2, 64x4, 32x4), on either side of the lines from 32x8 tiles to these and
between their plane counts, and a bound on the time of such a block."""
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
    check((5, 9, kmax), form)


# the last two: more than 8192 workgroups of 64x4 tiles, four planes without FULLNS too
THIN = [(3, 1, 256), (3, 1, 257), (3, 2, 6144), (3, 1, 6147), (35, 3, 128), (35, 3, 129), (33, 4, 3073),
        (33, 12, 1027), (33, 4, 3072), (33, 3, 8193)]


@pytest.mark.parametrize("dims,form", [(d, f) for d in THIN for f in FORMS if d[2] < 8000 or f in ("roe", "sst")])
def test_thin_tiles(hip_device, dims, form):
    check(dims, form)


@pytest.mark.parametrize("form", ["roe", "sst"])
def test_thin_time(hip_device, form):
    """A 1024x1x256 block's built-in tiles take no longer than 64x4x8 tiles (32x8 tiles take half
    as long again, 64x2 tiles 0.6 of the time; hence the margin)."""
    from finflo_amd.ffhip import Context
    print(f"case thin block's residual time {form}", flush=True)
    prm = default_params(**FORMS[form])
    blk = make_block(1024, 1, 256, prm, seed=3, amp=0.02, kind="all", turb=(1.0, 80.0) if form == "sst" else None)
    ctx = Context(prm)
    ctx.register(blk)
    ctx.upload()
    ctx.statim()
    ctx.turbdi()
    ms = {}
    for shape in (-1, 0):
        ctx.tile_shape(shape)
        ctx.residi()
        ctx.profile(True)
        ctx.reset_stats()
        for _ in range(5):
            ctx.residi()
        ctx.finish()
        n, t = ctx.kernel_stats("k_residual_kw" if form == "sst" else "k_residual_tile")
        ctx.profile(False)
        ms[shape] = t / n
    ctx.close()
    print(ms, flush=True)
    assert ms[-1] < 1.15 * ms[0]


def check(dims, form):
    from finflo_amd.ffhip import Context
    print(f"case residual tiles {form} {dims}", flush=True)
    prm = default_params(**FORMS[form])
    kw = prm.iturb == 6
    blk = make_block(*dims, prm, lengths=(1.0, 1.0, 150.0), seed=3, amp=0.04, kind="all",
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
