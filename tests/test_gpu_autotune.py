"""The tile-shape autotuner of the residual kernels: every candidate (I, J, K) shape gives
the default shape's residual bit for bit (laminar Roe and k-omega, ragged blocks), the
autotuned cycles equal the default ones bit for bit, the tuner records a shape per block
size, and its choice is no slower than the default, also for blocks side by side on the pool."""
import numpy as np
import pytest

from finflo_amd.cases import make_block
from finflo_amd.layout import default_params

pytestmark = pytest.mark.gpu

NSHAPE = 8


@pytest.mark.parametrize("iturb", [0, 6], ids=["laminar", "sst"])
def test_every_shape_gives_the_same_residual(hip_device, iturb):
    from finflo_amd.ffhip import Context
    prm = default_params(iturb=iturb)
    for dims in ((37, 11, 9), (70, 20, 18)):
        print(f"case tile shapes iturb={iturb} dims={dims}", flush=True)
        blk = make_block(*dims, prm, distort=0.1, seed=5, amp=0.03, kind="all",
                         turb=(1.0, 80.0) if iturb else None)
        ref = None
        for sh in [-1] + list(range(NSHAPE)):
            b = blk.copy()
            ctx = Context(prm)
            ctx.tile_shape(sh)
            ctx.register(b)
            ctx.upload()
            ctx.statim()
            ctx.turbdi()
            r = ctx.residi()
            ctx.download()
            ctx.close()
            if ref is None:
                ref, rr = b.F.copy(), r
            else:
                np.testing.assert_array_equal(b.F, ref, err_msg=f"shape {sh}")
                np.testing.assert_array_equal(r, rr)


@pytest.mark.parametrize("iturb", [0, 6], ids=["laminar", "sst"])
def test_autotuned_cycles(hip_device, iturb):
    from finflo_amd.ffhip import Context
    print(f"case autotuned cycles iturb={iturb}", flush=True)
    prm = default_params(iturb=iturb)
    blk = make_block(96, 48, 32, prm, distort=0.05, seed=9, amp=0.02, kind="all",
                     turb=(1.0, 80.0) if iturb else None)
    a, b = blk.copy(), blk.copy()
    ca, cb = Context(prm), Context(prm)
    cb.autotune(True)
    for c, x in ((ca, a), (cb, b)):
        c.register(x)
        c.upload()
        c.cycle(ncycles=3)
        c.download()
    np.testing.assert_array_equal(a.F, b.F)
    tuned = cb.tuned_shape()
    print("tuned shape", tuned, flush=True)
    assert tuned is not None and tuned[1] > 0
    assert ca.tuned_shape() is None
    ca.close()
    cb.close()


@pytest.mark.parametrize("iturb", [0, 6], ids=["laminar", "sst"])
def test_tuned_is_not_slower(hip_device, iturb):
    """The tuner's time of its choice against the default shape's, on small blocks, where the
    default is far from every other candidate's time (48x24x24 laminar 23 us, the candidates 33
    and more); at two of three block sizes, for a launch that happens to be held up."""
    from finflo_amd.ffhip import Context
    prm = default_params(iturb=iturb)
    good = []
    for dims in ((48, 24, 24), (31, 15, 11), (64, 32, 24)):
        print(f"case tuned time iturb={iturb} dims={dims}", flush=True)
        blk = make_block(*dims, prm, seed=9, amp=0.02, kind="all", turb=(1.0, 80.0) if iturb else None)
        ctx = Context(prm)
        ctx.register(blk)
        ctx.upload()
        ctx.statim()
        ctx.turbdi()
        ctx.residi()
        ctx.profile(True)
        ctx.reset_stats()
        for _ in range(10):
            ctx.residi()
        ctx.finish()
        n, ms = ctx.kernel_stats("k_residual_kw" if iturb else "k_residual_tile")
        ctx.profile(False)
        ctx.autotune(True)
        ctx.residi()
        shape, tuned = ctx.tuned_shape()
        ctx.close()
        print("tuned", shape, tuned, "default", ms / n, flush=True)
        good.append(tuned < 1.2 * ms / n)
    assert sum(good) >= 2


def test_tuned_on_the_pool(hip_device):
    """Blocks side by side: a block is tuned while no other is at work, so the time of its choice
    is that of a block alone (a 48x24x24 block's residual takes 31 us, among the others' kernels
    more; at all of four blocks but one, for a launch that happens to be held up)."""
    from finflo_amd.ffhip import Context
    print("case tuned on the pool", flush=True)
    prm = default_params(iturb=6)
    kw = dict(distort=0.05, seed=9, amp=0.01, kind="all", turb=(1.0, 80.0))
    small = ((48, 24, 24), (31, 15, 11), (64, 32, 24), (40, 24, 16))
    dims = []
    for n, d in enumerate(small):
        dims += [(128, 96, 80 + 4 * n), d]
    ctx = Context(prm)
    ctx.block_streams(True)
    ctx.autotune(True)
    for n, d in enumerate(dims, start=1):
        ctx.register(make_block(*d, prm, **kw), block=n)
        ctx.upload(block=n)
    ctx.vcycle_blocks(list(range(1, len(dims) + 1)), 1, ncycles=1)
    tuned = {d: ctx.tuned_shape(block=n) for n, d in enumerate(dims, start=1)}
    ctx.close()
    good = []
    for d in small:
        one = Context(prm)
        one.register(make_block(*d, prm, **kw))
        one.upload()
        one.statim()
        one.turbdi()
        one.residi()
        one.profile(True)
        one.reset_stats()
        for _ in range(10):
            one.residi()
        one.finish()
        n, ms = one.kernel_stats("k_residual_kw")
        one.close()
        print(d, "tuned", tuned[d], "default alone", ms / n, flush=True)
        good.append(tuned[d][1] < 1.2 * ms / n)
    assert sum(good) >= len(good) - 1
