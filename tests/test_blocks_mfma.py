"""A store of vec@mat blocks alone (prefill_layout = 0) on the matrix-core
kernels that read the blocks: every forward against the oracle (indices
exact, outputs <= 1e-5 of the row's largest, the bar of the other expert
paths) and against the same call forced onto the fp32 kernels.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(om):
    c = om.Context()
    yield c
    c.close()


@pytest.fixture(scope="module")
def om():
    import ornith_moe
    return ornith_moe


def wide_scales(om, syn, seed):
    """Q6_K sub-scales over the int8 range, each block's first at an end."""
    rng = np.random.default_rng(seed)
    b = syn.down.reshape(-1, om.Q6K_BYTES)
    sc = rng.integers(-128, 128, (b.shape[0], 16))
    sc[:, 0] = np.where(rng.random(b.shape[0]) < 0.5, -128, 127)
    b[:, 192:208] = sc.astype(np.int8).view(np.uint8)


def forward(om, ctx, st, x, flags, mode=0, names=None, resid=True):
    T, D = x.shape
    xb, ob = ctx.upload(x), ctx.alloc(x.nbytes)
    ib, wb = ctx.alloc(T * st.k * 4), ctx.alloc(T * st.k * 4)
    if names is not None:
        om.lib().gpu_profile_enable(ctx.ptr, 1)
        om.lib().gpu_profile_reset(ctx.ptr)
    st.forward(0, xb, T, ob, resid=xb if resid else None, idx=ib, w=wb, flags=flags, mode=mode)
    if names is not None:
        names += [n for n, (_, calls) in om.profile(ctx).items() if calls]
        om.lib().gpu_profile_enable(ctx.ptr, 0)
    got = (ctx.download(ob, np.float32, x.shape), ctx.download(ib, np.uint32, (T, st.k)),
           ctx.download(wb, np.float32, (T, st.k)))
    for b in (xb, ob, ib, wb):
        b.free()
    return got


def row_err(a, ref):
    return (np.abs(a - ref).max(axis=1) / np.abs(ref).max(axis=1)).max()


# Shapes: one block column and several, slices from 4 steps to the longest
# taken (2048 / 32 = 64); token counts at one and two row tiles' edges, the
# step from 16- to 32-row items (64 / 65), experts over several items.
@pytest.mark.parametrize("D,H,E,k,wide,shared", [(256, 256, 4, 2, False, True),
                                                 (512, 1024, 6, 3, True, True),
                                                 (2048, 256, 3, 2, True, False),
                                                 (2048, 512, 16, 8, True, True)])
@pytest.mark.parametrize("T", [1, 15, 17, 64, 65, 131])
def test_blocks_mfma(om, ctx, D, H, E, k, wide, shared, T):
    syn = om.SyntheticLayer(7 * D + H, 0, D, H, E, shared)
    if wide:
        wide_scales(om, syn, H)
    st = om.Store(ctx, 1, D, H, E, k, shared, prefill_layout=False)
    st.load_layer(0, syn)
    x = om.synth_normal(T, om.synth_stream(0, om.SYN_ACT, 0), T * D, 1.0).reshape(T, D)
    x[T // 2] *= 1e4  # rows of very different size in one item
    names = []
    out, idx, w = forward(om, ctx, st, x, om.MOE_NORM if T % 2 else 0, names=names)
    assert {"moe_gateup_blk", "moe_down_blk"} <= set(names)
    valu, vidx, _ = forward(om, ctx, st, x, (om.MOE_NORM if T % 2 else 0) | om.MOE_PATH_VALU)
    kw = {"sh_" + n: syn.shared(n) for n in ("gate", "up", "down")} if shared else {}
    ref, ridx, rw = O.moe_layer(D=D, H=H, E=E, k=k, x=x, resid=x, router_W=syn.router,
                                norm_w=np.ones(D, np.float32) if T % 2 else None,
                                gate=syn.routed("gate"), up=syn.routed("up"),
                                down=syn.routed("down"), **kw)
    assert np.array_equal(idx, ridx) and np.array_equal(vidx, ridx)
    assert np.allclose(w, rw, rtol=1e-5)
    assert row_err(out, ref) <= 1e-5 and row_err(valu, ref) <= 1e-5
    st.close()


# Values that count 2^b below others whose weights are 0.
#   x    x[0] = 2^b, gate and up rows 0 empty
#   w    gate and up rows 0 with the largest d, x[0] = 0
#   mid  x[1] = 2^b goes to the first 256 hidden values alone (gate row 1 is 1
#        there and empty beyond), whose down rows are empty
#   sparse  x[0] = 2^b as above, and two small values the only others
# The bar is the other tests': fp32 arithmetic loses nothing here.
@pytest.mark.parametrize("what,b", [("w", 0)] + [(w, b) for w in ("x", "mid", "sparse")
                                                 for b in (0, 16, 20, 24, 30, 45, 60, 75)])
@pytest.mark.parametrize("D,H,T", [(256, 512, 20), (2048, 512, 70), (1024, 1024, 3)])
def test_blocks_mfma_wide_range(om, ctx, D, H, T, what, b):
    E, k = 4, 2
    syn = om.SyntheticLayer(D + H, 0, D, H, E, True)
    wide_scales(om, syn, D)
    x = om.synth_normal(T, om.synth_stream(0, om.SYN_ACT, 0), T * D, 1.0).reshape(T, D)
    if what == "sparse":
        x[:, :] = 0
        x[:, [D // 2, D - 1]] = 1.5, -0.7
    syn.router[:2] = 0
    gate, up = (a.reshape(E + 1, D, H // 256, om.Q4K_BYTES) for a in (syn.gate, syn.up))
    down = syn.down.reshape(E + 1, H, D // 256, om.Q6K_BYTES)
    if what == "mid":
        x[:, 0], x[:, 1] = 0, 2.0 ** b
        up[:, 1] = 0
        gate[:, 1] = 0
        gate[:, 1, 0, :2] = np.float16(1).reshape(1).view(np.uint8)
        gate[:, 1, 0, 4:8] = gate[:, 1, 0, 12:16] = 1  # scales 1, mins 0
        gate[:, 1, 0, 16:] = 0x11
        down[:, :256, :, 208:] = 0
    elif what == "w":
        x[:, 0] = 0
        gate[:, 0, :, :4] = up[:, 0, :, :4] = np.float16([65504, 65504]).view(np.uint8)
    else:
        x[:, 0] = 2.0 ** b
        gate[:, 0, :, :4] = up[:, 0, :, :4] = 0
    st = om.Store(ctx, 1, D, H, E, k, True, prefill_layout=False)
    st.load_layer(0, syn)
    names = []
    out, idx, _ = forward(om, ctx, st, x, 0, names=names, resid=False)
    assert {"moe_gateup_blk", "moe_down_blk"} <= set(names)
    valu, _, _ = forward(om, ctx, st, x, om.MOE_PATH_VALU, resid=False)
    ref, ridx, _ = O.moe_layer(D=D, H=H, E=E, k=k, x=x, router_W=syn.router,
                               gate=syn.routed("gate"), up=syn.routed("up"), down=syn.routed("down"),
                               **{"sh_" + n: syn.shared(n) for n in ("gate", "up", "down")})
    st.close()
    assert np.array_equal(idx, ridx)
    assert row_err(out, ref) <= 1e-5 and row_err(valu, ref) <= 1e-5


def test_blocks_mfma_row_isolation(om, ctx):
    """A NaN row poisons its own output and no other, and an expert's rows may
    come in any order."""
    D, H, E, k, T = 256, 256, 4, 2, 40
    syn = om.SyntheticLayer(3, 0, D, H, E, True)
    st = om.Store(ctx, 1, D, H, E, k, True, prefill_layout=False)
    st.load_layer(0, syn)
    x = om.synth_normal(5, om.synth_stream(0, om.SYN_ACT, 0), T * D, 1.0).reshape(T, D)
    out, idx, _ = forward(om, ctx, st, x, 0)
    y = x.copy()
    y[11, 3] = np.nan
    got, _, _ = forward(om, ctx, st, y, 0)
    keep = np.arange(T) != 11
    assert np.isnan(got[11]).all() and np.array_equal(got[keep], out[keep])
    perm = np.random.default_rng(1).permutation(T)
    assert np.array_equal(forward(om, ctx, st, x[perm], 0)[0], out[perm])
    st.close()


# Batches that fit gpu_moe_forward_noalloc's 32 MiB with the fp32 kernels'
# plan: the first two would not with slices for 4096 work groups (51 and 52
# MB), the last misses by its row maxima and stays with the fp32 kernels.
@pytest.mark.parametrize("D,H,E,k,shared,T,blk", [(2048, 512, 8, 8, False, 64, True),
                                                  (1024, 1024, 8, 8, False, 64, True),
                                                  (256, 256, 8, 8, True, 905, False)])
def test_blocks_mfma_fixed_scratch(om, ctx, D, H, E, k, shared, T, blk):
    st = om.Store(ctx, 1, D, H, E, k, shared, prefill_layout=False)
    st.fill_synthetic(0, 5)
    x = om.synth_normal(9, om.synth_stream(0, om.SYN_ACT, 0), T * D, 1.0).reshape(T, D)
    names = []
    ref = forward(om, ctx, st, x, 0, names=names)
    assert ("moe_gateup_blk" in names) == blk
    xb, ob = ctx.upload(x), ctx.alloc(x.nbytes)
    st.forward(0, xb, T, ob, resid=xb, noalloc=True)
    assert np.array_equal(ctx.download(ob, np.float32, x.shape), ref[0])
    st.close()
    for b in (xb, ob):
        b.free()
