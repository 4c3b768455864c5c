"""Dispatch of batches at the edges of its instances (8192 and 16,384 pairs)
against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O


@pytest.fixture(scope="module")
def om():
    import ornith_moe
    ornith_moe.lib()
    return ornith_moe


@pytest.fixture(scope="module")
def ctx(om):
    c = om.Context()
    yield c
    c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,k,shared", [(17, 16, 8, True), (1024, 256, 8, True),
                                          (1025, 256, 8, True), (2048, 16, 8, False),
                                          (2049, 16, 8, True), (8193, 4, 1, True)])
def test_dispatch_pairs(om, ctx, T, E, k, shared):
    """Expert indices the oracle's, outputs within 1e-5 of a row's largest
    value (as for the other layers; one expert per token: below): a pair on a wrong row, or a row with
    another token, is off by the row itself."""
    D = H = 256
    syn = om.SyntheticLayer(47, 0, D, H, E, shared)
    st = om.Store(ctx, 1, D, H, E, k, shared)
    x = om.synth_normal(47, om.synth_stream(0, om.SYN_ACT, 0), T * D, 1.0).reshape(T, D)
    xb, ob, ib = ctx.upload(x), ctx.alloc(x.nbytes), ctx.alloc(T * k * 4)
    try:
        st.load_layer(0, syn)
        st.forward(0, xb, T, ob, idx=ib)
        out, idx = ctx.download(ob, np.float32, x.shape), ctx.download(ib, np.uint32, (T, k))
    finally:
        st.close()
        for b in (xb, ob, ib):
            b.free()
    sh = {"sh_" + n: syn.shared(n) for n in ("gate", "up", "down")} if shared else {}
    ref, ridx, _ = O.moe_layer(D=D, H=H, E=E, k=k, x=x, router_W=syn.router,
                               gate=syn.routed("gate"), up=syn.routed("up"),
                               down=syn.routed("down"), **sh)
    assert np.array_equal(idx, ridx)
    # With one expert per token some rows rest on SiLU's tail alone (g down to
    # -35), where an error of g is a relative one of the result: 256 roundings
    # of partial sums of about 100 (sum |x w| is up to 388), 16 * 2^-24 * 100 =
    # 1e-4.  A pair on a wrong row is off by about 1.
    err = (np.abs(out - ref).max(axis=1) / np.abs(ref).max(axis=1)).max()
    assert err <= (1e-4 if k == 1 else 1e-5), err
