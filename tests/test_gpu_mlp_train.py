"""The training kernel of the learned proposal at the sizes where it can go
wrong: around a tile of 16 pairs, around one tile per workgroup (4096 pairs)
and past it, with parameters, pairs and workspace at addresses of 4 bytes'
alignment, a workspace full of NaN, and nothing written past its end.  Against float64 with
the parameters rounded to bf16: a gradient is a sum over the pairs of products
of sums of at most 128 terms, all rounded to float32 (6e-8); ten such
roundings of the largest value in a layer and the square root of the number of
additions in a row (at most 300 here) stay below 2e-5 of it."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tracker():
    from gpustreamlines_amd._device import DeviceTracker

    return DeviceTracker(dict(dimx=2, dimy=2, dimz=2, dimt=32, model_type=2, nverts=32, nedges=32, max_sline_len=501,
                              step_size=0.25, max_angle=1.0472, tc_threshold=0.1, relative_peak_thresh=0.25,
                              min_separation_angle=0.785, min_signal=1.0))


@pytest.mark.parametrize("n,shift", [(1, 0), (15, 1), (16, 0), (17, 3), (33, 0), (4095, 0), (4096, 2), (4097, 0),
                                     (9001, 1)])
def test_gradient_sizes(n, shift):
    from gpustreamlines_amd import learned as LP

    rng = np.random.default_rng(n)
    pairs = np.zeros((n, LP.PAIR), np.float32)
    pairs[:, :LP.N_IN] = rng.normal(size=(n, LP.N_IN))
    pairs[:, LP.N_IN:] = rng.uniform(0, 6, size=(n, LP.N_OUT))
    p = LP.init_params(4)
    p[LP.B1:LP.W2] = rng.normal(size=LP.W2 - LP.B1) * 0.1
    dt = _tracker()
    bufs = []

    def up(a):
        bufs.append(dt.alloc(a.nbytes))
        bufs[-1].upload(a)
        return bufs[-1]

    try:
        ws = dt.mlp_workspace_bytes(n)
        pd = up(np.concatenate([np.zeros(shift, np.float32), p]))
        xd = up(np.concatenate([np.zeros(shift, np.float32), pairs.ravel()]))
        wd = up(np.full(ws // 4 + 64, np.nan, np.float32))
        gd, ld = up(np.full(LP.NPARAM + 16, 7.0, np.float32)), up(np.full(4, 7.0, np.float32))
        out = []
        for _ in range(2):
            dt.mlp_loss_grad_async(pd.ptr + 4 * shift, xd.ptr + 4 * shift, n, ld.ptr, gd.ptr, wd.ptr + 4 * shift)
            dt.synchronize()
            out.append((ld.download(np.zeros(4, np.float32)), gd.download(np.zeros(LP.NPARAM + 16, np.float32))))
        tail = wd.download(np.zeros(ws // 4 + 64, np.float32))[ws // 4 + shift:]
    finally:
        for b in bufs:
            b.free()
        dt.close()
    assert np.isnan(tail).all()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    loss, g = out[0]
    assert (loss[1:] == 7.0).all() and (g[LP.NPARAM:] == 7.0).all()
    pr = LP.from_bf16(LP.to_bf16(p)).astype(np.float64)
    x, t = pairs[:, :LP.N_IN].astype(np.float64), pairs[:, LP.N_IN:].astype(np.float64)
    want = LP.grad_np(pr, x, t)
    assert abs(loss[0] - LP.loss_np(pr, x, t)) < 2e-5 * max(1.0, abs(float(loss[0])))
    for s, e in [(LP.W1, LP.B1), (LP.B1, LP.W2), (LP.W2, LP.B2), (LP.B2, LP.W3), (LP.W3, LP.B3), (LP.B3, LP.NPARAM)]:
        np.testing.assert_allclose(g[s:e], want[s:e], atol=2e-5 * np.abs(want[s:e]).max(), rtol=0)
