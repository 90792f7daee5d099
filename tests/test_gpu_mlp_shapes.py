"""The fused network kernels at the edges of their range: one layer and eight,
widths that leave waves without a column tile or with several, padded and full
input and output tiles, ragged row counts, a batch whose rows are not a
multiple of the depth steps loaded together, and a prediction longer than one
chunk, against the CPU oracle with the BF16 operand rounding mirrored."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# nin, width, depth, nout, rows of the gradient batch, rows of the prediction
SHAPES = [(1, 16, 1, 1, 16, 1), (5, 128, 3, 2, 1040, 17), (17, 144, 2, 3, 48, 33), (64, 512, 8, 16, 32, 16),
          (5, 32, 2, 2, 16, 16385)]


def _rounding_response(mo, lay, p, x, t, go):
    exact, noise = mo._mm, np.random.default_rng(0)

    def rounded(a, b, rnd):
        c = exact(a, b, rnd)
        return c * (1.0 + 2.0 ** -24 * np.sqrt(a.shape[1]) * noise.standard_normal(c.shape))

    mo._mm = rounded
    try:
        _, g = mo.loss_grad(lay, p.astype(float), x.astype(float), t.astype(float), rnd=True)
    finally:
        mo._mm = exact
    return np.linalg.norm(g - go)


@pytest.mark.parametrize("nin,width,depth,nout,rows,prows", SHAPES)
def test_network_shapes_match_oracle(gpu_solver, nin, width, depth, nout, rows, prows):
    from oracle import mlp_oracle as mo
    lib, check = gpu_solver.lib, gpu_solver._check
    fp = lambda a: a.ctypes.data_as(C.POINTER(C.c_float))      # noqa: E731
    lay = mo.Layout(nin, width, depth, nout)
    rng = np.random.default_rng(nin + width)
    p = lay.random_params(rng, 1.0 / np.sqrt(width)).astype(np.float32)
    x = rng.uniform(-1, 1, (rows, nin)).astype(np.float32)
    t = rng.standard_normal((rows, nout)).astype(np.float32)
    h = C.c_void_p()
    check(lib.stab_mlp_create(gpu_solver.ctx, nin, width, depth, nout, 1, C.byref(h)))
    try:
        assert lib.stab_mlp_nparams(h) == lay.nparams
        check(lib.stab_mlp_set_params(h, fp(p)))
        loss, g = np.zeros(1, np.float32), np.zeros(lay.nparams, np.float32)
        check(lib.stab_mlp_loss_grad(h, rows, fp(x), fp(t), fp(loss), fp(g)))
        lo, go = mo.loss_grad(lay, p.astype(float), x.astype(float), t.astype(float), rnd=True)
        # FP32 rounding of the sums moves some operands of the next layer to the other BF16 neighbour, and deep
        # networks carry that on: the bound is what the oracle itself moves by when its products carry errors
        # of the size of an FP32 sum of K terms
        assert abs(loss[0] - lo) <= 1e-4 * lo
        assert np.linalg.norm(g - go) <= 2.0 * _rounding_response(mo, lay, p, x, t, go) + 1e-6 * np.linalg.norm(go)
        for k, (off, o, i, ob) in enumerate(lay.layers()):       # padded weights get no gradient
            W = g[off:off + o * i].reshape(o, i)
            if k == 0:
                assert np.all(W[:, nin:] == 0)
            if k == depth:
                assert np.all(W[nout:] == 0) and np.all(g[ob + nout:ob + o] == 0)
        # one Adam step on the whole set, in order, from that gradient
        hist, p1 = np.zeros(1, np.float32), np.zeros(lay.nparams, np.float32)
        check(lib.stab_mlp_train(h, rows, fp(x), fp(t), rows, 1, 1e-3, 7, fp(hist)))
        check(lib.stab_mlp_get_params(h, fp(p1)))
        po, _, _ = mo.adam_step(p.astype(float), g.astype(float), 0.0, 0.0, 1, 1e-3)
        assert hist[0] == loss[0]
        assert np.max(np.abs(p1 - po)) <= 1e-6         # 1e-3 of the rate: FP32 rounding of the update
        # prediction with scaling, from the updated weights
        ish, isc = rng.uniform(-0.2, 0.2, nin).astype(np.float32), rng.uniform(0.5, 1.5, nin).astype(np.float32)
        osh, osc = rng.uniform(-1, 1, nout).astype(np.float32), rng.uniform(0.5, 20.0, nout).astype(np.float32)
        check(lib.stab_mlp_set_scaling(h, fp(ish), fp(isc), fp(osh), fp(osc)))
        xp = rng.uniform(-1, 1, (prows, nin)).astype(np.float32)
        y = np.full((prows + 1, nout), 77.0, np.float32)
        check(lib.stab_mlp_predict(h, prows, fp(xp), fp(y)))
        _, yo = mo.forward(lay, p1.astype(float), (xp.astype(float) - ish) * isc, rnd=True)
        # one flipped operand of K = width moves an output by 2^-8 |w| |a| <= 2^-8 / sqrt(width) times a few
        assert np.max(np.abs(y[:prows] * osc - (yo[:, :nout] + osh * osc))) <= 2e-2 / np.sqrt(width) + 1e-4
        assert np.all(y[prows] == 77.0)                # nothing past the last row
    finally:
        lib.stab_mlp_destroy(h)
