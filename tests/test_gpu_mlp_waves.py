"""Networks whose layers take more than eight waves per 16-row tile: widths of
sixteen tiles, one more (a wave with two), and the widest ragged one, against
the oracle as in test_gpu_mlp_shapes; and the deepest, widest network at few
rows, where every weight goes through one CU: it must not take longer than the
181 us (prediction) and 308 us (step) that a launch per layer over all CUs took
on this card."""
import ctypes as C
import time

import numpy as np
import pytest

from test_gpu_mlp_shapes import test_network_shapes_match_oracle as _match_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nin,width,depth,nout,rows,prows", [(5, 256, 3, 2, 32, 17), (5, 272, 2, 2, 16, 15),
                                                             (33, 496, 3, 5, 48, 33)])
def test_wide_layers_match_oracle(gpu_solver, nin, width, depth, nout, rows, prows):
    _match_oracle(gpu_solver, nin, width, depth, nout, rows, prows)


def test_few_rows_of_the_largest_network(gpu_solver):
    lib, check = gpu_solver.lib, gpu_solver._check
    fp = lambda a: a.ctypes.data_as(C.POINTER(C.c_float))      # noqa: E731
    rng = np.random.default_rng(5)
    x, t = rng.uniform(-1, 1, (16, 64)).astype(np.float32), rng.standard_normal((16, 16)).astype(np.float32)
    y, hist = np.zeros((16, 16), np.float32), np.zeros(32, np.float32)
    h = C.c_void_p()
    check(lib.stab_mlp_create(gpu_solver.ctx, 64, 512, 8, 16, 1, C.byref(h)))
    try:
        us = {"predict": [], "step": []}
        for rep in range(25):
            t0 = time.perf_counter()
            check(lib.stab_mlp_predict(h, 16, fp(x), fp(y)))
            t1 = time.perf_counter()
            check(lib.stab_mlp_train(h, 16, fp(x), fp(t), 16, 32, 1e-4, 7, fp(hist)))
            t2 = time.perf_counter()
            if rep > 4:
                us["predict"].append(1e6 * (t1 - t0))
                us["step"].append(1e6 * (t2 - t1) / 32)
    finally:
        lib.stab_mlp_destroy(h)
    med = {k: float(np.median(v)) for k, v in us.items()}
    print(med)
    assert med["predict"] <= 181.0 and med["step"] <= 308.0
