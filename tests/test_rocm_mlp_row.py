"""forward() and evaluate() of three-layer networks over at most 2,048 rows (mlp_row_kernel: one, two, four or eight rows per workgroup) against 64-bit sums, through the
C ABI: the edges of each row count, inputs at the edges of a sixteen and of both instantiations, widths that fill no wavefront or no 64-position chunk.

fp32 tolerance: sums of at most 256 products and a fixed tree, three layers deep, stay within 3 * 256 * 2^-24 of the largest magnitude (4.6e-5) whatever the order;
1e-5 is what sums of random signs keep with room to spare."""
import numpy as np
import pytest

import helpers
from helpers import Mlp, rel_err

pytestmark = pytest.mark.gpu
ACT = {"relu": lambda v: np.maximum(v, 0), "tanh": np.tanh, "identity": lambda v: v, "sigmoid": lambda v: 1 / (1 + np.exp(-v))}

CASES = [
    # batch, in, hidden, out, hidden activation, output activation
    (1, 17, 256, 6, "relu", "tanh"),           # acting
    (1, 1, 68, 1, "relu", "identity"),         # the narrowest that comes here
    (256, 32, 256, 16, "tanh", "identity"),    # the last batch of one row per workgroup; the most outputs
    (257, 33, 256, 1, "relu", "identity"),     # two rows per workgroup, the last group ragged; inputs beyond two sixteens
    (512, 128, 200, 5, "sigmoid", "sigmoid"),  # the most inputs; a width that ends inside a wavefront's units
    (513, 16, 252, 3, "relu", "tanh"),         # four rows per workgroup
    (1025, 17, 256, 6, "tanh", "identity"),    # eight
    (1023, 17, 128, 6, "tanh", "tanh"),        # three rows in the last workgroup of four; wavefronts without units
    (1607, 5, 256, 16, "tanh", "sigmoid"),     # seven in the last of eight
    (2048, 3, 96, 2, "identity", "identity"),  # the largest
    (1024, 40, 200, 2, "relu", "identity"),    # the last batch of four rows for every network: from here on sixteen-row tiles ...
    (1025, 33, 256, 6, "relu", "tanh"),
    (2000, 17, 252, 6, "tanh", "identity"),
    (2047, 32, 256, 4, "relu", "identity"),    # ... but for eight rows of the widest with few inputs
    (1300, 40, 256, 2, "identity", "tanh"),    # ... and for networks that the tiles do not take
]


def dense(x, params, dims, ha, oa):
    kept = []
    for i in range(3):
        w, params = params[:dims[i] * dims[i + 1]].reshape(dims[i + 1], dims[i]), params[dims[i] * dims[i + 1]:]
        pre = x @ w.T + params[:dims[i + 1]]
        x, params = ACT[oa if i == 2 else ha](pre), params[dims[i + 1]:]
        kept.append((pre, x))
    return kept


@pytest.mark.parametrize("case", CASES)
def test_rows_against_64_bit_sums(rocm, case):
    print("case", case, flush=True)
    B, I, H, O, ha, oa = case
    dims = [I, H, H, O]
    rng = np.random.default_rng(B + I + H)
    params = helpers.random_params(rng, dims)
    x = rng.standard_normal((B, I + 3)).astype(np.float32)       # rows wider apart than the inputs
    net = Mlp(rocm, dims, params, B, ha, oa)
    xd, yd = rocm.array(x), rocm.array(np.full((B + 1, O + 2), 7, np.float32))
    ws, wsn = net.workspace()
    rocm.call("mlp_evaluate", net.layers, net.n, xd.ptr, I + 3, yd.ptr, O + 2, B, ws, wsn)
    rocm.call("mlp_forward", net.layers, net.n, xd.ptr, I + 3, B)
    rocm.sync()
    y = yd.numpy()
    assert np.all(y[B] == 7) and np.all(y[:, O:] == 7)
    for l, (pre, out) in enumerate(dense(x[:, :I].astype(np.float64), params.astype(np.float64), dims, ha, oa)):
        assert rel_err(net.pre[l].numpy().reshape(pre.shape), pre) <= 1e-5 and rel_err(net.out[l].numpy().reshape(out.shape), out) <= 1e-5, l
    assert np.array_equal(y[:B, :O], net.out[2].numpy().reshape(B, O))
