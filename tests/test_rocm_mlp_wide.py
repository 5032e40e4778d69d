"""Parity of the forward + backward call on sixteen-row tiles (three-layer networks of hidden width up to 256 over at most 4,096 rows: mlp_wide_kernel, a workgroup of
sixteen wavefronts per tile, the weight gradients over the whole batch by a second launch) with the CPU checker and with the library's other paths for the same
call (RLT_MLP_WIDE=0), through the C ABI.

fp32 tolerance: 1e-5 relative to the largest magnitude of the tensor compared (the contraction order differs from the checker's)."""
import ctypes as C

import numpy as np
import pytest

import helpers
from helpers import Mlp, rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5


def run(backend, dims, params, x, dy, hidden_act, use_target, mse_scale, repeat=1, want_y=True):
    B = x.shape[0]
    net = Mlp(backend, dims, params, B, hidden_act, "identity")
    xd, yd, dyd = backend.array(x), backend.zeros((B, dims[-1])), backend.array(dy)
    ws, wsn = net.workspace()
    backend.call("mlp_zero_gradient", net.layers, net.n)
    for _ in range(repeat):
        if use_target:
            backend.call("mlp_forward_backward", net.layers, net.n, xd.ptr, dims[0], yd.ptr if want_y else None, dims[-1], None, 0, dyd.ptr, dims[-1], mse_scale, B, ws, wsn)
        else:
            backend.call("mlp_forward_backward", net.layers, net.n, xd.ptr, dims[0], yd.ptr if want_y else None, dims[-1], dyd.ptr, dims[-1], None, 0, 0.0, B, ws, wsn)
    backend.sync()
    return yd.numpy(), net.grads.numpy(), net.offsets


CASES = [
    # batch, in, hidden, out, hidden activation, target?
    (256, 17, 256, 6, "relu", False),        # the benchmark's network at its small batch
    (4096, 17, 256, 6, "relu", True),        # ... and at its middle one: 256 workgroups
    (37, 17, 256, 6, "tanh", False),         # a ragged last tile
    (1, 3, 64, 1, "relu", True),             # one row
    (300, 35, 256, 1, "relu", True),         # a critic of the Ant's width (27 + 8 inputs): the first layer in more than two chunks
    (100, 128, 200, 16, "fast_tanh", False), # the widest input and output, a hidden width that is no multiple of 16
    (2048, 1, 16, 2, "sigmoid", False),      # the narrowest
    (512, 64, 33, 6, "tanh", False),         # the most rows that one workgroup of the gradients' launch takes; two columns of the second tile of 32
    (513, 65, 256, 2, "tanh", True),         # ... and one more: two groups of workgroups share the batch; the first layer in five chunks
    (2051, 17, 250, 3, "tanh", False),       # eight groups
    (513, 128, 128, 3, "relu", False),       # few tiles: eight groups for two groups' rows
    # the workgroups' blocks added up: the narrowest with spare wavefronts, the widest, the last and the first batch of each line, without spare wavefronts
    (16, 3, 65, 1, "relu", True), (255, 1, 97, 16, "fast_tanh", False), (300, 60, 112, 2, "relu", False), (4096, 17, 100, 5, "tanh", True),
    (1024, 65, 80, 3, "tanh", False), (1025, 65, 80, 3, "tanh", False), (768, 20, 144, 4, "relu", True), (769, 20, 144, 4, "relu", True), (257, 1, 150, 1, "sigmoid", False),
    # tiles of four, eight and sixteen rows: one row of a tile, the last batch of each and the first of the next (widths without tiles of four: from one to sixteen whole units of 16)
    (5, 17, 256, 6, "relu", False), (1024, 17, 256, 6, "relu", True), (1025, 33, 256, 6, "relu", False), (2048, 17, 256, 1, "relu", False), (2049, 17, 256, 6, "relu", True),
    (1021, 100, 241, 16, "tanh", False), (9, 17, 128, 2, "relu", False), (2047, 128, 240, 6, "tanh", True), (257, 5, 200, 6, "relu", False), (1030, 17, 200, 6, "fast_tanh", False),
    (4096, 21, 112, 2, "relu", False), (4096, 22, 112, 2, "relu", True), (550, 20, 144, 4, "tanh", False), (551, 20, 144, 4, "tanh", True), (257, 60, 128, 3, "relu", True), (256, 60, 128, 3, "relu", True),
]


@pytest.mark.parametrize("case", CASES)
def test_sixteen_row_tiles_match_the_checker_and_the_other_paths(oracle, rocm, case, monkeypatch):
    print("case", case, flush=True)
    B, I, H, O, ha, use_target = case
    dims = [I, H, H, O]
    rng = np.random.default_rng(B * 31 + I + H)
    params = helpers.random_params(rng, dims)
    x = rng.standard_normal((B, I)).astype(np.float32)
    dy = rng.standard_normal((B, O)).astype(np.float32)
    ref = run(oracle, dims, params, x, dy, ha, use_target, 1.0 / B)
    got = run(rocm, dims, params, x, dy, ha, use_target, 1.0 / B)
    monkeypatch.setenv("RLT_MLP_WIDE", "0")
    other = run(rocm, dims, params, x, dy, ha, use_target, 1.0 / B)
    monkeypatch.delenv("RLT_MLP_WIDE")
    for name, want in (("checker", ref), ("other path", other)):
        assert rel_err(got[0], want[0]) <= TOL, (name, "y", rel_err(got[0], want[0]))
        for (off, nw, nb) in ref[2]:      # per-layer weight and bias gradients individually (a small layer must not hide behind a large one)
            ew = rel_err(got[1][off:off + nw], want[1][off:off + nw]); eb = rel_err(got[1][off + nw:off + nw + nb], want[1][off + nw:off + nw + nb])
            assert ew <= TOL and eb <= TOL, (name, off, ew, eb)
    assert np.abs(got[1]).max() > 0


def test_gradients_accumulate_and_the_output_may_be_null(oracle, rocm):
    """Two calls add up (the reduction adds onto the layers' gradients, as backward() does); y = NULL is allowed."""
    dims = [17, 256, 256, 6]
    rng = np.random.default_rng(3)
    params = helpers.random_params(rng, dims)
    x, dy = rng.standard_normal((500, 17)).astype(np.float32), rng.standard_normal((500, 6)).astype(np.float32)
    once = run(rocm, dims, params, x, dy, "relu", False, 0.0)
    twice = run(rocm, dims, params, x, dy, "relu", False, 0.0, repeat=2, want_y=False)
    assert rel_err(twice[1], 2.0 * once[1]) <= 1e-6 and not twice[0].any()
    ref = run(oracle, dims, params, x, dy, "relu", False, 0.0, repeat=2)
    assert rel_err(twice[1], ref[1]) <= TOL


@pytest.mark.parametrize("B,H", [(256, 256), (300, 200), (1025, 128), (4096, 250)])
def test_the_output_may_replace_the_input(rocm, B, H):
    """y in the memory of x, in layers as wide as the output and in rows farther apart: outputs and gradients are those of the call with memory of its own."""
    rng = np.random.default_rng(B)
    for I, O, ld in ((6, 6, 6), (17, 3, 20)):
        dims = [I, H, H, O]
        params = helpers.random_params(rng, dims)
        x, dy = rng.standard_normal((B, ld)).astype(np.float32), rng.standard_normal((B, O)).astype(np.float32)
        res = []
        for apart in (True, False):
            net = Mlp(rocm, dims, params, B, "relu", "identity")
            xd, yd, dyd = rocm.array(x), rocm.zeros((B, ld)), rocm.array(dy)
            ws, wsn = net.workspace()
            rocm.call("mlp_zero_gradient", net.layers, net.n)
            y = yd if apart else xd
            rocm.call("mlp_forward_backward", net.layers, net.n, xd.ptr, ld, y.ptr, ld, dyd.ptr, O, None, 0, 0.0, B, ws, wsn)
            rocm.sync()
            res.append((y.numpy()[:, :O], net.grads.numpy(), net.offsets))
        assert np.array_equal(res[0][0], res[1][0])
        for off, nw, nb in res[0][2]:
            for at, n in ((off, nw), (off + nw, nb)):
                assert rel_err(res[1][1][at:at + n], res[0][1][at:at + n]) <= TOL, (I, off, rel_err(res[1][1][at:at + n], res[0][1][at:at + n]))


@pytest.mark.parametrize("place", [(17, 0, 6), (6, 0, 20), (17, 17, 17), (17, 5, 17), (20, 3, 6)])
@pytest.mark.parametrize("B, H", [(5, 256), (9, 200), (16, 256), (16, 250)])
def test_the_output_may_replace_other_rows_of_the_input_where_one_workgroup_has_the_batch(oracle, rocm, B, H, place):
    """Up to sixteen rows: y packed over the rows of x, farther apart than they are, a row behind them, across the end of a row; y over the rows of the target; hidden outputs and y of a pass that is
    only forward. Outputs and gradients are those of the oracle's call with memory of its own. (tanh: a relu unit whose pre-activation rounding
    moves across 0, 5.8e-8 from it at (9, 200, second place), has another gradient.)"""
    ldx, shift, ldy = place
    dims, O, rng = [6 if ldx == 6 else 17, H, H, 6], 6, np.random.default_rng(B + H + ldy)
    params = helpers.random_params(rng, dims)
    memory = rng.standard_normal(B * 20 + 64).astype(np.float32)
    rows = lambda m, at, ld, n: np.stack([m[at + b * ld:at + b * ld + n] for b in range(B)])      # noqa: E731
    x, target = rows(memory, 0, ldx, dims[0]), rng.standard_normal((B, O)).astype(np.float32)
    want = run(oracle, dims, params, x, target, "tanh", True, 1.0 / B)
    over_target = memory.copy()
    for b in range(B):
        over_target[b * ldx:b * ldx + O] = target[b]
    for over in ("x", "target"):
        net = Mlp(rocm, dims, params, B, "tanh", "identity")
        ws, wsn = net.workspace()
        xd, td = (rocm.array(memory), rocm.array(target)) if over == "x" else (rocm.array(x), rocm.array(over_target))
        y = xd if over == "x" else td
        rocm.call("mlp_zero_gradient", net.layers, net.n)
        rocm.call("mlp_forward_backward", net.layers, net.n, xd.ptr, ldx if over == "x" else dims[0], y.offset(shift), ldy, None, 0, td.ptr, O if over == "x" else ldx, 1.0 / B, B, ws, wsn)
        rocm.sync()
        assert rel_err(rows(y.numpy(), shift, ldy, O), want[0]) <= TOL
        for off, nw, nb in want[2]:
            for at, n in ((off, nw), (off + nw, nb)):
                assert rel_err(net.grads.numpy()[at:at + n], want[1][at:at + n]) <= TOL, (over, at)
    if H % 4:      # (the other widths' passes of few rows are the one-row kernel's)
        net = Mlp(rocm, dims, params, B, "tanh", "identity")
        ws, wsn = net.workspace()
        xd = rocm.array(memory)
        rocm.call("mlp_evaluate", net.layers, net.n, xd.ptr, ldx, xd.offset(shift), ldy, B, ws, wsn)
        xh = rocm.array(np.concatenate([memory, np.zeros(B * H, np.float32)]))
        net.layers[0].output = xh.ptr
        rocm.call("mlp_forward", net.layers, net.n, xh.ptr, ldx, B)
        rocm.sync()
        assert rel_err(rows(xd.numpy(), shift, ldy, O), want[0]) <= TOL and rel_err(net.out[2].numpy(), want[0]) <= TOL


def test_the_call_takes_the_sixteen_row_tiles_where_this_file_says_so(rocm, monkeypatch):
    """Which path ran: the sixteen-row tiles and the path the call takes without them (RLT_MLP_WIDE=0) agree to tolerance but not bit for bit."""
    dims = [17, 256, 256, 6]
    rng = np.random.default_rng(4)
    params = helpers.random_params(rng, dims)
    x, dy = rng.standard_normal((256, 17)).astype(np.float32), rng.standard_normal((256, 6)).astype(np.float32)
    wide = run(rocm, dims, params, x, dy, "relu", False, 0.0)
    monkeypatch.setenv("RLT_MLP_WIDE", "0")
    other = run(rocm, dims, params, x, dy, "relu", False, 0.0)
    assert rel_err(wide[1], other[1]) <= TOL and not np.array_equal(wide[1], other[1])


def forward_then_backward(backend, dims, params, x, dy, ha, oa):
    """The reference's call pattern: forward() (keeps every layer's pre-activations and outputs), then backward() of a given gradient."""
    B = x.shape[0]
    net = Mlp(backend, dims, params, B, ha, oa)
    xd, dyd = backend.array(x), backend.array(dy)
    ws, wsn = net.workspace()
    backend.call("mlp_zero_gradient", net.layers, net.n)
    backend.call("mlp_forward", net.layers, net.n, xd.ptr, dims[0], B)
    backend.call("mlp_backward", net.layers, net.n, xd.ptr, dims[0], dyd.ptr, dims[-1], None, 0, B, 1, ws, wsn)
    backend.sync()
    return dict(grads=net.grads.numpy(), d_output=dyd.numpy(), offsets=net.offsets, pre=[p.numpy() for p in net.pre], out=[o.numpy() for o in net.out])


@pytest.mark.parametrize("case", [(256, 17, 256, 6, "relu", "identity"), (4096, 17, 256, 6, "relu", "tanh"), (37, 35, 200, 1, "tanh", "identity"), (100, 128, 72, 16, "fast_tanh", "sigmoid"),
                                  (1000, 3, 64, 2, "sigmoid", "identity"), (300, 128, 64, 3, "relu", "identity"), (4096, 2, 33, 1, "tanh", "identity"), (768, 20, 144, 4, "relu", "tanh"),
                                  (257, 128, 20, 16, "relu", "identity"), (1, 5, 16, 2, "tanh", "identity"), (2051, 17, 100, 2, "tanh", "identity"), (2052, 17, 100, 2, "tanh", "identity"),
                                  (128, 17, 100, 16, "relu", "tanh"), (129, 17, 100, 16, "relu", "tanh"), (600, 21, 112, 1, "relu", "identity"), (600, 22, 112, 1, "relu", "identity")])
def test_backward_alone_on_sixteen_row_tiles_matches_the_checker_and_the_other_paths(oracle, rocm, case, monkeypatch):
    """backward() after forward(): the tiles read the hidden layers' outputs back from memory; the last layer may have any activation (its derivative is applied to the
    given gradient before the kernel runs, in place as in the reference)."""
    print("case", case, flush=True)
    B, I, H, O, ha, oa = case
    dims = [I, H, H, O]
    rng = np.random.default_rng(B + 7 * I + H)
    params = helpers.random_params(rng, dims)
    x, dy = rng.standard_normal((B, I)).astype(np.float32), rng.standard_normal((B, O)).astype(np.float32)
    ref = forward_then_backward(oracle, dims, params, x, dy, ha, oa)
    got = forward_then_backward(rocm, dims, params, x, dy, ha, oa)
    monkeypatch.setenv("RLT_MLP_WIDE", "0")
    other = forward_then_backward(rocm, dims, params, x, dy, ha, oa)
    monkeypatch.delenv("RLT_MLP_WIDE")
    for name, want in (("checker", ref), ("other path", other)):
        assert rel_err(got["d_output"], want["d_output"]) <= TOL, name
        for l in range(3):      # what forward() keeps: every layer's pre-activations and outputs (hidden widths beyond 64 take the tiles in forward() as well)
            assert rel_err(got["pre"][l], want["pre"][l]) <= TOL and rel_err(got["out"][l], want["out"][l]) <= TOL, (name, l)
        for (off, nw, nb) in ref["offsets"]:
            ew = rel_err(got["grads"][off:off + nw], want["grads"][off:off + nw]); eb = rel_err(got["grads"][off + nw:off + nw + nb], want["grads"][off + nw:off + nw + nb])
            assert ew <= TOL and eb <= TOL, (name, off, ew, eb)
    assert not np.array_equal(got["grads"], other["grads"])      # two different kernels ran



# (hidden width 72: the workgroups' blocks of sixteen rows; 200: the batch shared out to wavefronts and groups of workgroups)
@pytest.mark.parametrize("H", [72, 200])
@pytest.mark.parametrize("B,row", [(300, 80), (300, 299), (1100, 150)])
def test_an_infinite_input_stays_in_its_column_and_infinite(rocm, B, row, H):
    """The wavefronts' shares of the batch do not end where their chunks of 32 rows do: a row behind a share's end is another share's, and its infinity meets no zero there.
    d_pre1 of a tanh network is not zero, so that column of the first layer's gradient is infinite and everything else finite."""
    dims = [17, H, H, 6]
    rng = np.random.default_rng(B + row)
    params = helpers.random_params(rng, dims)
    x, dy = rng.standard_normal((B, 17)).astype(np.float32), rng.standard_normal((B, 6)).astype(np.float32)
    net = Mlp(rocm, dims, params, B, "tanh", "identity")
    xd, dyd = rocm.array(x), rocm.array(dy)
    x[row, 3] = np.inf
    xi = rocm.array(x)
    ws, wsn = net.workspace()
    rocm.call("mlp_zero_gradient", net.layers, net.n)
    rocm.call("mlp_forward", net.layers, net.n, xd.ptr, 17, B)
    rocm.call("mlp_backward", net.layers, net.n, xi.ptr, 17, dyd.ptr, 6, None, 0, B, 1, ws, wsn)
    rocm.sync()
    grads = net.grads.numpy()
    off, nw, _ = net.offsets[0]
    infinite = np.zeros(grads.shape, bool)
    infinite[off:off + nw].reshape(H, 17)[:, 3] = True
    assert np.isinf(grads[infinite]).all() and np.isfinite(grads[~infinite]).all()


@pytest.mark.parametrize("H", [72, 200])
@pytest.mark.parametrize("B", [17, 300])
def test_an_infinite_weight_that_the_activation_saturates_leaves_finite_gradients(oracle, rocm, B, H):
    """The last tile's rows beyond the batch are zeros, which an infinite weight makes NaNs of; they are no part of the batch. One unit of the first hidden layer reads one
    positive input through an infinite weight: its tanh is one and its derivative zero in every row, and no gradient is infinite."""
    dims = [17, H, H, 6]
    rng = np.random.default_rng(B + H)
    params = helpers.random_params(rng, dims)
    params[:H * 17].reshape(H, 17)[5, 2] = np.inf
    x, dy = rng.standard_normal((B, 17)).astype(np.float32), rng.standard_normal((B, 6)).astype(np.float32)
    x[:, 2] = np.abs(x[:, 2]) + 0.1
    ref = run(oracle, dims, params, x, dy, "tanh", False, 0.0)
    got = run(rocm, dims, params, x, dy, "tanh", False, 0.0)
    assert np.isfinite(ref[1]).all() and np.isfinite(got[1]).all()
    assert rel_err(got[0], ref[0]) <= TOL and rel_err(got[1], ref[1]) <= TOL


@pytest.mark.parametrize("B, I", [(1, 1), (3, 16), (5, 33), (1024, 128), (1025, 64), (2047, 17), (2048, 33), (2049, 36), (4095, 3)])
def test_second_layers_of_256_units_wherever_they_lie(oracle, rocm, B, I):
    """256 units: a second layer on 16 bytes is read as it lies, one that is not from copies. Forward + backward in one call and as calls of their own, tiles of four, eight and sixteen rows, the first
    layer in one to eight chunks of sixteen columns."""
    dims = [I, 256, 256, 6]
    rng = np.random.default_rng(B + I)
    params = helpers.random_params(rng, dims)
    x, dy = rng.standard_normal((B, I)).astype(np.float32), rng.standard_normal((B, 6)).astype(np.float32)
    ref = run(oracle, dims, params, x, dy, "tanh", False, 0.0)
    for shift in (0, 1):
        net = Mlp(rocm, dims, params, B, "tanh", "identity")
        off, nw, _ = net.offsets[1]
        second = rocm.array(np.concatenate([np.zeros(shift, np.float32), params[off:off + nw]]))
        net.layers[1].weights = second.offset(shift)
        xd, yd, dyd = rocm.array(x), rocm.zeros((B, 6)), rocm.array(dy)
        ws, wsn = net.workspace()
        for separate in (False, True):
            rocm.call("mlp_zero_gradient", net.layers, net.n)
            if separate:
                rocm.call("mlp_forward", net.layers, net.n, xd.ptr, I, B)
                rocm.call("mlp_backward", net.layers, net.n, xd.ptr, I, dyd.ptr, 6, None, 0, B, 1, ws, wsn)
            else:
                rocm.call("mlp_forward_backward", net.layers, net.n, xd.ptr, I, yd.ptr, 6, dyd.ptr, 6, None, 0, 0.0, B, ws, wsn)
            rocm.sync()
            y, grads = (net.out[2] if separate else yd).numpy(), net.grads.numpy()
            assert rel_err(y, ref[0]) <= TOL, (shift, separate)
            for off, nw, nb in ref[2]:
                assert rel_err(grads[off:off + nw], ref[1][off:off + nw]) <= TOL and rel_err(grads[off + nw:off + nw + nb], ref[1][off + nw:off + nw + nb]) <= TOL, (shift, separate, off)


@pytest.mark.parametrize("dims, shift", [([17, 128, 128, 6], 0), ([17, 256, 256, 6], 1)])
def test_passes_that_need_copies_of_the_weights_are_recorded_after_one_that_needs_none(dims, shift):
    """A handle whose only pass so far, of 256 units on 16 bytes, read its layers as they lie: one of another width, or whose second layer lies elsewhere, is recorded all the same, and every replay
    leaves what the call by itself leaves, bit for bit."""
    be, graph, B = helpers.RocmBackend(), C.c_void_p(), 64
    rng = np.random.default_rng(dims[1])
    try:
        def network(dims, shift):
            params = helpers.random_params(rng, dims)
            net = Mlp(be, dims, params, B, "tanh", "identity")
            off, nw, _ = net.offsets[1]
            net.second = be.array(np.concatenate([np.zeros(shift, np.float32), params[off:off + nw]]))
            net.layers[1].weights = net.second.offset(shift)
            return net
        x, y, dy = be.array(rng.standard_normal((B, 17)).astype(np.float32)), be.zeros((B, 6)), be.array(rng.standard_normal((B, 6)).astype(np.float32))

        def step(net):
            ws, wsn = net.workspace()
            be.call("mlp_zero_gradient", net.layers, net.n)
            return be.device.lib.rlt_rocm_mlp_forward_backward(be.device.handle, net.layers, net.n, x.ptr, 17, y.ptr, 6, dy.ptr, 6, None, 0, 0.0, B, ws, wsn)
        assert step(network([17, 256, 256, 6], 0)) == 0
        net = network(dims, shift)
        be.sync()
        be.call("graph_begin_capture")
        try:
            rc = step(net)
        finally:
            be.call("graph_end_capture", C.byref(graph))
        assert rc == 0
        replays = []
        for _ in range(3):
            be.call("graph_launch", graph)
            be.sync()
            replays.append((y.numpy(), net.grads.numpy()))
        assert step(net) == 0
        be.sync()
        for got in replays:
            assert got[1].any() and np.array_equal(got[0], y.numpy()) and np.array_equal(got[1], net.grads.numpy())
        be.call("graph_destroy", graph)
    finally:
        be.close()
