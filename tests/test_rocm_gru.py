"""GRU forward and backward through time on the GPU, through the C ABI, against the CPU checker and against vectors written by the reference.

fp32 tolerance: 1e-5 relative to the largest magnitude of the tensor compared (contraction orders differ from the checker's)."""
import ctypes as C

import numpy as np
import pytest

import helpers
from helpers import rel_err
from test_oracle_golden import gru_golden_case

pytestmark = pytest.mark.gpu
TOL = 1e-5
KEYS = ("output", "post", "npp", "dx", "dy", "dW_i", "db_i", "dW_h", "db_h")


def run_pair(oracle, rocm, S, B, I, H, seed, with_reset, **kw):
    rng = np.random.default_rng(seed)
    params, x, dy, reset = helpers.gru_random_case(rng, S, B, I, H, with_reset)
    res = []
    for b in (oracle, rocm):
        g = helpers.GruOnBackend(b, S, B, I, H, params)
        g.forward(x, reset)
        g.backward(dy, **kw)
        b.sync()
        res.append(g.results())
    return res


@pytest.mark.parametrize("shape", [(7, 5, 6, 8), (1, 3, 4, 16), (24, 40, 11, 32), (12, 37, 20, 48), (9, 130, 3, 64), (5, 2, 7, 100)])
@pytest.mark.parametrize("with_reset", [False, True])
def test_gru_matches_checker(oracle, rocm, shape, with_reset):
    print("case", shape, with_reset, flush=True)
    S, B, I, H = shape
    want, got = run_pair(oracle, rocm, S, B, I, H, sum(shape), with_reset)
    for k in KEYS:
        assert rel_err(got[k], want[k]) <= TOL, (k, rel_err(got[k], want[k]))


def test_gru_backward_input_only_and_gradient_accumulation(oracle, rocm):
    S, B, I, H = 6, 9, 5, 32
    want, got = run_pair(oracle, rocm, S, B, I, H, 3, True, want_w=0)
    for k in ("dx", "dy"):
        assert rel_err(got[k], want[k]) <= TOL
    for k in ("dW_i", "db_i", "dW_h", "db_h"):
        assert not got[k].any()                                   # backward_input leaves the gradients alone
    rng = np.random.default_rng(5)
    params, x, dy, reset = helpers.gru_random_case(rng, S, B, I, H, False)
    g = helpers.GruOnBackend(rocm, S, B, I, H, params)
    g.forward(x); g.backward(dy, want_d_input=False); rocm.sync()
    once = g.results()
    g.backward(dy, want_d_input=False); rocm.sync()
    twice = g.results()
    for k in ("dW_i", "db_i", "dW_h"):
        assert rel_err(twice[k], 2 * once[k]) <= 1e-6           # gradients accumulate
    assert rel_err(twice["db_h"][2 * H:], 2 * once["db_h"][2 * H:]) <= 1e-6 and np.array_equal(twice["db_h"][:2 * H], twice["db_i"][:2 * H])
    assert not once["dx"].any()


@pytest.mark.parametrize("case", ["plain", "reset"])
def test_gru_against_reference_vectors(rocm, case):
    (S, B, I, H), params, x, dy, reset, want = gru_golden_case(case)
    g = helpers.GruOnBackend(rocm, S, B, I, H, params)
    g.forward(x, reset); g.backward(dy); rocm.sync()
    got = g.results()
    for k in KEYS:
        assert rel_err(got[k], want[k]) <= TOL, (k, rel_err(got[k], want[k]))


def test_gru_benchmark_shape(oracle, rocm):
    """I = 146, H = 64, S = 64 (the sequence-model benchmark): batch 64 against the checker; batch 1,024 through properties that do not need
    it -- batch rows are independent, so its first 64 rows reproduce the batch-64 run, and the gradients are linear in the upstream gradient."""
    S, I, H = 64, 146, 64
    want, got = run_pair(oracle, rocm, S, 64, I, H, 21, False)
    for k in KEYS:
        assert rel_err(got[k], want[k]) <= 2e-5, (k, rel_err(got[k], want[k]))
    rng = np.random.default_rng(21)
    params, x64, dy64, _ = helpers.gru_random_case(rng, S, 64, I, H, False)
    x = rng.standard_normal((S, 1024, I)).astype(np.float32); dy = rng.standard_normal((S, 1024, H)).astype(np.float32)
    x[:, :64], dy[:, :64] = x64, dy64
    g = helpers.GruOnBackend(rocm, S, 1024, I, H, params)
    g.forward(x); g.backward(dy); rocm.sync()
    big = g.results()
    for k in ("output", "post", "npp", "dx", "dy"):
        assert rel_err(big[k][:, :64], got[k]) <= 2e-6, k
    g2 = helpers.GruOnBackend(rocm, S, 1024, I, H, params)
    g2.forward(x); g2.backward(-2.0 * dy); rocm.sync()
    lin = g2.results()
    for k in ("dW_i", "db_i", "dW_h", "db_h", "dx"):
        assert rel_err(lin[k], -2.0 * big[k]) <= 2e-6, k


def test_gru_weight_gradients_over_a_long_batch(oracle, rocm):
    """16,384 (step, row) pairs and more take the weight-gradient kernel that keeps the whole 192 x 146 / 192 x 64 gradient in one workgroup's accumulators:
    batch 256 against the checker; batch 1,024 as the sum of its four quarters run separately (the gradients add over batch rows)."""
    S, I, H = 64, 146, 64
    print("batch 256 against the checker", flush=True)
    want, got = run_pair(oracle, rocm, S, 256, I, H, 33, True)
    for k in KEYS:
        assert rel_err(got[k], want[k]) <= 2e-5, (k, rel_err(got[k], want[k]))
    print("batch 1,024 against its quarters", flush=True)
    rng = np.random.default_rng(34)
    params, x, dy, reset = helpers.gru_random_case(rng, S, 1024, I, H, True)
    g = helpers.GruOnBackend(rocm, S, 1024, I, H, params)
    g.forward(x, reset); g.backward(dy); rocm.sync()
    whole = g.results()
    parts = []
    for q in range(4):
        sl = slice(256 * q, 256 * (q + 1))
        gq = helpers.GruOnBackend(rocm, S, 256, I, H, params)
        gq.forward(np.ascontiguousarray(x[:, sl]), None if reset is None else np.ascontiguousarray(reset[:, sl])); gq.backward(np.ascontiguousarray(dy[:, sl])); rocm.sync()
        parts.append(gq.results())
    for k in ("dW_i", "db_i", "dW_h", "db_h"):
        assert rel_err(whole[k], sum(p[k] for p in parts)) <= 1e-5, k
    for k in ("output", "dx"):
        assert rel_err(whole[k][:, 256:512], parts[1][k]) <= 2e-6, k


@pytest.mark.parametrize("hidden", [16, 32, 64])
@pytest.mark.parametrize("steps,batch", [(1, 9), (3, 2), (62, 5), (63, 3), (64, 6), (65, 1), (127, 7), (130, 5)])
def test_gru_at_the_edges_of_the_blocks_of_steps(oracle, rocm, steps, batch, hidden):
    """Reset flags are read for 63 or 64 steps at once, saved values requested up to four steps ahead: sequences that end around both. The tolerance is that of the long sequences."""
    print("case", steps, batch, hidden, flush=True)
    want, got = run_pair(oracle, rocm, steps, batch, 5, hidden, steps + hidden, True)
    for k in KEYS:
        assert rel_err(got[k], want[k]) <= 2e-5, (k, rel_err(got[k], want[k]))


@pytest.mark.parametrize("with_reset", [False, True])
@pytest.mark.parametrize("case", [(1, 3072, 3, 64), (1, 3073, 3, 64), (5, 3074, 4, 64), (24, 3121, 2, 64), (23, 3122, 2, 64), (74, 1025, 2, 64), (73, 1025, 2, 64)])
def test_gru_backward_on_both_sides_of_the_line_to_whole_rows(oracle, rocm, case, with_reset):
    """Width 64: the last batch with four steps' values requested ahead and the first with two (more than 3,072 rows), the last sequences that go through the kernel of sixteen units per
    wavefront and the first through that of a row per wavefront (more than 1,024 rows and 256 MB of saved values and gradients), last workgroups of one and two rows, one step. Tolerance as
    for the long batch above."""
    print("case", case, with_reset, flush=True)
    S, B, I, H = case
    want, got = run_pair(oracle, rocm, S, B, I, H, 36, with_reset)
    for k in KEYS:
        assert rel_err(got[k], want[k]) <= 2e-5, (k, rel_err(got[k], want[k]))


@pytest.mark.parametrize("case", [(32, 64, 34, 64), (33, 63, 160, 64), (16, 129, 66, 33), (64, 256, 64, 50), (64, 257, 146, 64), (64, 256, 36, 16),
                                  (32, 64, 96, 64), (33, 63, 98, 43), (16, 129, 128, 43), (32, 65, 130, 64), (64, 1024, 34, 44), (64, 64, 98, 44), (17, 241, 98, 43)])
def test_gru_at_the_edges_of_the_kernels_that_keep_a_layer_in_registers(oracle, rocm, case):
    """Input gates with their weights in registers (2,048 rows and more, 129 to 192 gates, even inputs from 34 to 160, padded to 64, 96, 128 or 160) and weight gradients in one workgroup's
    accumulators (16,384 rows and more, even widths from 66 to 160; from 34 on for 129 gates and 65,536 rows), the last batch whose columns are shared out (4,096 rows) and the first behind it: the smallest and largest inputs, ragged last rows, gates and widths that fill
    no tile. Tolerance as for the long batch above."""
    print("case", case, flush=True)
    S, B, I, H = case
    want, got = run_pair(oracle, rocm, S, B, I, H, 35, True)
    for k in KEYS:
        assert rel_err(got[k], want[k]) <= 2e-5, (k, rel_err(got[k], want[k]))


@pytest.mark.parametrize("fast_tanh", [False, True])
@pytest.mark.parametrize("case", [(1, 1, 64), (2, 3, 64), (3, 2, 64), (4, 5, 64), (5, 256, 64), (5, 257, 64), (4, 512, 64), (4, 513, 64), (20, 512, 64), (20, 513, 64), (19, 400, 64), (63, 2, 64),
                                  (64, 3, 64), (65, 1, 64), (66, 2, 64), (128, 1, 64), (129, 2, 64), (3, 1, 16), (4, 256, 16), (4, 257, 16), (8, 768, 16), (8, 769, 16), (2, 1280, 16),
                                  (2, 1281, 16), (65, 2, 16), (129, 1, 16), (3, 5, 32), (7, 300, 32), (8, 1280, 32), (8, 1281, 32), (64, 2, 32), (130, 1, 32)])
def test_gru_with_a_workgroup_per_row(oracle, rocm, case, fast_tanh):
    """Widths 64, 32 and 16 over at most 512, 1,280 and 1,280 rows (backward 512, 1,280 and 768, from four, eight or twenty steps on), with more inputs than the kernels beside the recurrence
    take: steps around the groups of four and the 64 whose reset flags are read at once, with resets and without, the last batches of a row per workgroup and the first of several. Tolerance as for the long batch above."""
    print("case", case, fast_tanh, flush=True)
    S, B, H = case
    for with_reset in (False, True):
        params, x, dy, reset = helpers.gru_random_case(np.random.default_rng(39 + S + B), S, B, 161, H, with_reset)
        results = []
        for b in (oracle, rocm):
            g = helpers.GruOnBackend(b, S, B, 161, H, params, fast_tanh=fast_tanh)
            g.forward(x, reset)
            g.backward(dy)
            b.sync()
            results.append(g.results())
        for k in KEYS:
            assert rel_err(results[1][k], results[0][k]) <= 2e-5, (k, rel_err(results[1][k], results[0][k]))


@pytest.mark.parametrize("want_d_input", [False, True])
@pytest.mark.parametrize("case", [(1, 1, 1), (2, 3, 15), (3, 5, 16), (4, 4, 17), (5, 2, 31), (22, 4, 146), (23, 4, 146), (40, 6, 146), (65, 7, 145), (130, 9, 158), (66, 6, 159), (71, 5, 160),
                                  (70, 3, 161), (24, 1021, 40), (24, 1024, 33), (24, 1025, 33), (24, 1022, 146), (25, 1023, 159), (25, 1023, 160), (26, 1024, 161), (25, 998, 130), (27, 1001, 100), (64, 40, 64), (64, 129, 64)])
def test_gru_with_input_gates_and_weight_gradients_beside_the_recurrence(oracle, rocm, case, want_d_input):
    """Width 64 over at most 1,024 rows: inputs around whole sixteens, the most that the accumulators and the registers of W_i hold (160) and one more, steps around the groups of
    four, last workgroups of one to four rows, workspaces that just hold the blocks of sums and that do not, both sides of the lines to the launches. Tolerance as for the long batch above."""
    print("case", case, want_d_input, flush=True)
    S, B, I = case
    want, got = run_pair(oracle, rocm, S, B, I, 64, 37, True, want_d_input=want_d_input)
    for k in KEYS:
        assert rel_err(got[k], want[k]) <= 2e-5, (k, rel_err(got[k], want[k]))


@pytest.mark.parametrize("case", [(1, 1, 1, 16), (1, 2, 33, 32), (3, 1, 32, 64), (1, 31, 5, 16), (3, 43, 65, 32), (5, 26, 31, 64), (9, 57, 64, 64), (4, 257, 1, 16), (2, 1100, 3, 32), (33, 128, 97, 16), (64, 71, 146, 64),
                                  (40, 1100, 66, 64), (31, 2114, 66, 64), (32, 2048, 66, 64), (32, 2048, 67, 64), (3, 5, 1024, 16), (3, 5, 1025, 16)])
def test_gru_weight_gradients_of_all_steps_in_one_launch(oracle, rocm, case):
    """Shares of the rows of less than eight steps of four rows, last steps of one to three rows, inputs around pairs of column tiles, more sequences than a workgroup has threads, both sides
    of the line to the kernel that keeps a whole gradient in one workgroup and of the most inputs. Tolerance as for the long batch above."""
    print("case", case, flush=True)
    S, B, I, H = case
    for want_d_input in (False, True):
        want, got = run_pair(oracle, rocm, S, B, I, H, 38, True, want_d_input=want_d_input)
        for k in KEYS:
            assert rel_err(got[k], want[k]) <= 2e-5, (k, rel_err(got[k], want[k]))


@pytest.mark.parametrize("case", [(64, 4, 3), (33, 70, 17), (40, 1000, 146), (30, 9, 64)])
def test_gru_states_may_replace_the_inputs(rocm, case):
    """A forward pass whose output buffer begins where its inputs do (rows narrower, wider and as wide as the states): the results of the call with memory of its own, whose input
    gates may be summed in another order."""
    S, B, I = case
    H, rng = 64, np.random.default_rng(S + I)
    params, x, _, reset = helpers.gru_random_case(rng, S, B, I, H, True)
    results = []
    for apart in (True, False):
        g = helpers.GruOnBackend(rocm, S, B, I, H, params)
        memory = rocm.array(np.concatenate([x.ravel(), np.zeros(S * B * max(H - I, 0), np.float32)]))
        flags = rocm.array(reset)
        if not apart:
            g.c.output = memory.ptr
        rocm.call("gru_forward", C.byref(g.c), memory.ptr, flags.ptr, S, B, g.ws, g.wsn)
        rocm.sync()
        results.append([g.out.numpy().ravel() if apart else memory.numpy()[:S * B * H], g.post.numpy(), g.npp.numpy()])
    for want, got in zip(*results):
        assert want.any() and rel_err(got, want) <= TOL


@pytest.mark.parametrize("case", [(32, 64, 44), (64, 64, 52), (33, 65, 48)])
def test_gru_gates_may_replace_as_many_inputs(rocm, case):
    """A forward pass whose inputs, 3 H to a row, lie where it leaves the gates: the results of the call with memory of its own, bit for bit (2,048 to 4,096 rows, the layer of whose input gates is shared out by
    columns where inputs and gates are apart)."""
    S, B, H = case
    params, x, _, reset = helpers.gru_random_case(np.random.default_rng(S + H), S, B, 3 * H, H, True)
    results = []
    for apart in (True, False):
        g = helpers.GruOnBackend(rocm, S, B, 3 * H, H, params)
        flags, xd = rocm.array(reset), rocm.array(x)
        if not apart:
            g.post.upload(x)
        rocm.call("gru_forward", C.byref(g.c), xd.ptr if apart else g.post.ptr, flags.ptr, S, B, g.ws, g.wsn)
        rocm.sync()
        results.append([g.out.numpy(), g.post.numpy(), g.npp.numpy()])
    for want, got in zip(*results):
        assert want.any() and np.array_equal(got, want)


def test_a_backward_pass_is_recorded_with_the_scratch_memory_of_a_shorter_one(rocm):
    """A handle whose scratch memory a call of a few steps has sized: a longer backward pass is recorded all the same (its shares of the rows want 1.3 MB, contractions less), and every replay
    leaves the gradients of the call on a handle that may allocate, to the file's tolerance."""
    S, B, I, H, rng = 16, 16, 146, 64, np.random.default_rng(3)
    params, x, dy, reset = helpers.gru_random_case(rng, S, B, I, H, True)
    want = helpers.GruOnBackend(rocm, S, B, I, H, params)
    want.forward(x, reset)
    want.backward(dy)
    rocm.sync()
    want, be, graph = want.results(), helpers.RocmBackend(), C.c_void_p()
    try:
        few = helpers.GruOnBackend(be, 2, 2, I, H, params)
        few.forward(x[:2, :2], reset[:2, :2])
        few.backward(dy[:2, :2])
        g = helpers.GruOnBackend(be, S, B, I, H, params)
        g.forward(x, reset)
        g.dy, g.dx = be.array(dy), be.zeros((S, B, I))
        be.sync()
        be.call("graph_begin_capture")
        try:
            rc = be.device.lib.rlt_rocm_gru_backward(be.device.handle, C.byref(g.c), g.x.ptr, g.dy.ptr, g.dx.ptr, g.reset.ptr, S, B, 1, g.ws, g.wsn)
        finally:
            be.call("graph_end_capture", C.byref(graph))
        assert rc == 0
        for _ in range(3):
            g.dy.upload(dy)
            be.call("fill_f32", g.grads.ptr, 1, g.grads.shape[0], g.grads.shape[0], 0.0)
            be.call("graph_launch", graph)
            be.sync()
            got = g.results()
            for k in KEYS:
                assert rel_err(got[k], want[k]) <= TOL, k
        be.call("graph_destroy", graph)
    finally:
        be.close()


@pytest.mark.parametrize("case", [(48, 256, 3), (64, 256, 16), (20, 512, 16), (33, 257, 32)])
def test_a_backward_pass_is_recorded_without_scratch_memory(rocm, case):
    """A handle on which nothing has run but forward passes: few enough rows for a workgroup each, whose weight gradients, as launches of their own, want scratch memory that a recording stream cannot ask for, and
    which the pass with the gradients beside the recurrence does without (steps * (54 + 92) <= 3,400 + (0.35 + 0.0037 inputs) * steps * sequences for these inputs: beyond that line, as with 128
    sequences of 64 steps of 3 inputs, a recording has always needed it). Every replay leaves the gradients of the call on a handle that may allocate, to the file's tolerance."""
    print("case", case, flush=True)
    (S, B, I), H, rng = case, 64, np.random.default_rng(4)
    params, x, dy, reset = helpers.gru_random_case(rng, S, B, I, H, True)
    want = helpers.GruOnBackend(rocm, S, B, I, H, params)
    want.forward(x, reset)
    want.backward(dy)
    rocm.sync()
    want, be, graph = want.results(), helpers.RocmBackend(), C.c_void_p()
    try:
        g = helpers.GruOnBackend(be, S, B, I, H, params)
        g.forward(x, reset)
        g.dy, g.dx = be.array(dy), be.zeros((S, B, I))
        be.sync()
        be.call("graph_begin_capture")
        try:
            rc = be.device.lib.rlt_rocm_gru_backward(be.device.handle, C.byref(g.c), g.x.ptr, g.dy.ptr, g.dx.ptr, g.reset.ptr, S, B, 1, g.ws, g.wsn)
        finally:
            be.call("graph_end_capture", C.byref(graph))
        assert rc == 0
        for _ in range(3):
            g.dy.upload(dy)
            be.call("fill_f32", g.grads.ptr, 1, g.grads.shape[0], g.grads.shape[0], 0.0)
            be.call("graph_launch", graph)
            be.sync()
            got = g.results()
            for k in KEYS:
                assert rel_err(got[k], want[k]) <= TOL, k
        be.call("graph_destroy", graph)
    finally:
        be.close()
