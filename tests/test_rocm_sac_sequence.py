"""Sequential models with GRU layers and SAC's train_critic / train_actor on sequence batches, through the C ABI, against the CPU checker.

Tolerance: 1e-5 relative to the largest magnitude of the reference tensor (fp32); the device agent starts every loop step from the checker's
state (parameters, Adam moments and ages), so that differences do not accumulate through Adam's sign-like first steps."""
import ctypes as C

import numpy as np
import pytest

import helpers
from helpers import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-5


def copy_net(src, dst):
    for name in ("params", "grads", "m", "v", "age"):
        a = getattr(src, name)
        if a is not None:
            getattr(dst, name).upload(a.numpy())


def copy_agent(src, dst):
    copy_net(src.actor, dst.actor)
    for k in range(2):
        copy_net(src.critics[k], dst.critics[k]); copy_net(src.targets[k], dst.targets[k])
    dst.log_alpha.upload(src.log_alpha.numpy()); dst.alpha_age.upload(src.alpha_age.numpy())


def compare_agents(got, want, where, tol=TOL):
    for name, a, b in [("actor", got.actor, want.actor)] + [(f"critic{k}", got.critics[k], want.critics[k]) for k in range(2)]:
        assert rel_err(a.grads.numpy(), b.grads.numpy()) <= tol, (where, name, "gradients", rel_err(a.grads.numpy(), b.grads.numpy()))
        assert rel_err(a.params.numpy(), b.params.numpy()) <= tol, (where, name, "parameters", rel_err(a.params.numpy(), b.params.numpy()))
    for k in range(2):
        assert rel_err(got.targets[k].params.numpy(), want.targets[k].params.numpy()) <= tol, (where, "target", k)
    assert rel_err(got.log_alpha.numpy(), want.log_alpha.numpy()) <= tol, (where, "log_alpha", got.log_alpha.numpy(), want.log_alpha.numpy())
    for key in ("target", "next_lp", "next_q0", "next_q1", "d_ci0", "d_ci1", "d_ao", "a_lp"):
        # the log-probabilities hold log(1 - a^2 + 1e-6): for an action within 1e-3 of +-1 one ulp of tanh moves that term by 1e-4 (the
        # reference's own formula, equally sensitive on the CPU); what is formed from them (targets, log_alpha) is held to the tolerance
        t = 10 * tol if key.endswith("_lp") else tol
        assert rel_err(got.buf[key].numpy(), want.buf[key].numpy()) <= t, (where, key, rel_err(got.buf[key].numpy(), want.buf[key].numpy()))
    assert got.ages() == want.ages()


# (steps, batch, in, hidden, out, GRU layers, fast_tanh, resets)
MODEL_CASES = [(6, 16, 4, 16, 1, 1, True, True), (7, 5, 3, 8, 2, 2, False, True), (5, 33, 17, 64, 6, 1, True, True), (9, 64, 11, 64, 3, 2, True, False),
               (1, 7, 4, 16, 1, 1, True, False), (12, 130, 6, 32, 2, 1, False, True)]


@pytest.mark.parametrize("case", MODEL_CASES)
def test_sequential_model_forward_and_backward_match_checker(oracle, rocm, case):
    print("case", case, flush=True)
    S, B, I, H, O, n_gru, fast, with_reset = case
    rng = np.random.default_rng(S * 100 + B)
    specs = [(0, I, H, "relu")] + [(1, H, H, "identity")] * n_gru + [(0, H, H, "tanh"), (0, H, O, "identity")]
    model_against_checker(oracle, rocm, rng, specs, helpers.random_seq_params(rng, specs), S, B, fast, with_reset)


def model_against_checker(oracle, rocm, rng, specs, params, S, B, fast, with_reset):
    I, O = specs[0][1], specs[-1][2]
    x, g = rng.standard_normal((S, B, I + 2)).astype(np.float32), rng.standard_normal((S, B, O)).astype(np.float32)      # the input has a leading dimension of I + 2
    reset = (rng.uniform(size=(S, B)) < 0.2).astype(np.uint8)
    res = {}
    for be in (oracle, rocm):
        net = helpers.SeqNet(be, specs, params, S, B, fast_tanh=fast)
        ws, wsn = net.workspace()
        xd, rd = be.array(x), be.array(reset)
        r = rd.ptr if with_reset else None
        be.call("seq_zero_gradient", net.layers, net.n)
        be.call("seq_forward", net.layers, net.n, xd.ptr, I + 2, r, S, B, ws, wsn)
        out = {"y": net.output()}
        gd, dx = be.array(g), be.zeros((S, B, I))
        be.call("seq_backward", net.layers, net.n, xd.ptr, I + 2, gd.ptr, dx.ptr, r, S, B, 1, 0, ws, wsn)
        be.sync()
        out["grads"], out["dx"], out["d_output_after"] = net.grads.numpy(), dx.numpy(), gd.numpy()
        for flag in (0, 1):       # backward_input with and without the resets handed to the inner layers
            gd2, dx2 = be.array(g), be.zeros((S, B, I))
            be.call("seq_backward", net.layers, net.n, None, 0, gd2.ptr, dx2.ptr, r, S, B, 0, flag, ws, wsn)
            be.sync()
            out[f"dx_input_only_{flag}"] = dx2.numpy()
        res[be.name] = out
    for k, want in res["oracle"].items():
        assert rel_err(res["rocm"][k], want) <= TOL, (k, rel_err(res["rocm"][k], want))
    if with_reset and reset[1:].any() and S > 1:
        assert rel_err(res["oracle"]["dx_input_only_0"], res["oracle"]["dx_input_only_1"]) > 1e-3
        assert rel_err(res["oracle"]["dx_input_only_1"], res["oracle"]["dx"]) <= 1e-6


def with_initial_states(rng, specs, params):
    """The GRU layers' initial hidden states, which random_seq_params leaves at zero, drawn as well."""
    at = 0
    for kind, i, o, _ in specs:
        at += o * i + o if kind == 0 else 3 * o * i + 3 * o + 3 * o * o + 4 * o
        if kind:
            params[at - o:at] = rng.uniform(-0.5, 0.5, o)
    return params


# dense, GRU, GRU, dense: all layers of a pass in one launch (seq_stack.hip). (steps, batch, in, hidden, out, fast_tanh, hidden activation): the narrowest and widest inputs and
# outputs, one step, steps that fill neither the pairs nor the groups of six that the loops are unrolled to, exact and rational gates
STACK_CASES = [(7, 3, 1, 16, 1, True, "relu"), (13, 5, 16, 16, 16, False, "tanh"), (1, 2, 4, 16, 2, False, "relu"), (6, 9, 1, 32, 16, False, "sigmoid"), (11, 4, 16, 32, 1, True, "relu"),
               (1, 7, 3, 32, 3, True, "fast_tanh"), (2, 1, 5, 32, 2, False, "identity"), (100, 33, 9, 16, 5, True, "relu"), (65, 20, 13, 32, 7, False, "tanh"),
               # several hundred rows and the lines up to which a pass is one launch: the last with it, the first without (whose backward pass with weight gradients still is)
               (5, 700, 4, 32, 1, True, "relu"), (2, 2048, 3, 16, 2, True, "relu"), (2, 2049, 3, 16, 2, True, "relu"), (17, 1024, 4, 32, 1, True, "relu"), (17, 1025, 4, 32, 1, True, "relu"),
               (1, 16385, 2, 16, 1, True, "relu")]


@pytest.mark.parametrize("with_reset", [False, True])
@pytest.mark.parametrize("case", STACK_CASES)
def test_recurrent_approximators_in_one_launch_match_checker(oracle, rocm, case, with_reset):
    print("case", case, with_reset, flush=True)
    S, B, I, H, O, fast, act = case
    rng = np.random.default_rng(S * 10 + I)
    specs = [(0, I, H, act), (1, H, H, "identity"), (1, H, H, "identity"), (0, H, O, "identity")]
    model_against_checker(oracle, rocm, rng, specs, with_initial_states(rng, specs, helpers.random_seq_params(rng, specs)), S, B, fast, with_reset)


@pytest.mark.parametrize("place", ["loss gradient", "input", "row behind the loss gradient"])
@pytest.mark.parametrize("want_w", [1, 0])
@pytest.mark.parametrize("H", [16, 32])
def test_the_gradient_of_a_recurrent_approximators_input_may_replace_what_it_was_formed_from(rocm, H, want_w, place):
    """d_input in the memory of d_output or of x, or over rows of d_output that other rows of the batch come to later: the results of the call with memory of its own. The
    tolerance is that of the cases above (the call takes the layers one after the other then, other sums in fp32)."""
    S, B, I, O = 9, 21, 5, 5
    rng = np.random.default_rng(H + want_w)
    specs = [(0, I, H, "relu"), (1, H, H, "identity"), (1, H, H, "identity"), (0, H, O, "identity")]
    params = with_initial_states(rng, specs, helpers.random_seq_params(rng, specs))
    x, g = rng.standard_normal((S, B, I)).astype(np.float32), rng.standard_normal((S, B, O)).astype(np.float32)
    res = []
    for apart in (True, False):
        net = helpers.SeqNet(rocm, specs, params, S, B)
        ws, wsn = net.workspace()
        xd, gd = rocm.array(x), rocm.array(np.concatenate([g.ravel(), np.zeros(B * O, np.float32)]))
        own = rocm.zeros((S, B, I))
        rocm.call("seq_forward", net.layers, net.n, xd.ptr, I, None, S, B, ws, wsn)
        to = own.ptr if apart else xd.ptr if place == "input" else gd.ptr if place == "loss gradient" else gd.offset(O)
        rocm.call("seq_backward", net.layers, net.n, xd.ptr if want_w else None, I, gd.ptr, to, None, S, B, want_w, 0, ws, wsn)
        rocm.sync()
        dx = own.numpy().ravel() if apart else xd.numpy().ravel() if place == "input" else gd.numpy().ravel()[(0 if place == "loss gradient" else O):][:S * B * I]
        res.append((dx.copy(), net.grads.numpy()))
    assert rel_err(res[1][0], res[0][0]) <= TOL and rel_err(res[1][1], res[0][1]) <= TOL, (rel_err(res[1][0], res[0][0]), rel_err(res[1][1], res[0][1]))
    assert np.abs(res[0][0]).max() > 0


@pytest.mark.parametrize("want_w", [1, 0])
@pytest.mark.parametrize("H", [16, 32])
def test_an_infinite_gradient_of_a_recurrent_approximator_stays_infinite(oracle, rocm, H, want_w):
    """One output weight makes one unit's gradient overflow; every gate's gradient has the same sign and every weight on the way to the input is positive, so that the input's
    gradient is plus infinity everywhere (lanes without a gate that multiplied it by a zero weight made NaNs of it)."""
    S, B, I = 1, 3, 2
    rng = np.random.default_rng(H)
    specs = [(0, I, H, "identity"), (1, H, H, "identity"), (1, H, H, "identity"), (0, H, 1, "identity")]
    parts = [rng.uniform(0.1, 0.2, I * H), np.zeros(H)]
    for _ in range(2):      # n well below the initial state, the n gate's hidden part positive
        parts += [rng.uniform(0.01, 0.02, 3 * H * H), np.concatenate([np.zeros(2 * H), np.full(H, -3.0)]), rng.uniform(0.01, 0.02, 3 * H * H), np.zeros(3 * H), np.full(H, 0.9)]
    out = np.full(H, 1.0); out[3] = 1e30
    params = np.concatenate(parts + [out, np.zeros(1)]).astype(np.float32)
    x, g = rng.uniform(0.1, 1.0, (S, B, I)).astype(np.float32), np.full((S, B, 1), 1e20, np.float32)
    for be in (oracle, rocm):
        net = helpers.SeqNet(be, specs, params, S, B)
        ws, wsn = net.workspace()
        xd, gd, dx = be.array(x), be.array(g), be.zeros((S, B, I))
        be.call("seq_forward", net.layers, net.n, xd.ptr, I, None, S, B, ws, wsn)
        be.call("seq_backward", net.layers, net.n, xd.ptr if want_w else None, I, gd.ptr, dx.ptr, None, S, B, want_w, 0, ws, wsn)
        be.sync()
        assert (dx.numpy() == np.inf).all(), (be.name, dx.numpy())


def stacked_agents(rng, backends, S, B, OBS, ACT, actor_hidden, critic_hidden, first, spread=1.0):
    """SAC agents whose networks are all dense, GRU, GRU, dense"""
    specs = lambda i, h, o: [(0, i, h, "relu"), (1, h, h, "identity"), (1, h, h, "identity"), (0, h, o, "identity")]
    actor_specs, critic_specs = specs(OBS, actor_hidden, 2 * ACT), specs(OBS + ACT, critic_hidden, 1)
    draw = lambda s: with_initial_states(rng, s, helpers.random_seq_params(rng, s))
    critics = [draw(critic_specs) for _ in range(2)]
    params = np.concatenate([draw(actor_specs)] + critics + [c.copy() * spread for c in critics] + [np.array([np.log(0.5)], np.float32)]).astype(np.float32)
    hyper = dict(sas=helpers.capi.SasParameters(-20.0, 2.0, 1e-6, -float(ACT)))
    return params, [helpers.SacSequenceOnBackend(be, actor_specs, critic_specs, params, S, B, OBS, ACT, first, hyper) for be in backends]


# (steps, batch, observations, actions, actor's width, critics' width, first step in the targets)
STACKED_AGENTS = [(1, 3, 3, 1, 16, 32, True), (7, 13, 5, 2, 16, 32, False), (13, 5, 12, 4, 32, 16, True), (31, 64, 3, 1, 16, 16, True), (100, 40, 8, 8, 32, 32, False),
                  (2, 4800, 3, 1, 16, 16, True), (2, 4801, 3, 1, 16, 16, True)]      # the last batch whose passes share launches, and the first that does not


@pytest.mark.parametrize("case", STACKED_AGENTS)
def test_sac_sequence_updates_of_recurrent_approximators_in_shared_launches(oracle, rocm, case):
    """Actor and critics dense, GRU, GRU, dense: the passes of an update share launches (stacked_train_critics), the gradients are stored instead of added onto what the last
    update left, two optimisers share a launch. Three loop steps, the gradient tensors filled with other values before each."""
    print("case", case, flush=True)
    S, B, OBS, ACT = case[:4]
    rng = np.random.default_rng(S + B)
    _, agents = stacked_agents(rng, (oracle, rocm), S, B, OBS, ACT, *case[4:])
    T = S + 1 if case[6] else S
    for i in range(3):
        data = synthetic_sequence_batch(rng, S, B, OBS + ACT)
        nc, na = rng.standard_normal((T, B, ACT)).astype(np.float32), rng.standard_normal((S, B, ACT)).astype(np.float32)
        copy_agent(agents[0], agents[1])
        for a in agents:
            for net in (a.actor, *a.critics):
                stale = np.zeros(net.grads.shape, np.float32)      # the initial hidden states have no gradient: whatever stands there is the optimiser's
                stale[:net.specs[0][1] * net.specs[0][2]] = 3.0
                net.grads.upload(stale)
            a.log_alpha.upload(np.where(np.arange(4) == 1, 5.0, a.log_alpha.numpy()))
            a.set_batch(data); a.train(nc, na)
        # (the tolerance of the larger shapes above: fp32 sums over the steps in another order)
        compare_agents(agents[1], agents[0], (case, i), tol=2e-5)


@pytest.mark.parametrize("case", STACKED_AGENTS)
def test_both_critics_of_recurrent_approximators_in_one_call_leave_the_bits_of_the_two_calls(rocm, case):
    S, B, OBS, ACT = case[:4]
    rng = np.random.default_rng(S * 3 + B)
    params, agents = stacked_agents(rng, (rocm, rocm), S, B, OBS, ACT, *case[4:], spread=0.9)
    T = S + 1 if case[6] else S
    for i in range(3):
        data = synthetic_sequence_batch(rng, S, B, OBS + ACT)
        nc, na = rng.standard_normal((T, B, ACT)).astype(np.float32), rng.standard_normal((S, B, ACT)).astype(np.float32)
        for a, together in zip(agents, (False, True)):
            a.set_batch(data); a.train(nc, na, both_critics_in_one_call=together)
        assert np.array_equal(agents[0].parameters(), agents[1].parameters()) and agents[0].ages() == agents[1].ages(), (case, i)
        for key in ("target", "d_output", "next_q0", "next_q1", "next_lp", "nsavi"):
            assert np.array_equal(agents[0].buf[key].numpy(), agents[1].buf[key].numpy()), (case, i, key)
    assert np.abs(agents[1].parameters() - params).max() > 1e-4


@pytest.mark.parametrize("shared", ["critics", "actor and alpha"])
def test_optimisers_of_recurrent_approximators_that_share_an_age_step_one_after_the_other(rocm, shared):
    """One call for both critics against the two calls, and the actor's step against a copy whose ages are apart: where two optimisers count in one place the second goes on from
    the first's count, as two steps in a row do."""
    S, B, OBS, ACT = 7, 13, 5, 2
    rng = np.random.default_rng(11)
    _, agents = stacked_agents(rng, (rocm, rocm), S, B, OBS, ACT, 16, 32, False)
    data = synthetic_sequence_batch(rng, S, B, OBS + ACT)
    nc, na = rng.standard_normal((S, B, ACT)).astype(np.float32), rng.standard_normal((S, B, ACT)).astype(np.float32)
    for a, together in zip(agents, (False, True)):
        a.set_batch(data)
        if shared == "critics":
            a.c.critic_age[1] = a.c.critic_age[0]
        elif together:
            a.c.alpha_age = a.c.actor_age
        else:
            a.alpha_age.upload(np.array([2], np.uint32))
        a.train(nc, na, both_critics_in_one_call=together)
    assert np.array_equal(agents[0].parameters(), agents[1].parameters())
    assert [a.ages()[1 if shared == "critics" else 0] for a in agents] == ([3, 3] if shared == "critics" else [2, 3])


def test_a_second_critic_wider_than_the_workspace_is_sized_for_is_refused(rocm):
    S, B, OBS, ACT = 7, 13, 3, 1
    rng = np.random.default_rng(12)
    agent, wide = (stacked_agents(rng, (rocm,), S, B, OBS, ACT, 16, width, False)[1][0] for width in (16, 32))
    noise = rocm.array(rng.standard_normal((S, B, ACT)).astype(np.float32))
    lib, h = rocm.device.lib, rocm.device.handle
    agent.set_batch(synthetic_sequence_batch(rng, S, B, OBS + ACT))
    agent.c.critics[1], agent.c.critic_adam_tensors[1] = wide.critics[1].layers, wide.critics[1].adam
    assert lib.rlt_rocm_sac_sequence_train_critics(h, C.byref(agent.c), noise.ptr) == helpers.capi.RLT_E_INVALID_ARGUMENT
    assert lib.rlt_rocm_sac_sequence_train_critic(h, C.byref(agent.c), 1, noise.ptr) == helpers.capi.RLT_E_INVALID_ARGUMENT
    assert lib.rlt_rocm_sac_sequence_train_actor(h, C.byref(agent.c), noise.ptr) == helpers.capi.RLT_E_INVALID_ARGUMENT
    rocm.sync()


@pytest.mark.parametrize("n_layers", [3, 5])
def test_sac_sequence_updates_against_reference_vectors(oracle, rocm, n_layers):
    """The reference's own run (fixture): every loop step on the device from the checker's state, compared after the step in gradients,
    parameters, target networks, log_alpha and the training buffers; the checker itself must land on the fixture's snapshots bit for bit."""
    g = helpers.sac_sequence_golden()
    actor_specs, critic_specs, (B, S, obs, act, first, steps), hyper = helpers.sac_sequence_golden_case(g, n_layers)
    p = f"l{n_layers}_"
    agents = [helpers.SacSequenceOnBackend(be, actor_specs, critic_specs, g[p + "parameters_before"], S, B, obs, act, bool(first), hyper) for be in (oracle, rocm)]
    for i in range(steps):
        print("step", i, flush=True)
        copy_agent(agents[0], agents[1])
        for a in agents:
            helpers.sac_sequence_golden_step(a, g, n_layers, i)
        compare_agents(agents[1], agents[0], (n_layers, i))
        if i in g[p + "snapshots"]:
            assert np.array_equal(agents[0].parameters(), g[f"{p}s{i}_after"])


def synthetic_sequence_batch(rng, S, B, D):
    """A batch with the structure gather_batch produces: sequences end at random steps (final-step mask), the step after an end is a reset
    and carries the next observation; the `next` flags are the same ones shifted by a step."""
    final = (rng.uniform(size=(S, B)) < 0.3).astype(np.uint8); final[-1] = 1
    reset = np.zeros((S, B), np.uint8); reset[0] = 1; reset[1:] = final[:-1]
    next_reset = np.zeros((S + 1, B), np.uint8); next_reset[0] = 1; next_reset[1:] = final
    next_final = np.zeros((S + 1, B), np.uint8); next_final[1:] = final
    return dict(observations_actions_base=rng.standard_normal((S + 1, B, D)).astype(np.float32), rewards=rng.standard_normal((S, B)).astype(np.float32),
                terminated=(rng.uniform(size=(S, B)) < 0.1).astype(np.uint8), reset=reset, next_reset_base=next_reset, final_step_mask=final, next_final_step_mask_base=next_final)


@pytest.mark.parametrize("case", [(32, 128, 11, 3, 64, True), (10, 100, 5, 2, 32, False), (100, 100, 3, 1, 32, True)])
def test_sac_sequence_updates_at_larger_shapes(oracle, rocm, case):
    """Wider networks (hidden 64 takes the register-resident GRU kernels), several action dimensions, longer sequences -- up to the sequence
    length and batch size of the reference's recurrent Pendulum configuration (100 x 100) -- on synthetic batches, two loop steps each."""
    print("case", case, flush=True)
    S, B, OBS, ACT, H, first = case
    rng = np.random.default_rng(S + B)
    actor_specs = [(0, OBS, H, "relu"), (1, H, H, "identity"), (0, H, 2 * ACT, "identity")]
    critic_specs = [(0, OBS + ACT, H, "relu"), (1, H, H, "identity"), (1, H, H, "identity"), (0, H, 1, "identity")]
    critics = [helpers.random_seq_params(rng, critic_specs) for _ in range(2)]
    params = np.concatenate([helpers.random_seq_params(rng, actor_specs)] + critics + [c.copy() for c in critics] + [np.array([np.log(0.5)], np.float32)])
    hyper = dict(sas=helpers.capi.SasParameters(-20.0, 2.0, 1e-6, -float(ACT)))
    agents = [helpers.SacSequenceOnBackend(be, actor_specs, critic_specs, params, S, B, OBS, ACT, first, hyper) for be in (oracle, rocm)]
    T = S + 1 if first else S
    for i in range(2):
        data = synthetic_sequence_batch(rng, S, B, OBS + ACT)
        nc, na = rng.standard_normal((T, B, ACT)).astype(np.float32), rng.standard_normal((S, B, ACT)).astype(np.float32)
        copy_agent(agents[0], agents[1])
        for a in agents:
            a.set_batch(data); a.train(nc, na)
        compare_agents(agents[1], agents[0], (case, i), tol=2e-5)


@pytest.mark.parametrize("case", [(1, 1, 0), (7, 13, 3), (3, 85, 1), (2, 60001, 2)])
def test_sac_sequence_updates_at_the_edges_of_the_steps_between_the_passes(oracle, rocm, case):
    """One row, rows that fill neither a workgroup nor a word of the masks, masks off word boundaries, and more rows than the launches have threads; one loop step. The tolerance is
    that of the larger shapes (fp32 sums over the rows in another order)."""
    print("case", case, flush=True)
    S, B, shift = case
    OBS, ACT, H = 5, 2, 16
    rng = np.random.default_rng(S + B)
    actor_specs = [(0, OBS, H, "relu"), (1, H, H, "identity"), (0, H, 2 * ACT, "identity")]
    critic_specs = [(0, OBS + ACT, H, "relu"), (1, H, H, "identity"), (0, H, 1, "identity")]
    critics = [helpers.random_seq_params(rng, critic_specs) for _ in range(2)]
    params = np.concatenate([helpers.random_seq_params(rng, actor_specs)] + critics + [c.copy() for c in critics] + [np.array([np.log(0.5)], np.float32)])
    hyper = dict(sas=helpers.capi.SasParameters(-20.0, 2.0, 1e-6, -float(ACT)))
    agents = [helpers.SacSequenceOnBackend(be, actor_specs, critic_specs, params, S, B, OBS, ACT, True, hyper) for be in (oracle, rocm)]
    data = synthetic_sequence_batch(rng, S, B, OBS + ACT)
    shifted = {k: rocm.array(np.concatenate([np.zeros(shift, np.uint8), data[k].ravel()])) for k in ("final_step_mask", "next_final_step_mask_base", "reset")}
    for k, m in shifted.items():
        setattr(agents[1].c.batch, k, m.offset(shift))
    nc, na = rng.standard_normal((S + 1, B, ACT)).astype(np.float32), rng.standard_normal((S, B, ACT)).astype(np.float32)
    for a in agents:
        a.set_batch(data); a.train(nc, na)
    compare_agents(agents[1], agents[0], case, tol=2e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [(100, 100, 3, 1, 32, True), (10, 100, 5, 2, 32, False), (48, 64, 11, 3, 64, True)])
def test_both_critics_in_one_call_leave_the_bits_of_the_two_calls(rocm, case):
    """rlt_rocm_sac_sequence_train_critics (the target part once, the two critics' passes side by side on the handle's two streams from 48 steps up) against
    rlt_rocm_sac_sequence_train_critic for critic 0 and then for critic 1: three loop steps each from the same parameters, batches and noise; every parameter and the
    training buffers that both leave behind, bit for bit."""
    S, B, OBS, ACT, H, first = case
    rng = np.random.default_rng(S * 3 + B)
    actor_specs = [(0, OBS, H, "relu"), (1, H, H, "identity"), (0, H, 2 * ACT, "identity")]
    critic_specs = [(0, OBS + ACT, H, "relu"), (1, H, H, "identity"), (1, H, H, "identity"), (0, H, 1, "identity")]
    critics = [helpers.random_seq_params(rng, critic_specs) for _ in range(2)]
    params = np.concatenate([helpers.random_seq_params(rng, actor_specs)] + critics + [c.copy() * 0.9 for c in critics] + [np.array([np.log(0.5)], np.float32)])
    hyper = dict(sas=helpers.capi.SasParameters(-20.0, 2.0, 1e-6, -float(ACT)))
    agents = [helpers.SacSequenceOnBackend(rocm, actor_specs, critic_specs, params, S, B, OBS, ACT, first, hyper) for _ in range(2)]
    T = S + 1 if first else S
    for i in range(3):
        data = synthetic_sequence_batch(rng, S, B, OBS + ACT)
        nc, na = rng.standard_normal((T, B, ACT)).astype(np.float32), rng.standard_normal((S, B, ACT)).astype(np.float32)
        for a, together in zip(agents, (False, True)):
            a.set_batch(data); a.train(nc, na, both_critics_in_one_call=together)
        assert np.array_equal(agents[0].parameters(), agents[1].parameters()), (case, i)
        for key in ("target", "d_output", "next_q0", "next_q1", "next_lp", "nsavi"):
            if key in agents[0].buf:
                assert np.array_equal(agents[0].buf[key].numpy(), agents[1].buf[key].numpy()), (case, i, key)
        assert agents[0].ages() == agents[1].ages()
    assert np.abs(agents[1].parameters() - params).max() > 1e-4


def test_sac_sequence_of_length_one_equals_single_step_update_on_device(rocm):
    """Sequence length 1, dense layers only, every step final: the sequence entry points and the single-step entry points of the same library."""
    rng = np.random.default_rng(5)
    B, H, OBS, ACT = 256, 64, 3, 1
    actor_specs = [(0, OBS, H, "relu"), (0, H, H, "relu"), (0, H, 2 * ACT, "identity")]
    critic_specs = [(0, OBS + ACT, H, "relu"), (0, H, H, "relu"), (0, H, 1, "identity")]
    critics = [helpers.random_seq_params(rng, critic_specs) for _ in range(2)]
    params = np.concatenate([helpers.random_seq_params(rng, actor_specs)] + critics + [c.copy() for c in critics] + [np.array([np.log(0.5)], np.float32)])
    oab = rng.standard_normal((2, B, OBS + ACT)).astype(np.float32)
    rewards, terminated = rng.standard_normal((1, B)).astype(np.float32), (rng.uniform(size=(1, B)) < 0.2).astype(np.uint8)
    ones = np.ones((1, B), np.uint8)
    seq = helpers.SacSequenceOnBackend(rocm, actor_specs, critic_specs, params, 1, B, OBS, ACT, include_first=False)
    seq.set_batch(dict(observations_actions_base=oab, rewards=rewards, terminated=terminated, reset=ones, next_reset_base=np.ones((2, B), np.uint8), final_step_mask=ones,
                       next_final_step_mask_base=np.ones((2, B), np.uint8)))
    one = helpers.SacOnBackend(rocm, B, H, params)
    one.set_batch(oab, rewards[0], terminated[0])
    nc, na = rng.standard_normal((1, B, ACT)).astype(np.float32), rng.standard_normal((1, B, ACT)).astype(np.float32)
    seq.train(nc, na)
    n1, n2 = rocm.array(nc), rocm.array(na)
    for k in range(2):
        rocm.call("sac_train_critic", C.byref(one.c), k, n1.ptr)
    rocm.call("sac_update_critic_targets", C.byref(one.c))
    rocm.call("sac_train_actor", C.byref(one.c), n2.ptr)
    rocm.sync()
    assert rel_err(seq.parameters(), one.parameters()) <= TOL


def test_sac_sequence_rejects_inconsistent_arguments(rocm):
    rng = np.random.default_rng(0)
    specs_a, specs_c = [(0, 3, 16, "relu"), (1, 16, 16, "identity"), (0, 16, 2, "identity")], [(0, 4, 16, "relu"), (1, 16, 16, "identity"), (0, 16, 1, "identity")]
    critics = [helpers.random_seq_params(rng, specs_c) for _ in range(4)]
    params = np.concatenate([helpers.random_seq_params(rng, specs_a)] + critics + [np.zeros(1, np.float32)])
    agent = helpers.SacSequenceOnBackend(rocm, specs_a, specs_c, params, 4, 8, 3, 1)
    noise = rocm.zeros((5, 8, 1))
    lib, h = rocm.device.lib, rocm.device.handle
    assert lib.rlt_rocm_sac_sequence_train_critic(h, C.byref(agent.c), 2, noise.ptr) == helpers.capi.RLT_E_INVALID_ARGUMENT
    assert lib.rlt_rocm_sac_sequence_train_actor(h, C.byref(agent.c), None) == helpers.capi.RLT_E_INVALID_ARGUMENT
    agent.c.workspace_bytes = 16
    assert lib.rlt_rocm_sac_sequence_train_critic(h, C.byref(agent.c), 0, noise.ptr) == helpers.capi.RLT_E_INVALID_ARGUMENT
    agent.c.workspace_bytes = agent.ws.nbytes
    agent.c.action_dim = 2        # the actor's last layer has 2 outputs = 2 * 1
    assert lib.rlt_rocm_sac_sequence_update_critic_targets(h, C.byref(agent.c)) == helpers.capi.RLT_E_INVALID_ARGUMENT
    assert lib.rlt_rocm_seq_forward(h, agent.actor.layers, 3, noise.ptr, 2, None, 4, 8, None, 0) == helpers.capi.RLT_E_INVALID_ARGUMENT      # leading dimension below the input width
