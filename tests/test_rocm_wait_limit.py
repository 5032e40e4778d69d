"""The bounded waits of the kernels whose workgroups wait for each other (the persistent SAC loop, rl/algorithms/sac/loop/core/operations_generic.h:110-155
in one launch; the update kernels that end with the optimiser's step; the updates of wider agents, whose passes hand values over): with the bound set to one poll from the host (rlt_rocm_set_wait_limit) the first
workgroups to arrive give up at once, every kernel still ends normally, and the next rlt_rocm_check_status reports RLT_E_DEVICE_TIMEOUT. The error is
sticky on that handle, so each case runs on a device handle of its own; the same calls on a fresh handle with the default bound succeed."""
import ctypes as C

import numpy as np
import pytest

import helpers
from test_rocm_sac_update import agent_parameters, batch_of

pytestmark = pytest.mark.gpu
capi = helpers.capi


def one_critic_update(backend, params, batch):
    rng = np.random.default_rng(5)
    agent = helpers.SacOnBackend(backend, batch, 64, params, masks=False)
    agent.set_batch(*batch_of(rng, batch, 3, 1))
    noise = backend.array(rng.standard_normal((batch, 1)).astype(np.float32))
    rc = backend.device.lib.rlt_rocm_sac_train_critic(backend.device.handle, C.byref(agent.c), 0, noise.ptr)
    return rc, agent


def test_update_kernel_gives_up_and_reports():
    params = agent_parameters(np.random.default_rng(1), 3, 1)
    impatient = helpers.RocmBackend()
    try:
        impatient.call("set_wait_limit", 1)
        rc, _ = one_critic_update(impatient, params, 256)
        assert rc == 0                                   # the launch itself succeeds
        lib, h = impatient.device.lib, impatient.device.handle
        assert lib.rlt_rocm_check_status(h) == capi.RLT_E_DEVICE_TIMEOUT
        assert b"gave up waiting" in lib.rlt_rocm_error_string(capi.RLT_E_DEVICE_TIMEOUT)
        assert lib.rlt_rocm_check_status(h) == capi.RLT_E_DEVICE_TIMEOUT      # sticky: the handle's results are void from here on
    finally:
        impatient.close()
    patient = helpers.RocmBackend()
    try:
        rc, agent = one_critic_update(patient, params, 256)
        assert rc == 0 and patient.device.lib.rlt_rocm_check_status(patient.device.handle) == 0
        assert np.abs(agent.parameters() - params).max() > 1e-5 and int(agent.critics[0].age.numpy()[0]) == 2
    finally:
        patient.close()


def test_persistent_loop_gives_up_and_reports(oracle):
    batch = 256
    loop, cfg = helpers.make_loop(oracle, batch)
    for _ in range(cfg.n_warmup_steps):
        assert oracle.lib.rlt_oracle_sac_loop_step(loop) == 0
    params = helpers.loop_parameters(oracle, loop)
    impatient = helpers.RocmBackend()
    try:
        impatient.call("set_wait_limit", 1)
        agent = helpers.SacOnBackend(impatient, batch, 64, params, masks=False)
        runner = helpers.RunnerOnBackend(impatient, 10000, oracle, loop)
        lib, h = impatient.device.lib, impatient.device.handle
        assert lib.rlt_rocm_sac_pendulum_loop(h, C.byref(agent.c), C.byref(runner.c), C.byref(runner.rb.c), 50, 7, 0, None, None) == 0
        assert lib.rlt_rocm_check_status(h) == capi.RLT_E_DEVICE_TIMEOUT      # the kernel left its step loop and ended
    finally:
        impatient.close()
        oracle.lib.rlt_oracle_sac_loop_destroy(loop)


@pytest.mark.parametrize("minibatches", [0, 3])      # 0: a minibatch call; an epoch of three waits at the head of its launches too
def test_update_kernel_that_sums_per_xcd_gives_up_and_reports(minibatches):
    """PPO's minibatch kernel at 8,192 rows (rl/algorithms/ppo/operations_generic.h:163-309): its 256 workgroups add their blocks of partial gradient sums up
    per XCD inside the launch, which makes the 16 workgroups of a network on one XCD wait for each other."""
    O, A, H, B = 105, 8, 64, 8192
    rng = np.random.default_rng(4)
    params = np.concatenate([helpers.random_params(rng, [O, H, H, A]), np.log(np.full(A, 0.5, np.float32)), helpers.random_params(rng, [O, H, H, 1])])
    ld = O + A + 3
    data = rng.standard_normal((B, ld)).astype(np.float32)
    pp = capi.ppo_parameters()

    def one_update(backend):
        agent = helpers.PpoOnBackend(backend, O, A, H, H, B, params, "tanh", "tanh", capi.adam_parameters(3e-4, epsilon=1e-8))
        dd = backend.array(data)
        index = backend.array(np.tile(np.arange(B, dtype=np.uint32), max(minibatches, 1)))
        columns = (dd.offset(0), dd.offset(0), dd.offset(O), dd.offset(O + A), dd.offset(O + A + 1), dd.offset(O + A + 2), ld)
        lib, h = backend.device.lib, backend.device.handle
        if minibatches: rc = lib.rlt_rocm_ppo_train_epoch(h, C.byref(agent.c), C.byref(pp), *columns, index.ptr, minibatches, None)
        else: rc = lib.rlt_rocm_ppo_train_minibatch(h, C.byref(agent.c), C.byref(pp), *columns, None, None)
        return rc, agent

    impatient = helpers.RocmBackend()
    try:
        impatient.call("set_wait_limit", 1)
        rc, _ = one_update(impatient)
        assert rc == 0
        assert impatient.device.lib.rlt_rocm_check_status(impatient.device.handle) == capi.RLT_E_DEVICE_TIMEOUT
    finally:
        impatient.close()
    patient = helpers.RocmBackend()
    try:
        rc, agent = one_update(patient)
        assert rc == 0 and patient.device.lib.rlt_rocm_check_status(patient.device.handle) == 0
        assert np.abs(agent.parameters() - params).max() > 1e-5 and int(agent.actor.age.numpy()[0]) == 1 + max(minibatches, 1)
    finally:
        patient.close()


def test_ppo_epoch_that_gives_up_leaves_the_agent_as_it_was():
    """An epoch of three minibatches of 8,192 rows steps copies of the networks and brings them into the tensors with its last launch, which leaves parameters, log_std, moments and ages alone
    where a workgroup of the epoch gave up."""
    O, A, H, B, NMB = 17, 6, 64, 8192, 3
    rng = np.random.default_rng(6)
    params = np.concatenate([helpers.random_params(rng, [O, H, H, A]), np.log(np.full(A, 0.5, np.float32)), helpers.random_params(rng, [O, H, H, 1])])
    ld = O + A + 3
    data, pp = rng.standard_normal((B, ld)).astype(np.float32), capi.ppo_parameters()
    for limit, status in ((1, capi.RLT_E_DEVICE_TIMEOUT), (0, 0)):
        be = helpers.RocmBackend()
        try:
            agent = helpers.PpoOnBackend(be, O, A, H, H, B, params, "tanh", "tanh", capi.adam_parameters(3e-4, epsilon=1e-8))
            dd, index = be.array(data), be.array(np.tile(np.arange(B, dtype=np.uint32), NMB))
            state = lambda: [agent.parameters(), agent.m_log_std.numpy(), agent.v_log_std.numpy()] + [t.numpy() for net in (agent.actor, agent.critic) for t in (net.m, net.v, net.age)]      # noqa: E731
            before = state()
            be.call("set_wait_limit", limit)
            lib, h = be.device.lib, be.device.handle
            assert lib.rlt_rocm_ppo_train_epoch(h, C.byref(agent.c), C.byref(pp), dd.offset(0), dd.offset(0), dd.offset(O), dd.offset(O + A), dd.offset(O + A + 1), dd.offset(O + A + 2), ld,
                                                index.ptr, NMB, None) == 0
            after = state()      # read before the status, whose error sticks
            assert lib.rlt_rocm_check_status(h) == status
            assert [np.array_equal(a, b) for a, b in zip(before, after)] == [limit == 1] * len(before)
        finally:
            be.close()


def wide_state(agent, nets):
    """parameters, moments and ages of the trained networks, and every parameter of the agent"""
    return [agent.parameters()] + [a.numpy() for n in nets for a in (n.m, n.v, n.age)]


# (entry point, batch): one launch of gradients, and the batch shared out to groups of workgroups whose sums a third launch adds up
@pytest.mark.parametrize("batch", [100, 513])
@pytest.mark.parametrize("update", ["sac_train_critics", "sac_train_actor", "td3_train_critics"])
def test_update_of_a_wider_agent_gives_up_and_leaves_the_agent_as_it_was(update, batch):
    print("case", update, batch, flush=True)
    obs, act, hidden, rng = 6, 2, 256, np.random.default_rng(batch)
    nets = [[obs, hidden, hidden, 2 * act]] if update.startswith("sac") else [[obs, hidden, hidden, act]] * 2
    params = np.concatenate([helpers.random_params(rng, dims) for dims in nets + [[obs + act, hidden, hidden, 1]] * 4] + ([np.array([np.log(0.5)], np.float32)] if update.startswith("sac") else []))
    data, noise = batch_of(rng, batch, obs, act), rng.standard_normal((batch, act)).astype(np.float32)

    def run(limit):
        be = helpers.RocmBackend()
        try:
            if update.startswith("sac"):
                agent = helpers.SacOnBackend(be, batch, hidden, params, masks=False, obs=obs, act=act)
                agent.set_batch(*data)
            else:
                agent = helpers.Td3OnBackend(be, batch, hidden, params, obs=obs, act=act)
                agent.set_batch(*data, 0.1 * noise)
            trained = [agent.actor] if update.endswith("actor") else agent.critics
            before = wide_state(agent, trained)
            alpha = [agent.log_alpha.numpy(), agent.alpha_age.numpy()] if update == "sac_train_actor" else []
            nd = be.array(noise)
            be.call("set_wait_limit", limit)
            lib, h = be.device.lib, be.device.handle
            if update == "sac_train_critics":
                rc = lib.rlt_rocm_sac_train_critics(h, C.byref(agent.c), nd.ptr, 1)
            elif update == "sac_train_actor":
                rc = lib.rlt_rocm_sac_train_actor(h, C.byref(agent.c), nd.ptr)
            else:
                rc = lib.rlt_rocm_td3_train_critics(h, C.byref(agent.c), nd.ptr, nd.ptr)
            assert rc == 0
            after = wide_state(agent, trained)      # read before the status, whose error sticks
            if alpha:
                assert np.array_equal(agent.log_alpha.numpy()[[0, 2, 3]], alpha[0][[0, 2, 3]]) == (limit == 1) and agent.alpha_age.numpy()[0] == alpha[1][0] + (limit != 1)
            return before, after, lib.rlt_rocm_check_status(h)
        finally:
            be.close()

    before, after, status = run(1)
    assert status == capi.RLT_E_DEVICE_TIMEOUT
    assert all(np.array_equal(a, b) for a, b in zip(before, after))
    before, after, status = run(0)
    assert status == 0 and not any(np.array_equal(a, b) for a, b in zip(before, after))
