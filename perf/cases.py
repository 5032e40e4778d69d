"""Workloads of the dense-network training hot path as a program on this library runs them, for measuring one tree of the code against another.

listed() are the sizes that this repository's configurations, zoo agents and benchmark name, with one ragged batch among them; draw() spreads over
the ranges that they stand for. prepare() lays a case's networks, optimiser state and data out in GPU memory (torch's allocator holds it, the
library gets the pointers), run() makes one pass through the C ABI and returns the buffers that it wrote.

Networks are taken in the middle of a training: Adam's moments are filled and its age is past the bias correction's reach, so that a step
depends smoothly on the gradient.
"""
import ctypes as C
import importlib.util
import math
import os
import sys

import numpy as np
import torch


def _package():
    if "rl_tools_amd" not in sys.modules:
        path = os.path.join(os.getcwd(), "rl-tools_amd")
        spec = importlib.util.spec_from_file_location("rl_tools_amd", os.path.join(path, "__init__.py"), submodule_search_locations=[path])
        module = importlib.util.module_from_spec(spec)
        sys.modules["rl_tools_amd"] = module
        spec.loader.exec_module(module)
    return sys.modules["rl_tools_amd"]


capi = _package().capi
builders = _package().builders

# ------------------------------------------------------------------ the cases


def listed():
    return [
        # acting: the policy of one environment on its observation, between two environment steps
        dict(name="act_1", kind="evaluate", inputs=17, outputs=6, batch=1),
        # supervised steps of 17-256-256-6 at the smallest, an ordinary and the largest batch: clear, forward + backward on an MSE target, Adam ...
        dict(name="mlp_step_256", kind="mlp", inputs=17, outputs=6, batch=256, separate=False),
        # ... and with forward(), the loss gradient and backward() as calls of their own, on a batch that fills no tile evenly
        dict(name="mlp_calls_4001", kind="mlp", inputs=17, outputs=6, batch=4001, separate=True),
        dict(name="mlp_step_65536", kind="mlp", inputs=17, outputs=6, batch=65536, separate=False),
        # whole SAC loop steps on the Pendulum (environment step, gather, both critics, targets, actor), twenty to a launch
        dict(name="sac_loop_20", kind="sac_loop", steps=20, batch=256),
        # one set of SAC updates of the AcrobotSwingup's agent
        dict(name="sac_set_256", kind="sac", observation=6, action=1, hidden=256, batch=256),
        # one set of TD3 updates of the Ant's agent
        dict(name="td3_set_256", kind="td3", observation=27, action=8, hidden=256, batch=256),
        # a PPO iteration's training half: advantages of 4,096 environments x 128 steps, then four epochs of minibatches of 8,192
        dict(name="ppo_8192", kind="ppo", observation=105, action=8, envs=4096, steps=128, minibatch=8192, epochs=4),
        # vectorised collection: one sampled step of 65,536 Pendulums into their replay rings, and a batch of 4,096 out of them
        dict(name="collect_65536", kind="collect", envs=65536, capacity=16, batch=4096),
        # sequence model steps (GRU 146-64 over 64 steps, head 64-64-4), few and many sequences
        dict(name="gru_64", kind="gru", inputs=146, hidden=64, steps=64, batch=64),
        dict(name="gru_1024", kind="gru", inputs=146, hidden=64, steps=64, batch=1024),
        # one set of SAC updates with recurrent networks: 100 sequences of 100 steps (the Pendulum with memory)
        dict(name="sac_sequences_100", kind="sac_sequence", steps=100, batch=100),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["evaluate", "mlp", "mlp", "mlp", "sac_loop", "sac", "td3", "ppo", "collect", "gru", "gru", "sac_sequence"])
    if kind == "evaluate":
        return dict(kind=kind, inputs=rng.randint(3, 32), outputs=rng.randint(1, 8), batch=_log(rng, 1, 1024))
    if kind == "mlp":
        return dict(kind=kind, inputs=rng.randint(3, 32), outputs=rng.randint(1, 8), batch=_log(rng, 200, 65536), separate=rng.random() < 0.5)
    if kind == "sac_loop":      # the loop takes batches of whole sixteens
        return dict(kind=kind, steps=_log(rng, 5, 60), batch=16 * rng.randint(4, 16))
    if kind in ("sac", "td3"):
        return dict(kind=kind, observation=rng.randint(3, 27), action=rng.randint(1, 8), hidden=rng.choice([64, 256, 256]), batch=rng.randint(64, 256))
    if kind == "ppo":
        envs, steps = _log(rng, 256, 4096), rng.randint(64, 128)
        return dict(kind=kind, observation=rng.randint(3, 105), action=rng.randint(1, 8), envs=envs, steps=steps, minibatch=min(8192, envs * steps // rng.randint(8, 64)),
                    epochs=rng.randint(1, 4))
    if kind == "collect":
        return dict(kind=kind, envs=_log(rng, 500, 65536), capacity=rng.randint(4, 16), batch=_log(rng, 100, 4096))
    if kind == "gru":
        return dict(kind=kind, inputs=rng.randint(3, 146), hidden=rng.choice([16, 32, 64, 64]), steps=rng.randint(16, 64), batch=_log(rng, 16, 1024))
    return dict(kind=kind, steps=rng.randint(20, 100), batch=rng.randint(32, 100))


# ------------------------------------------------------------------ memory and handle

_DTYPES = {"float32": torch.float32, "uint8": torch.uint8, "uint32": torch.int32, "int32": torch.int32, "uint64": torch.int64}
_device = None


def _handle():
    """The library's handle of the GPU: one per process, as a program keeps it."""
    global _device
    if _device is None:
        _device = capi.Device(0)
    return _device


class _Memory:
    """A torch tensor as the builders' device array."""

    def __init__(self, tensor):
        self.tensor, self.shape, self.ptr = tensor, tuple(tensor.shape), tensor.data_ptr()
        self.nbytes = tensor.numel() * tensor.element_size()

    def offset(self, elements):
        return self.ptr + int(elements) * self.tensor.element_size()

    def upload(self, array):
        self.tensor.copy_(torch.from_numpy(np.ascontiguousarray(array).view(str(self.tensor.dtype).replace("torch.", ""))).reshape(self.shape))
        return self

    def numpy(self):
        return self.tensor.cpu().numpy()


class _Backend:
    """What the package's builders ask of a backend, with torch's memory. One for each state, which it keeps alive."""

    name = "rocm"

    def __init__(self, seed):
        self.library = _handle()
        self.device = self
        self.lib, self.handle = self.library.lib, self.library.handle
        self.rng = np.random.default_rng(seed)
        self.generator = torch.Generator("cuda").manual_seed(seed)
        self.kept = []
        self._workspace = None

    def keep(self, tensor):
        m = _Memory(tensor.contiguous())
        self.kept.append(m)
        return m

    def array(self, a):
        a = np.array(a, order="C")
        return self.keep(torch.from_numpy(a.view(np.int32) if a.dtype == np.uint32 else a).cuda())

    def zeros(self, shape, dtype=np.float32):
        return self.keep(torch.zeros(tuple(shape), dtype=_DTYPES[np.dtype(dtype).name], device="cuda"))

    def empty(self, shape, dtype=np.float32):
        return self.keep(torch.empty(tuple(shape), dtype=_DTYPES[np.dtype(dtype).name], device="cuda"))

    def workspace(self, nbytes):
        if self._workspace is None or self._workspace.nbytes < nbytes:
            self._workspace = self.empty((max(int(nbytes), 4),), np.uint8)
        return self._workspace.ptr, self._workspace.nbytes

    def randn(self, *shape):
        return torch.randn(shape, generator=self.generator, device="cuda")

    def rand(self, *shape):
        return torch.rand(shape, generator=self.generator, device="cuda")

    def call(self, name, *args):
        self.library.call(name, *args)

    def middle_of_training(self, m, v, age=None, gradient=1e-3):
        m.tensor.copy_(0.3 * gradient * self.randn(*m.shape))
        v.tensor.copy_(gradient * gradient * (0.5 + self.rand(*v.shape)))
        if age is not None:
            age.tensor.fill_(1000)


def _network_outputs(net):
    return [net.params.tensor, net.grads.tensor, net.m.tensor, net.v.tensor]


# ------------------------------------------------------------------ what each kind of case prepares and runs


def _prepare_evaluate(b, c):
    dims = [c["inputs"], 256, 256, c["outputs"]]
    net = builders.Mlp(b, dims, builders.random_params(b.rng, dims), c["batch"], "relu", "tanh", trainable=False)
    x, y = b.keep(b.randn(c["batch"], dims[0])), b.zeros((c["batch"], dims[3]))
    workspace = net.workspace()

    def run():
        b.call("mlp_evaluate", net.layers, net.n, x.ptr, dims[0], y.ptr, dims[3], c["batch"], *workspace)
        return y.tensor
    return run


def _prepare_mlp(b, c):
    dims, n = [c["inputs"], 256, 256, c["outputs"]], c["batch"]
    net = builders.Mlp(b, dims, builders.random_params(b.rng, dims), n)
    b.middle_of_training(net.m, net.v, net.age)
    x, target = b.keep(b.randn(n, dims[0])), b.keep(b.randn(n, dims[3]))
    y, d = b.zeros((n, dims[3])), b.zeros((n, dims[3]))
    workspace = net.workspace()
    adam = capi.adam_parameters(epsilon=1e-8)
    inputs, outputs = dims[0], dims[3]

    def run():
        b.call("mlp_zero_gradient", net.layers, net.n)
        if c["separate"]:
            b.call("mlp_forward", net.layers, net.n, x.ptr, inputs, n)
            b.call("mse_gradient", net.out[2].ptr, outputs, target.ptr, outputs, d.ptr, outputs, n, outputs, 1.0, None)
            b.call("mlp_backward", net.layers, net.n, x.ptr, inputs, d.ptr, outputs, None, 0, n, 1, *workspace)
        else:
            b.call("mlp_forward_backward", net.layers, net.n, x.ptr, inputs, y.ptr, outputs, None, 0, target.ptr, outputs, 2.0 / (n * outputs), n, *workspace)
        b.call("adam_step", net.adam, net.n_adam, C.byref(adam), net.age.ptr, 0.0, None)
        kept = [t.tensor for t in net.pre + net.out] if c["separate"] else [y.tensor]
        return _network_outputs(net) + kept
    return run


def _agent_parameters(b, actor, critic, twice_actor):
    actor_parameters = builders.random_params(b.rng, actor)
    critics = [builders.random_params(b.rng, critic) for _ in range(2)]
    return np.concatenate([actor_parameters] * (2 if twice_actor else 1) + critics + critics)


def _sac_agent(b, observation, action, hidden, batch):
    parameters = _agent_parameters(b, [observation, hidden, hidden, 2 * action], [observation + action, hidden, hidden, 1], False)
    agent = builders.SacOnBackend(b, batch, hidden, np.append(parameters, np.float32(math.log(0.5))), masks=False, obs=observation, act=action)
    for net in [agent.actor] + agent.critics:
        b.middle_of_training(net.m, net.v, net.age)
    agent.alpha_age.tensor.fill_(1000)
    agent.log_alpha.tensor[3] = 1e-2
    return agent


def _sac_outputs(agent):
    nets = sum((_network_outputs(net) for net in [agent.actor] + agent.critics), [])
    return nets + [t.params.tensor for t in agent.targets] + [agent.log_alpha.tensor, agent.target_q.tensor]


def _transitions(b, agent, batch, observation, action):
    """A batch of transitions: observations of unit variance, actions inside (-1, 1), few terminal ones."""
    oab = b.randn(2, batch, observation + action)
    oab[:, :, observation:] = torch.tanh(oab[:, :, observation:])
    agent.oab.tensor.copy_(oab)
    agent.rewards.tensor.copy_(b.randn(batch))
    agent.terminated.tensor.copy_(b.rand(batch) < 0.05)


def _pendulum_transitions(b, rows):
    """Rows of a Pendulum's replay ring: [observation, action, reward, next observation, terminated, truncated]."""
    angle, speed, action = (2 * b.rand(rows) - 1) * math.pi, b.randn(rows).clamp(-8, 8), 2 * b.rand(rows) - 1
    reward = -(angle.square() + 0.1 * speed.square() + 0.001 * (2 * action).square())
    next_speed = (speed + (15.0 * torch.sin(angle) + 3.0 * 2 * action) * 0.05).clamp(-8, 8)
    next_angle = angle + next_speed * 0.05
    zero = torch.zeros_like(angle)
    return torch.stack([torch.cos(angle), torch.sin(angle), speed, action, reward, torch.cos(next_angle), torch.sin(next_angle), next_speed, zero, zero], 1)


def _pendulum_runner(b, envs, capacity):
    """Environments in the middle of their episodes, with full rings."""
    ring = builders.ReplayOnBackend(b, envs, capacity)
    ring.data.tensor.copy_(_pendulum_transitions(b, envs * capacity))
    ring.position.tensor.copy_((b.rand(envs) * capacity).int().clamp(max=capacity - 1))
    ring.full.tensor.fill_(1)
    states = b.keep(torch.stack([(2 * b.rand(envs) - 1) * math.pi, 2 * b.rand(envs) - 1], 1))
    episode_step, episode_return, truncated = b.zeros((envs,), np.uint32), b.zeros((envs,)), b.zeros((envs,), np.uint8)
    episode_step.tensor.copy_((b.rand(envs) * 199).int())
    runner = capi.PendulumRunner(states.ptr, episode_step.ptr, episode_return.ptr, truncated.ptr, envs, 200, capi.pendulum_parameters())
    outputs = [m.tensor for m in (states, episode_step, episode_return, truncated, ring.data, ring.position, ring.full)]
    return runner, ring, outputs


def _prepare_sac_loop(b, c):
    agent = _sac_agent(b, 3, 1, 64, c["batch"])
    runner, ring, runner_outputs = _pendulum_runner(b, 1, 10000)
    loss = b.zeros((c["steps"], 2))
    outputs = capi.SacLoopOutputs()
    outputs.critic_loss = loss.ptr
    done = [0]

    def run():
        b.call("sac_pendulum_loop", C.byref(agent.c), C.byref(runner), C.byref(ring.c), c["steps"], 1234, done[0], None, C.byref(outputs))
        done[0] += c["steps"]
        return _sac_outputs(agent)[:-1] + runner_outputs + [loss.tensor]
    return run


def _prepare_sac(b, c):
    agent = _sac_agent(b, c["observation"], c["action"], c["hidden"], c["batch"])
    _transitions(b, agent, c["batch"], c["observation"], c["action"])
    noise = b.zeros((c["batch"], c["action"]))
    passes = [0]

    def run():
        passes[0] += 1
        b.call("sac_train_critics_drawn", C.byref(agent.c), noise.ptr, 77, 2 * passes[0], 1)
        b.call("sac_train_actor_drawn", C.byref(agent.c), noise.ptr, 77, 2 * passes[0] + 1)
        return _sac_outputs(agent)
    return run


def _prepare_td3(b, c):
    observation, action, hidden = c["observation"], c["action"], c["hidden"]
    parameters = _agent_parameters(b, [observation, hidden, hidden, action], [observation + action, hidden, hidden, 1], True)
    agent = builders.Td3OnBackend(b, c["batch"], hidden, parameters, obs=observation, act=action)
    for net in [agent.actor] + agent.critics:
        b.middle_of_training(net.m, net.v, net.age)
    _transitions(b, agent, c["batch"], observation, action)
    noise = b.zeros((2, c["batch"], action))
    passes = [0]

    def run():
        passes[0] += 1
        k = 4 * passes[0]
        draws = capi.Td3CriticDraws(1, k, (C.c_uint64 * 2)(k + 1, k + 2), 0.2, 0.5)
        b.call("td3_train_critics_drawn", C.byref(agent.c), C.byref(draws), noise.ptr, 1)
        b.call("td3_train_actor_drawn", C.byref(agent.c), 1, k + 3, noise.ptr)
        b.call("td3_update_actor_target", C.byref(agent.c))
        nets = sum((_network_outputs(net) for net in [agent.actor] + agent.critics), [])
        return nets + [t.params.tensor for t in [agent.actor_target] + agent.targets] + [agent.target_q.tensor]
    return run


def _tanh_network(x, parameters, dims):
    for i in range(3):
        w, parameters = parameters[:dims[i] * dims[i + 1]].view(dims[i + 1], dims[i]), parameters[dims[i] * dims[i + 1]:]
        x = torch.addmm(parameters[:dims[i + 1]], x, w.t())
        x, parameters = torch.tanh(x) if i < 2 else x, parameters[dims[i + 1]:]
    return x


def _prepare_ppo(b, c):
    O, A, envs, steps = c["observation"], c["action"], c["envs"], c["steps"]
    rows, n = envs * steps, min(c["minibatch"], envs * steps)
    adims, cdims = [O, 64, 64, A], [O, 64, 64, 1]
    actor = builders.random_params(b.rng, adims)
    actor[-(64 * A + A):] *= 0.1
    parameters = np.concatenate([actor, np.log(np.full(A, 0.5, np.float32)), builders.random_params(b.rng, cdims)]).astype(np.float32)
    agent = builders.PpoOnBackend(b, O, A, 64, 64, n, parameters, "tanh", "tanh", capi.adam_parameters(3e-4, epsilon=1e-8))
    for net in (agent.actor, agent.critic):
        b.middle_of_training(net.m, net.v, net.age, gradient=1e-2)
    agent.v_log_std.tensor.fill_(1e-4)
    # the dataset as the collection leaves it: actions sampled around the actor's means, the critic's values, one row of values more per environment
    data = b.zeros((rows + envs, O + A + 7))
    t = data.tensor
    t[:, :O] = b.randn(rows + envs, O)
    noise = b.randn(rows + envs, A)
    t[:, O:O + A] = _tanh_network(t[:, :O], agent.actor.params.tensor, adims) + 0.5 * noise
    t[:, O + A] = (-0.5 * math.log(2 * math.pi) - math.log(0.5) - 0.5 * noise.square()).sum(1)
    t[:, O + A + 1] = b.randn(rows + envs)
    t[:, O + A + 3] = (b.rand(rows + envs) < 0.01).float()
    t[:, O + A + 2] = t[:, O + A + 3] * (b.rand(rows + envs) < 0.5)
    t[:, O + A + 4] = _tanh_network(t[:, :O], agent.critic.params.tensor, cdims)[:, 0]
    at = lambda column: data.offset(O + A + column)      # noqa: E731
    permutations = [b.keep(torch.randperm(rows, generator=b.generator, device="cuda", dtype=torch.int32)) for _ in range(c["epochs"])]
    losses = b.zeros((c["epochs"], rows // n))
    options = capi.ppo_parameters()
    ld = O + A + 7

    def run():
        b.call("ppo_gae", at(1), at(2), at(3), at(4), at(5), at(6), ld, envs, steps, 0.99, 0.95, 0)
        for e, permutation in enumerate(permutations):
            b.call("ppo_train_epoch", C.byref(agent.c), C.byref(options), data.ptr, data.ptr, data.offset(O), at(0), at(5), at(6), ld, permutation.ptr, rows // n,
                   losses.offset(e * (rows // n)))
        return _network_outputs(agent.actor) + _network_outputs(agent.critic) + [agent.log_std.tensor, losses.tensor, t[:rows, O + A + 5:]]
    return run


def _prepare_collect(b, c):
    runner, ring, outputs = _pendulum_runner(b, c["envs"], c["capacity"])
    dims = [3, 64, 64, 2]
    actor = builders.Mlp(b, dims, builders.random_params(b.rng, dims), c["envs"], "relu", "identity", trainable=False)
    sas = capi.SasParameters(-20.0, 2.0, 1e-6, -1.0)
    n = c["batch"]
    noise, oab, rewards, terminated = b.zeros((c["envs"],)), b.zeros((2, n, 4)), b.zeros((n,)), b.zeros((n,), np.uint8)
    env_indices, offsets = b.zeros((n,), np.uint32), b.zeros((n,), np.uint32)
    passes = [0]

    def run():
        passes[0] += 1
        k = 4 * passes[0]
        b.call("pendulum_runner_step_drawn", C.byref(runner), C.byref(ring.c), actor.layers, actor.n, C.byref(sas), noise.ptr, 5, k, k + 1)
        b.call("gather_batch_drawn", C.byref(ring.c), 5, k + 2, env_indices.ptr, offsets.ptr, 200, n, oab.ptr, rewards.ptr, terminated.ptr, None, None, None, None)
        return outputs + [oab.tensor, rewards.tensor, terminated.tensor]
    return run


def _prepare_gru(b, c):
    S, B, I, H = c["steps"], c["batch"], c["inputs"], c["hidden"]
    rows = S * B
    scale = lambda *shape: b.rng.uniform(-1, 1, shape) / math.sqrt(H)      # noqa: E731
    parameters = dict(W_i=scale(3 * H, I), b_i=scale(3 * H), W_h=scale(3 * H, H), b_h=scale(3 * H), h0=np.zeros(H))
    gru = builders.GruOnBackend(b, S, B, I, H, parameters)
    head = builders.Mlp(b, [H, 64, 4], builders.random_params(b.rng, [H, 64, 4]), rows, "tanh", "identity")
    b.middle_of_training(head.m, head.v)
    tensors, weights = [], []
    for k, (p, g) in enumerate(((gru.W_i, gru.dW_i), (gru.b_i, gru.db_i), (gru.W_h, gru.dW_h), (gru.b_h, gru.db_h))):
        m, v = b.zeros(p.shape), b.zeros(p.shape)
        b.middle_of_training(m, v)
        tensors.append(capi.AdamTensor(p.ptr, g.ptr, m.ptr, v.ptr, None, int(np.prod(p.shape)), 1 + k % 2))
        weights.append(p.tensor)
    tensors += [head.adam[i] for i in range(head.n_adam)]
    tensors = (capi.AdamTensor * len(tensors))(*tensors)
    age = b.array(np.array([1000], np.uint32))
    adam = capi.adam_parameters(epsilon=1e-8)
    x, target = b.keep(b.randn(S, B, I)), b.keep(b.randn(rows, 4))
    y, d_h = b.zeros((rows, 4)), b.zeros((S, B, H))
    workspace = head.workspace()
    n_gradients = gru.grads.tensor.numel()

    def run():
        b.call("fill_f32", gru.grads.ptr, 1, n_gradients, n_gradients, 0.0)
        b.call("mlp_zero_gradient", head.layers, head.n)
        b.call("gru_forward", C.byref(gru.c), x.ptr, None, S, B, gru.ws, gru.wsn)
        b.call("mlp_forward_backward_input", head.layers, head.n, gru.out.ptr, H, y.ptr, 4, None, 0, target.ptr, 4, 2.0 / (rows * 4), d_h.ptr, H, rows, *workspace)
        b.call("gru_backward", C.byref(gru.c), x.ptr, d_h.ptr, None, None, S, B, 1, gru.ws, gru.wsn)
        b.call("adam_step", tensors, len(tensors), C.byref(adam), age.ptr, 0.0, None)
        return weights + [gru.grads.tensor, gru.out.tensor, y.tensor] + _network_outputs(head)
    return run


_SEQUENCE_ACTOR = [(0, 3, 16, "relu"), (1, 16, 16, "identity"), (1, 16, 16, "identity"), (0, 16, 2, "identity")]
_SEQUENCE_CRITIC = [(0, 4, 32, "relu"), (1, 32, 32, "identity"), (1, 32, 32, "identity"), (0, 32, 1, "identity")]


def _prepare_sac_sequence(b, c):
    S, B = c["steps"], c["batch"]
    critics = [builders.random_seq_params(b.rng, _SEQUENCE_CRITIC) for _ in range(2)]
    parameters = np.concatenate([builders.random_seq_params(b.rng, _SEQUENCE_ACTOR)] + critics + critics + [np.zeros(1, np.float32)])
    agent = builders.SacSequenceOnBackend(b, _SEQUENCE_ACTOR, _SEQUENCE_CRITIC, parameters, S, B, 3, 1, True)
    for net in [agent.actor] + agent.critics:
        b.middle_of_training(net.m, net.v, net.age)
    agent.alpha_age.tensor.fill_(1000)
    agent.log_alpha.tensor[3] = 1e-2
    # sequences of a replay ring: some end inside the batch, the step after an end starts from the initial hidden state
    final = (b.rng.uniform(size=(S, B)) < 0.05).astype(np.uint8)
    final[-1] = 1
    reset, next_reset, next_final = np.zeros((S, B), np.uint8), np.zeros((S + 1, B), np.uint8), np.zeros((S + 1, B), np.uint8)
    reset[0], next_reset[0] = 1, 1
    reset[1:], next_reset[1:], next_final[1:] = final[:-1], final, final
    oab = b.rng.standard_normal((S + 1, B, 4)).astype(np.float32)
    oab[:, :, 3:] = np.tanh(oab[:, :, 3:])
    agent.set_batch(dict(observations_actions_base=oab, rewards=b.rng.standard_normal((S, B)).astype(np.float32), terminated=np.zeros((S, B), np.uint8), reset=reset,
                         next_reset_base=next_reset, final_step_mask=final, next_final_step_mask_base=next_final))
    noise_critic, noise_actor = b.keep(b.randn(S + 1, B, 1)), b.keep(b.randn(S, B, 1))

    def run():
        b.call("sac_sequence_train_critics", C.byref(agent.c), noise_critic.ptr)
        b.call("sac_sequence_update_critic_targets", C.byref(agent.c))
        b.call("sac_sequence_train_actor", C.byref(agent.c), noise_actor.ptr)
        nets = sum((_network_outputs(net) for net in [agent.actor] + agent.critics), [])
        return nets + [t.params.tensor for t in agent.targets] + [agent.log_alpha.tensor, agent.buf["target"].tensor]
    return run


_PREPARE = dict(evaluate=_prepare_evaluate, mlp=_prepare_mlp, sac_loop=_prepare_sac_loop, sac=_prepare_sac, td3=_prepare_td3, ppo=_prepare_ppo, collect=_prepare_collect,
                gru=_prepare_gru, sac_sequence=_prepare_sac_sequence)


def prepare(case, seed):
    backend = _Backend(seed)
    run_pass = _PREPARE[case["kind"]](backend, case)
    torch.cuda.synchronize()      # torch filled the buffers on its stream, the library works on its own
    return run_pass


def run(state):
    return state()


# ------------------------------------------------------------------ the work of a pass, and how far apart two correct passes may be


def _dense(dims):
    """(parameters, flop per row forward, flop per row of the weight gradients and the inner input gradients)"""
    products = [dims[i] * dims[i + 1] for i in range(len(dims) - 1)]
    return sum(products) + sum(dims[1:]), 2 * sum(products), 2 * sum(products) + 2 * sum(products[1:])


def _sequential(specs):
    parameters = builders.seq_param_count(specs)
    forward = sum(2 * i * o if kind == 0 else 6 * (i * o + o * o) for kind, i, o, _ in specs)
    return parameters, forward, 2 * forward


def _updates(actor, critic, batch, target_actor, row_bytes):
    """An actor-critic's update set: the target part once, two critics forward and backward, the actor through both (SAC) or the first (TD3) critic. Adam reads
    and writes 24 bytes per parameter, a soft update 12."""
    (pa, fa, ba), (pc, fc, bc) = actor, critic
    through = 1 if target_actor else 2
    flops = batch * (fa + 2 * fc + 2 * (fc + bc) + fa + through * 2 * fc + ba)
    return dict(bytes=28 * (pa + 2 * pc) + 12 * (2 * pc + (pa if target_actor else 0)) + batch * row_bytes, flops=flops)


def work(case):
    kind = case["kind"]
    if kind in ("evaluate", "mlp"):
        n, i, o = case["batch"], case["inputs"], case["outputs"]
        p, forward, backward = _dense([i, 256, 256, o])
        if kind == "evaluate":
            return dict(bytes=4 * (p + n * (i + o)), flops=n * forward)
        rows = i + 2 * o + (2 * (512 + o) if case["separate"] else 0)
        return dict(bytes=28 * p + 4 * n * rows, flops=n * (forward + backward))
    if kind == "sac_loop":
        one = _updates(_dense([3, 64, 64, 2]), _dense([4, 64, 64, 1]), case["batch"], False, 44)
        return dict(bytes=case["steps"] * case["batch"] * 44 + one["bytes"], flops=case["steps"] * one["flops"])
    if kind in ("sac", "td3"):
        O, A, H = case["observation"], case["action"], case["hidden"]
        return _updates(_dense([O, H, H, A if kind == "td3" else 2 * A]), _dense([O + A, H, H, 1]), case["batch"], kind == "td3", 8 * (O + A) + 5)
    if kind == "ppo":
        O, A, rows = case["observation"], case["action"], case["envs"] * case["steps"]
        used = rows // min(case["minibatch"], rows) * min(case["minibatch"], rows) * case["epochs"]
        (pa, fa, ba), (pc, fc, bc) = _dense([O, 64, 64, A]), _dense([O, 64, 64, 1])
        return dict(bytes=24 * rows + 4 * used * (O + A + 4) + 28 * (pa + pc), flops=used * (fa + ba + fc + bc))
    if kind == "collect":
        return dict(bytes=68 * case["envs"] + 85 * case["batch"], flops=case["envs"] * _dense([3, 64, 64, 2])[1])
    if kind == "gru":
        I, H, rows = case["inputs"], case["hidden"], case["steps"] * case["batch"]
        p, forward, backward = _dense([H, 64, 4])
        # the GRU keeps its gates and output for the way back; the head's input gradient is wanted as well
        return dict(bytes=4 * rows * (2 * I + 9 * H + 8) + 28 * (p + 3 * H * (I + H + 2)), flops=rows * (12 * I * H + 18 * H * H + forward + backward + 2 * H * 64))
    rows = case["steps"] * case["batch"]
    return _updates(_sequential(_SEQUENCE_ACTOR), _sequential(_SEQUENCE_CRITIC), rows, False, 30)


def tolerance(case):
    """Sums in another order, and parameters and inputs off by one rounding, move the outputs of every kind by 1e-7 to 7e-7 (largest element: 1e-5). Where a relu
    unit's pre-activation lies within that distance of zero, its gate falls the other way and one row's gradient through it comes or goes: seen at batches of 876
    and 57,000, that is 2 / batch of a gradient (largest element: 110 / batch). PPO's gradients jump in the same way where a row's ratio reaches the clip."""
    kind = case["kind"]
    if kind in ("evaluate", "collect", "gru"):
        return {"rel": 3e-6, "max": 1e-4}
    rows = case["minibatch"] if kind == "ppo" else case["batch"] * (case["steps"] if kind == "sac_sequence" else 1)
    return {"rel": min(0.02, 1e-5 + 4 / rows), "max": min(0.5, 1e-4 + 200 / rows)}
