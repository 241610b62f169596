"""Performance cases of the learner library: the work its users run, at the sizes they run it.

Twelve named cases and a generator of more over the same ranges.  A case is a dict of plain values whose
"kind" picks one of the entry points below; ``prepare`` builds what a training program holds before the
call (learner, weights, plans, captured graph, inputs), ``run`` makes one pass, ``exact`` repeats it in
64-bit arithmetic with plain torch.
"""

import math
from collections import OrderedDict

import torch

from robolearn_amd import kernels as K
from robolearn_amd.config import FlashSACConfig, PPOConfig
from robolearn_amd.flashsac import FlashSAC, critic_shapes
from robolearn_amd.networks import FlatStore, FusedOptimizer, Trunk
from robolearn_amd.ppo import WarpPPO

DEVICE = "cuda:0"


def listed():
    return [
        # the headline workload: a 29-DoF humanoid recipe, one update-to-data-2 step (an actor-phase update
        # and a critic-only update) replayed as the captured graph the training loop replays
        dict(name="flashsac_update_humanoid", kind="update", obs=123, act=37, batch=8192, actor_hidden=256,
             actor_blocks=2, critic_hidden=1024, critic_blocks=2, bins=101, amp=True),
        # a whole PPO update of the humanoid recipe: 4096 environments x 24 steps, 5 epochs x 4 minibatches
        dict(name="ppo_update_humanoid", kind="ppo_update", envs=4096, horizon=24, obs=123, act=37, layer1=512,
             layer2=256, layer3=128, epochs=5, minibatches=4),
        # forward and backward of the twin critics alone: the largest network, mixed precision
        dict(name="critic_humanoid_bf16", kind="critic", inputs=160, hidden=1024, blocks=2, bins=101, batch=8192,
             bf16=True),
        # the same of the medium recipe in both precisions a user can choose
        dict(name="critic_medium_bf16", kind="critic", inputs=39, hidden=512, blocks=2, bins=101, batch=2048,
             bf16=True),
        dict(name="critic_medium_fp32", kind="critic", inputs=39, hidden=512, blocks=2, bins=101, batch=2048,
             bf16=False),
        # the cart-pole recipe: small layers, launch latency counts
        dict(name="critic_cartpole_fp32", kind="critic", inputs=5, hidden=256, blocks=2, bins=101, batch=512,
             bf16=False),
        # one PPO minibatch through both MLPs, forward and backward
        dict(name="mlp_minibatch_fp32", kind="mlp", rows=24576, inputs=123, outputs=37, layer1=512, layer2=256,
             layer3=128),
        # playing a trained policy on a few environments: the smallest call, all latency
        dict(name="act_cartpole", kind="act", envs=64, obs=4, act=1, hidden=128, blocks=1),
        # one off-policy collection step: exploring actions, then the transition into the replay ring
        dict(name="collect_humanoid", kind="collect", envs=4096, obs=123, act=37, hidden=256, blocks=2),
        # one on-policy collection step: sampled actions and values, then the rollout row
        dict(name="rollout_humanoid", kind="rollout", envs=4096, obs=123, act=37, layer1=512, layer2=256, layer3=128),
        # distributional TD target with the cross-entropy and its gradient, both critics
        dict(name="td_cross_entropy", kind="td", batch=65536, bins=101),
        # Adam + unit-norm projection + target average over a 25-million-parameter network
        dict(name="optimizer_step", kind="optimizer", layers=24, width=1024),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng, low, high):
    """A layer width: usually a multiple of 32, sometimes only of 4."""
    value = _log_int(rng, low, high)
    step = 32 if rng.random() < 0.7 else 4
    return max(low, value // step * step)


def draw(rng):
    kind = rng.choice(("update", "ppo_update", "critic", "critic", "critic", "mlp", "act", "collect", "rollout", "td",
                       "optimizer"))
    if kind == "update":
        return dict(kind=kind, obs=rng.randint(4, 123), act=rng.randint(1, 37), batch=_log_int(rng, 256, 4096),
                    actor_hidden=_width(rng, 64, 256), actor_blocks=rng.randint(1, 2),
                    critic_hidden=_width(rng, 64, 512), critic_blocks=rng.randint(1, 2),
                    bins=rng.choice((51, 101, 151)), amp=rng.random() < 0.5)
    if kind == "ppo_update":
        return dict(kind=kind, envs=4 * _log_int(rng, 16, 1024), horizon=rng.randint(8, 24), obs=rng.randint(4, 123),
                    act=rng.randint(1, 37), layer1=_width(rng, 64, 512), layer2=_width(rng, 64, 256),
                    layer3=_width(rng, 32, 128), epochs=rng.randint(2, 5), minibatches=rng.choice((2, 4)))
    if kind == "critic":
        hidden, blocks = _width(rng, 64, 1024), rng.randint(1, 2)
        return dict(kind=kind, inputs=rng.randint(5, 160), hidden=hidden, blocks=blocks,
                    bins=rng.choice((21, 51, 101, 151)), batch=_log_int(rng, 128, 8192), bf16=rng.random() < 0.6)
    if kind == "mlp":
        return dict(kind=kind, rows=_log_int(rng, 512, 24576), inputs=rng.randint(4, 123), outputs=rng.randint(1, 37),
                    layer1=_width(rng, 64, 512), layer2=_width(rng, 64, 256), layer3=_width(rng, 32, 128))
    if kind == "act":
        return dict(kind=kind, envs=_log_int(rng, 1, 4096), obs=rng.randint(4, 123), act=rng.randint(1, 37),
                    hidden=_width(rng, 64, 256), blocks=rng.randint(1, 2))
    if kind == "collect":
        return dict(kind=kind, envs=_log_int(rng, 16, 4096), obs=rng.randint(4, 123), act=rng.randint(1, 37),
                    hidden=_width(rng, 64, 256), blocks=rng.randint(1, 2))
    if kind == "rollout":
        return dict(kind=kind, envs=_log_int(rng, 16, 4096), obs=rng.randint(4, 123), act=rng.randint(1, 37),
                    layer1=_width(rng, 64, 512), layer2=_width(rng, 64, 256), layer3=_width(rng, 32, 128))
    if kind == "td":
        return dict(kind=kind, batch=_log_int(rng, 256, 65536), bins=rng.randint(21, 151))
    return dict(kind=kind, layers=rng.randint(2, 24), width=_width(rng, 64, 1024))


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


# ---------------------------------------------------------------------------
# whole FlashSAC update
# ---------------------------------------------------------------------------
UPDATE_REPLAY = 65536
GAMMA = 0.99


def _update_prepare(case, seed):
    cfg = FlashSACConfig(seed=seed, normalize_reward=False, n_step=1, sample_batch_size=case["batch"],
                         buffer_max_length=UPDATE_REPLAY, buffer_min_length=case["batch"],
                         actor_hidden_dim=case["actor_hidden"], actor_num_blocks=case["actor_blocks"],
                         critic_hidden_dim=case["critic_hidden"], critic_num_blocks=case["critic_blocks"],
                         critic_num_bins=case["bins"], critic_min_v=-20.0, critic_max_v=20.0,
                         critic_target_update_tau=0.005, learning_rate_end=3e-4, gamma=GAMMA, use_amp=case["amp"])
    agent = FlashSAC(case["obs"], case["act"], num_envs=1, cfg=cfg)
    g = _generator(seed)
    n, o, a = UPDATE_REPLAY, case["obs"], case["act"]
    agent.load_replay({
        "observation": torch.randn(n, o, generator=g, device=DEVICE),
        "next_observation": torch.randn(n, o, generator=g, device=DEVICE),
        "action": torch.rand(n, a, generator=g, device=DEVICE) * 2 - 1,
        "reward": torch.randn(n, generator=g, device=DEVICE) * 0.5,
        "terminated": (torch.rand(n, generator=g, device=DEVICE) < 0.005).float(),
        "truncated": torch.zeros(n, device=DEVICE),
        "discount": torch.full((n,), GAMMA, device=DEVICE),
    })
    agent.capture_pair()
    return agent


def _update_run(agent):
    agent.update_pair(tensor_metrics=True)
    return {"parameters": agent.parameters(), "target": list(agent.critic.targets().values()),
            "metrics": agent.metrics_buffer}


def _network_flops(rows, inputs, hidden, blocks, members):
    return 2.0 * members * rows * (inputs * hidden + blocks * 8 * hidden * hidden)


def _update_work(case):
    B, O, A, ha, hc = case["batch"], case["obs"], case["act"], case["actor_hidden"], case["critic_hidden"]
    I, bins = O + A, case["bins"]

    def actor(rows):
        return _network_flops(rows, O, ha, case["actor_blocks"], 1) + 4.0 * rows * ha * A

    def critic(rows, head_rows):
        return _network_flops(rows, I, hc, case["critic_blocks"], 2) + 4.0 * head_rows * hc * bins

    critic_phase = actor(B) + critic(2 * B, B) + 3 * critic(2 * B, B)
    actor_phase = 3 * actor(2 * B) + 2 * critic(B, B)
    actor_parameters = O * ha + case["actor_blocks"] * 8 * ha * ha + 2 * ha * A
    critic_parameters = 2 * (I * hc + case["critic_blocks"] * 8 * hc * hc + hc * bins)
    state = 24 * actor_parameters + 2 * 32 * critic_parameters  # weights, both moments and the target, in and out
    batch = 2 * 4 * B * (2 * O + A + 4)
    return dict(bytes=float(state + batch), flops=actor_phase + 2 * critic_phase)


# ---------------------------------------------------------------------------
# PPO: whole update and rollout step
# ---------------------------------------------------------------------------
def _ppo(case, seed, horizon=1, epochs=1, minibatches=1):
    cfg = PPOConfig(hidden_dims=(case["layer1"], case["layer2"], case["layer3"]), activation="elu", std_type="log",
                    epochs=epochs, num_mini_batches=minibatches, clip_ratio=0.2, clip_value=True,
                    entropy_coefficient=0.005, schedule="adaptive", desired_kl=0.01, seed=seed)
    return WarpPPO(case["obs"], case["act"], case["envs"], horizon, cfg, device=DEVICE)


def _ppo_update_prepare(case, seed):
    ppo = _ppo(case, seed, case["horizon"], case["epochs"], case["minibatches"])
    g = _generator(seed)
    n = case["envs"]
    zeros = torch.zeros(n, dtype=torch.int32, device=DEVICE)
    obs = torch.randn(n, case["obs"], generator=g, device=DEVICE)
    for step in range(case["horizon"]):
        ppo.act(obs)
        following = torch.randn(n, case["obs"], generator=g, device=DEVICE)
        rewards = torch.randn(n, generator=g, device=DEVICE)
        done = (torch.rand(n, generator=g, device=DEVICE) < 1e-3).int()
        ppo.store(step, obs, rewards, done, zeros, following)
        obs = following
    # the graph of the update is captured by the first call; the learner then starts from its initial state
    state = ppo.state_dict()
    ppo.update()
    ppo.load_state_dict(state)
    return ppo


def _ppo_update_run(ppo):
    ppo.update()
    return {"parameters": list(ppo.parameters), "metrics": ppo.metrics, "advantages": ppo.advantages,
            "returns": ppo.returns}


def _mlp_flops(rows, inputs, outputs, case):
    widths = (inputs, case["layer1"], case["layer2"], case["layer3"], outputs)
    return 2.0 * rows * sum(a * b for a, b in zip(widths[:-1], widths[1:]))


def _mlp_parameters(inputs, outputs, case):
    widths = (inputs, case["layer1"], case["layer2"], case["layer3"], outputs)
    return sum((a + 1) * b for a, b in zip(widths[:-1], widths[1:]))


def _ppo_update_work(case):
    rows = case["envs"] * case["horizon"]
    each = 0.0
    for outputs in (case["act"], 1):
        # the first layer needs no input gradient
        each += 3 * _mlp_flops(rows, case["obs"], outputs, case) - 2.0 * rows * case["obs"] * case["layer1"]
    parameters = sum(_mlp_parameters(case["obs"], outputs, case) for outputs in (case["act"], 1))
    rollout = 4 * rows * (case["obs"] + 3 * case["act"] + 6)
    steps = case["epochs"] * case["minibatches"]
    return dict(bytes=float(case["epochs"] * rollout + 24 * steps * parameters), flops=each * case["epochs"])


def _rollout_prepare(case, seed):
    ppo = _ppo(case, seed)
    g = _generator(seed)
    n = case["envs"]
    return dict(ppo=ppo, obs=torch.randn(n, case["obs"], generator=g, device=DEVICE),
                following=torch.randn(n, case["obs"], generator=g, device=DEVICE),
                rewards=torch.randn(n, generator=g, device=DEVICE),
                terminated=(torch.rand(n, generator=g, device=DEVICE) < 0.01).int(),
                truncated=torch.zeros(n, dtype=torch.int32, device=DEVICE))


def _rollout_run(state):
    ppo = state["ppo"]
    actions = ppo.act(state["obs"])
    ppo.store(0, state["obs"], state["rewards"], state["terminated"], state["truncated"], state["following"])
    return {"actions": actions, "means": ppo.means, "stds": ppo.stds, "values": ppo.values,
            "next_values": ppo.next_values, "log_probs": ppo.log_probs, "rewards": ppo.rewards,
            "observations": ppo.observations}


def _rollout_exact(case, seed):
    state = _rollout_prepare(case, seed)
    weights = [p.double() for p in state["ppo"].parameters]

    def mlp(x, first):
        for i in range(4):
            x = x @ weights[first + 2 * i].t() + weights[first + 2 * i + 1]
            if i < 3:
                x = torch.where(x > 0, x, torch.expm1(x))
        return x

    obs, following = state["obs"].double(), state["following"].double()
    # the sampled actions and their log-probabilities hold the learner's own random draws
    return {"actions": None, "means": mlp(obs, 0), "stds": torch.exp(weights[16]).expand(case["envs"], -1),
            "values": mlp(obs, 8)[:, 0], "next_values": mlp(following, 8)[:, 0], "log_probs": None,
            "rewards": state["rewards"].double(), "observations": obs}


def _rollout_work(case):
    n, o, a = case["envs"], case["obs"], case["act"]
    flops = _mlp_flops(n, o, a, case) + 2 * _mlp_flops(n, o, 1, case)
    parameters = _mlp_parameters(o, a, case) + _mlp_parameters(o, 1, case)
    return dict(bytes=4.0 * (n * (3 * o + 4 * a + 12) + parameters), flops=flops)


# ---------------------------------------------------------------------------
# twin critics: training forward and backward as one captured graph
# ---------------------------------------------------------------------------
def _critic_inputs(case, seed):
    g = _generator(seed)
    I, h, bins, B = case["inputs"], case["hidden"], case["bins"], case["batch"]
    weights = OrderedDict()
    for name, shape in critic_shapes(I, h, case["blocks"], bins).items():
        value = torch.randn(shape, generator=g, device=DEVICE)
        if ".norm" in name or name.startswith("post_norm"):
            value = 1.0 + 0.1 * value if name.endswith("weight") else 0.1 * value
        elif name.endswith("bias"):
            value = 0.1 * value
        else:
            value = value / value.norm(dim=-1, keepdim=True)  # unit rows, as the projection keeps them
        weights[name] = value
    x = torch.randn(2 * B, I, generator=g, device=DEVICE) * (0.5 + torch.rand(I, generator=g, device=DEVICE))
    # the gradient a cross-entropy against a narrow target hands the logits
    target = torch.softmax(3.0 * torch.randn(2, B, bins, generator=g, device=DEVICE), -1)
    dlogits = (torch.softmax(torch.randn(2, B, bins, generator=g, device=DEVICE), -1) - target) / (2 * B)
    return weights, x, dlogits


class _Critic:
    def __init__(self, case, seed):
        I, h, bins, B = case["inputs"], case["hidden"], case["bins"], case["batch"]
        bf16 = case["bf16"]
        self.batch, self.rows, self.hidden, self.bins = B, 2 * B, h, bins
        self.mode = K.BF16 if bf16 else K.FP32_SPLIT
        weights, self.x, self.dlogits = _critic_inputs(case, seed)
        self.dlogits_op = self.dlogits.to(torch.bfloat16) if bf16 else self.dlogits
        self.store = FlatStore(critic_shapes(I, h, case["blocks"], bins), DEVICE, adam=False, shadows=bf16)
        self.p, self.g = self.store.params(), self.store.grads()
        for name, value in weights.items():
            self.p[name].copy_(value)
        self.store.enable_transposed([f"encoder.{i}.w{j}.weight" for i in range(case["blocks"]) for j in (1, 2)])
        self.store.refresh_shadows()
        self.w = self.store.shadows() or self.p
        self.net = Trunk(ensemble=2, in_dim=I, hidden=h, blocks=case["blocks"], max_rows=2 * B, device=DEVICE,
                         mode=self.mode, prefix_linear=".weight")
        self.workspace = torch.empty(256 << 20, dtype=torch.uint8, device=DEVICE)
        self.net.workspace = self.workspace
        self.running = {}
        for name, width in self.net.bn_layers():
            self.running[name + ".running_mean"] = torch.zeros(2, width, device=DEVICE)
            self.running[name + ".running_var"] = torch.ones(2, width, device=DEVICE)
        self.logits = torch.zeros(2, B, bins, device=DEVICE)
        self.partial = torch.zeros(2 * K.chunks(B) * bins, device=DEVICE)
        self.step()
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.step()
        for name, value in self.running.items():
            value.fill_(1.0 if name.endswith("var") else 0.0)

    def step(self):
        net, p, w, g, mode, ws = self.net, self.p, self.w, self.g, self.mode, self.workspace
        B, R, h, bins = self.batch, self.rows, self.hidden, self.bins
        net.forward(p, w, self.running, self.x, rows=R, x_stride=0, training=True)
        net.post_norm(p, rows=R, row0=0, count=B)
        K.linear_forward(net.z_op, w["predictor.w.weight"], self.logits, rows=B, in_dim=h, out_dim=bins, ensemble=2,
                         x_stride=R * h, bias=p["predictor.bias"], mode=mode, workspace=ws)
        K.linear_backward_weight(self.dlogits_op, net.z_op, g["predictor.w.weight"], rows=B, in_dim=h, out_dim=bins,
                                 ensemble=2, x_stride=R * h, mode=mode, workspace=ws)
        K.bias_grad(self.dlogits, g["predictor.bias"], self.partial, rows=B, channels=bins, ensemble=2)
        K.gemm(self.dlogits_op, w["predictor.w.weight"], net.dz, m=B, n=h, k=bins, batch=2, a_kcontig=True,
               b_kcontig=False, lda=bins, ldb=h, ldd=h, stride_a=B * bins, stride_b=bins * h, stride_d=R * h, mode=mode)
        net.post_norm_backward(p, g, rows=R, row0=0, count=B)
        net.backward(p, w, self.running, g, self.x, rows=R, x_stride=0, training=True, wt=self.store.transposed,
                     workspace=ws)


def _critic_run(critic):
    critic.graph.replay()
    return {"logits": critic.logits, "grads": critic.g, "running": critic.running}


def _critic_exact(case, seed):
    """The forward's results and the head's gradients.  The gradients below the head have no 64-bit value to
    be near: a ReLU input within rounding of zero passes on one side and is blocked on the other, and one
    such decision changes its row's gradient by more than all rounding together (5e-7 or 4e-3 of a tensor in
    fp32, by which decisions fall; 0.1 in bf16)."""
    weights, x, dlogits = _critic_inputs(case, seed)
    B, members = case["batch"], []
    for e in range(2):
        w = {name: value[e].double() for name, value in weights.items()}
        running = {}

        def norm(u, name):
            mean, var = u.mean(0), u.var(0, unbiased=False)
            running[name + ".running_mean"] = 0.01 * mean
            running[name + ".running_var"] = 0.99 + 0.01 * var * (u.shape[0] / (u.shape[0] - 1))
            return (u - mean) * torch.rsqrt(var + 1e-5) * w[name + ".weight"] + w[name + ".bias"]

        stream = norm(x.double(), "embedder.norm") @ w["embedder.w.weight"].t()
        for i in range(case["blocks"]):
            pre = f"encoder.{i}"
            r = torch.relu(norm(stream @ w[pre + ".w1.weight"].t(), pre + ".norm1"))
            stream = stream + torch.relu(norm(r @ w[pre + ".w2.weight"].t(), pre + ".norm2"))
        unit = stream[:B] * torch.rsqrt((stream[:B] ** 2).mean(-1, keepdim=True) + 1e-6)
        z = unit * w["post_norm.weight"]
        d = dlogits[e].double()
        grads = {"predictor.w.weight": d.t() @ z, "predictor.bias": d.sum(0),
                 "post_norm.weight": ((d @ w["predictor.w.weight"]) * unit).sum(0)}
        members.append((z @ w["predictor.w.weight"].t() + w["predictor.bias"], grads, running))
    stack = lambda i: {k: torch.stack([m[i][k] for m in members]) for k in members[0][i]}  # noqa: E731
    return {"logits": torch.stack([m[0] for m in members]), "grads": {**dict.fromkeys(weights), **stack(1)},
            "running": stack(2)}


def _critic_work(case):
    B, I, h, bins, blocks = case["batch"], case["inputs"], case["hidden"], case["bins"], case["blocks"]
    flops = 3 * (_network_flops(2 * B, I, h, blocks, 2) + 4.0 * B * h * bins)
    parameters = 2 * (I * h + blocks * 8 * h * h + h * bins)
    weight = 2 if case["bf16"] else 4
    return dict(bytes=float((weight + 4) * parameters + 4 * 2 * B * I + 2 * 2 * 4 * B * bins), flops=flops)


# ---------------------------------------------------------------------------
# stacked actor and critic MLPs of one PPO minibatch, forward and backward, captured
# ---------------------------------------------------------------------------
def _mlp_inputs(case, seed):
    g = _generator(seed)
    widths = (case["inputs"], case["layer1"], case["layer2"], case["layer3"], case["outputs"])
    weights, biases = [], []
    for a, b in zip(widths[:-1], widths[1:]):
        bound = 1.0 / math.sqrt(a)
        weights.append((torch.rand(2, b, a, generator=g, device=DEVICE) * 2 - 1) * bound)
        biases.append((torch.rand(2, b, generator=g, device=DEVICE) * 2 - 1) * bound)
    pitch = (case["inputs"] + 3) // 4 * 4  # rows of the gathered minibatch start 16-byte aligned
    x = torch.zeros(case["rows"], pitch, device=DEVICE)
    x[:, : case["inputs"]] = torch.randn(case["rows"], case["inputs"], generator=g, device=DEVICE)
    dout = torch.randn(2, case["rows"], case["outputs"], generator=g, device=DEVICE) / case["rows"]
    return widths, weights, biases, x, dout


class _Mlp:
    def __init__(self, case, seed):
        self.rows = R = case["rows"]
        self.widths, self.weights, self.biases, self.x, self.dout = _mlp_inputs(case, seed)
        z = lambda *s: torch.zeros(*s, device=DEVICE)  # noqa: E731
        self.hidden = [z(2, R, w) for w in self.widths[1:]]
        self.dhidden = [z(2, R, w) for w in self.widths[1:-1]]
        self.dw = [torch.zeros_like(w) for w in self.weights]
        self.db = [torch.zeros_like(b) for b in self.biases]
        self.workspace = torch.empty(64 << 20, dtype=torch.uint8, device=DEVICE)
        self.step()
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.step()

    def step(self):
        R, last, mode = self.rows, len(self.weights) - 1, K.FP32_SPLIT
        pitch = self.x.shape[1]
        inputs = [self.x] + self.hidden[:-1]
        for i, (w, b) in enumerate(zip(self.weights, self.biases)):
            K.linear_forward(inputs[i], w, self.hidden[i], rows=R, in_dim=self.widths[i], out_dim=self.widths[i + 1],
                             ensemble=2, x_stride=0 if i == 0 else None, bias=b, mode=mode,
                             epilogue="elu" if i < last else None, x_ld=pitch if i == 0 else None)
        d = self.dout
        for i in reversed(range(last + 1)):
            K.linear_backward_weight(d, inputs[i], self.dw[i], rows=R, in_dim=self.widths[i],
                                     out_dim=self.widths[i + 1], ensemble=2, x_stride=0 if i == 0 else None, mode=mode,
                                     workspace=self.workspace, x_ld=pitch if i == 0 else None, bias_grad=self.db[i])
            if i > 0:
                K.linear_backward_input(d, self.weights[i], self.dhidden[i - 1], rows=R, in_dim=self.widths[i],
                                        out_dim=self.widths[i + 1], ensemble=2, mode=mode, c=self.hidden[i - 1],
                                        epilogue="elu_grad")
                d = self.dhidden[i - 1]


def _mlp_run(mlp):
    mlp.graph.replay()
    return {"out": mlp.hidden[-1], "weights": mlp.dw, "biases": mlp.db}


def _mlp_exact(case, seed):
    _, weights, biases, x, dout = _mlp_inputs(case, seed)
    out, dws, dbs = [], [], []
    for e in range(2):
        leaves = [t[e].double().requires_grad_() for pair in zip(weights, biases) for t in pair]
        y = x[:, : case["inputs"]].double()
        for i in range(4):
            y = y @ leaves[2 * i].t() + leaves[2 * i + 1]
            if i < 3:
                y = torch.where(y > 0, y, torch.expm1(y.clamp(max=0.0)))
        grads = torch.autograd.grad(y, leaves, dout[e].double())
        out.append(y.detach())
        dws.append(grads[0::2])
        dbs.append(grads[1::2])
    return {"out": torch.stack(out), "weights": [torch.stack(p) for p in zip(*dws)],
            "biases": [torch.stack(p) for p in zip(*dbs)]}


def _mlp_work(case):
    R, I, A = case["rows"], case["inputs"], case["outputs"]
    flops = 2 * (3 * _mlp_flops(R, I, A, case) - 2.0 * R * I * case["layer1"])
    return dict(bytes=4.0 * (R * I + 4 * R * A + 4 * _mlp_parameters(I, A, case)), flops=flops)


# ---------------------------------------------------------------------------
# FlashSAC acting and collecting
# ---------------------------------------------------------------------------
COLLECT_STEPS = 3  # n-step window of the collection cases
COLLECT_ROWS = 16384


def _actor_agent(case, seed):
    cfg = FlashSACConfig(seed=seed, actor_hidden_dim=case["hidden"], actor_num_blocks=case["blocks"],
                         critic_hidden_dim=32, critic_num_blocks=1, sample_batch_size=256,
                         buffer_max_length=COLLECT_ROWS, buffer_min_length=256, n_step=COLLECT_STEPS, gamma=GAMMA)
    agent = FlashSAC(case["obs"], case["act"], num_envs=case["envs"], cfg=cfg)
    # statistics and biases of a policy that has trained for a while
    g = _generator(seed)
    for name, value in agent.actor_running.views.items():
        noise = torch.randn(value.shape, generator=g, device=DEVICE)
        value.copy_(0.2 * noise if name.endswith("mean") else 0.5 + torch.rand(value.shape, generator=g, device=DEVICE))
    for name, value in agent.actor.params().items():
        if name.endswith("bias"):
            value.copy_(0.1 * torch.randn(value.shape, generator=g, device=DEVICE))
    agent.actor.refresh_shadows()
    return agent, g


def _act_prepare(case, seed):
    agent, g = _actor_agent(case, seed)
    return agent, torch.randn(case["envs"], case["obs"], generator=g, device=DEVICE)


def _act_run(state):
    agent, observations = state
    return agent.act(observations, training=False)


def _act_exact(case, seed):
    agent, observations = _act_prepare(case, seed)
    p = {k: v.double() for k, v in agent.actor.params().items()}
    s = {k: v.double() for k, v in agent.actor_running.views.items()}

    def norm(u, name):
        u = (u - s[name + ".running_mean"]) * torch.rsqrt(s[name + ".running_var"] + 1e-5)
        return u * p[name + ".weight"] + p[name + ".bias"]

    x = norm(observations.double(), "embedder.norm") @ p["embedder.w.w.weight"].t()
    for i in range(case["blocks"]):
        pre = f"encoder.{i}"
        r = torch.relu(norm(x @ p[pre + ".w1.w.weight"].t(), pre + ".norm1"))
        x = x + torch.relu(norm(r @ p[pre + ".w2.w.weight"].t(), pre + ".norm2"))
    z = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * p["post_norm.weight"]
    return torch.tanh(z @ p["predictor.mean_w.w.weight"].t() + p["predictor.mean_bias"])


def _actor_work(case):
    n, o, a, h = case["envs"], case["obs"], case["act"], case["hidden"]
    flops = _network_flops(n, o, h, case["blocks"], 1) + 4.0 * n * h * a
    parameters = o * h + case["blocks"] * 8 * h * h + 2 * h * a
    return dict(bytes=4.0 * (n * (o + a) + parameters), flops=flops)


def _transitions(case, g):
    n = case["envs"]
    return dict(action=torch.rand(n, case["act"], generator=g, device=DEVICE) * 2 - 1,
                reward=torch.randn(n, generator=g, device=DEVICE),
                terminated=(torch.rand(n, generator=g, device=DEVICE) < 0.02).float(),
                truncated=(torch.rand(n, generator=g, device=DEVICE) < 0.02).float(),
                observation=torch.randn(n, case["obs"], generator=g, device=DEVICE),
                next_observation=torch.randn(n, case["obs"], generator=g, device=DEVICE))


def _collect_prepare(case, seed):
    agent, g = _actor_agent(case, seed)
    steps = [_transitions(case, g) for _ in range(COLLECT_STEPS)]
    for t in steps[:-1]:  # the window is full but for the step of the pass
        agent.process_transition(t)
    return dict(agent=agent, step=steps[-1], steps=steps)


def _collect_run(state):
    agent, t = state["agent"], state["step"]
    actions = agent.act(t["observation"], training=True)
    agent.observe(t["observation"], t["action"], t["reward"], t["terminated"], t["truncated"], t["next_observation"])
    return {"actions": actions, "reward": agent.replay["reward"], "discount": agent.replay["discount"],
            "observation": agent.replay["observation"], "next_observation": agent.replay["next_observation"],
            "returns": agent.reward_returns}


def _collect_exact(case, seed):
    steps = _collect_prepare(case, seed)["steps"]
    n = case["envs"]
    last = steps[-1]
    reward, following = last["reward"].double(), last["next_observation"].double()
    discount = torch.full((n,), GAMMA, dtype=torch.float64, device=DEVICE)
    for t in reversed(steps[:-1]):
        done = (t["terminated"] != 0) | (t["truncated"] != 0)
        reward = t["reward"].double() + torch.where(done, 0.0, GAMMA * reward)
        discount = torch.where(done, GAMMA, GAMMA * discount)
        following = torch.where(done[:, None], t["next_observation"].double(), following)
    returns = torch.zeros(n, dtype=torch.float64, device=DEVICE)
    for t in steps:
        done = (t["terminated"] != 0) | (t["truncated"] != 0)
        returns = t["reward"].double() + torch.where(done, 0.0, GAMMA * returns)

    def ring(value):
        full = torch.zeros((COLLECT_ROWS,) + tuple(value.shape[1:]), dtype=torch.float64, device=DEVICE)
        full[:n] = value
        return full

    # the exploring actions hold the learner's own random draws
    return {"actions": None, "reward": ring(reward), "discount": ring(discount),
            "observation": ring(steps[0]["observation"].double()), "next_observation": ring(following),
            "returns": returns}


def _collect_work(case):
    n, row = case["envs"], 2 * case["obs"] + case["act"]
    work = _actor_work(case)
    # the step in, its staged copy, the oldest staged step in and its committed row
    work["bytes"] += 4.0 * n * (4 * row + 3 * COLLECT_STEPS + 7)
    return work


# ---------------------------------------------------------------------------
# distributional TD target and cross-entropy
# ---------------------------------------------------------------------------
V_MIN, V_MAX = -10.0, 10.0


def _td_prepare(case, seed):
    g = _generator(seed)
    B, bins = case["batch"], case["bins"]
    s = dict(case=case, scale=1.0 / (2 * B))
    s["target_logits"] = torch.randn(2, B, bins, generator=g, device=DEVICE)
    s["logits"] = torch.randn(2, B, bins, generator=g, device=DEVICE)
    s["support"] = torch.linspace(V_MIN, V_MAX, bins, dtype=torch.float32).to(DEVICE)
    s["reward"] = torch.randn(B, generator=g, device=DEVICE)
    s["terminated"] = (torch.rand(B, generator=g, device=DEVICE) < 0.01).float()
    s["discount"] = torch.full((B,), GAMMA, device=DEVICE)
    s["next_log_probs"] = torch.randn(B, generator=g, device=DEVICE) * 5.0
    s["alpha"] = torch.full((1,), 0.01, device=DEVICE)
    s["dlogits"] = torch.empty(2, B, bins, device=DEVICE)
    s["loss_rows"] = torch.empty(2, B, device=DEVICE)
    s["entropy_rows"] = torch.empty(B, device=DEVICE)
    s["q_next"] = torch.empty(2, B, device=DEVICE)
    return s


def _td_run(s):
    B, bins = s["case"]["batch"], s["case"]["bins"]
    K.td_cross_entropy(s["target_logits"], None, B, s["logits"], None, B, s["support"], s["reward"], s["terminated"],
                       s["discount"], s["next_log_probs"], s["alpha"], min_v=V_MIN, max_v=V_MAX, batch=B, bins=bins,
                       scale=s["scale"], dlogits=s["dlogits"], loss_rows=s["loss_rows"],
                       entropy_rows=s["entropy_rows"], q_next=s["q_next"])
    return {k: s[k] for k in ("dlogits", "loss_rows", "entropy_rows", "q_next")}


def _td_exact(case, seed):
    s = {k: v.double() if torch.is_tensor(v) else v for k, v in _td_prepare(case, seed).items()}
    bins = case["bins"]
    log_p = torch.log_softmax(s["target_logits"], -1)
    q = (log_p.exp() * s["support"]).sum(-1)
    probs = torch.where((q[1] < q[0])[:, None], log_p[1], log_p[0]).exp()
    entropy = s["alpha"] * s["next_log_probs"]
    values = s["reward"][:, None] + (s["discount"] * (1 - s["terminated"]))[:, None] * (s["support"] - entropy[:, None])
    b = (values.clamp(V_MIN, V_MAX) - V_MIN) / ((V_MAX - V_MIN) / (bins - 1))
    lower = b.floor().long()
    frac = b - lower
    target = torch.zeros_like(probs).scatter_add_(1, lower, probs * (1 - frac))
    target.scatter_add_(1, (lower + 1).clamp(max=bins - 1), probs * frac)
    lp = torch.log_softmax(s["logits"], -1)
    return {"dlogits": s["scale"] * (lp.exp() * target.sum(-1, keepdim=True) - target),
            "loss_rows": -(target * lp).sum(-1), "entropy_rows": entropy, "q_next": q}


def _td_work(case):
    B, bins = case["batch"], case["bins"]
    return dict(bytes=4.0 * B * (6 * bins + 9), flops=60.0 * B * bins)


# ---------------------------------------------------------------------------
# optimizer step
# ---------------------------------------------------------------------------
TAU, RATE = 0.005, 3e-4


def _optimizer_shapes(case):
    shapes = OrderedDict()
    for i in range(case["layers"]):
        w = case["width"]
        out, inp = ((w, w), (4 * w, w // 4))[i % 2]
        shapes[f"layer{i}.weight"], shapes[f"layer{i}.bias"] = (out, inp), (out,)
    return shapes


class _Optimizer:
    def __init__(self, case, seed):
        g = _generator(seed)
        shapes = _optimizer_shapes(case)
        kinds = {n: 0 if n.endswith("weight") else 3 for n in shapes}  # unit rows; plain biases
        self.store = s = FlatStore(shapes, DEVICE, target=True)
        for name, view in s.params().items():
            value = torch.randn(view.shape, generator=g, device=DEVICE)
            view.copy_(value / value.norm(dim=-1, keepdim=True) if kinds[name] == 0 else 0.05 * value)
        noise = torch.randn(s.param.shape, generator=g, device=DEVICE)
        s.target.copy_(s.param + 0.01 * s.param * noise)
        s.grad.normal_(0.0, 1e-3, generator=g)
        s.m1.normal_(0.0, 1e-4, generator=g)
        s.m2.copy_(s.m1 * s.m1 + 1e-8)
        cfg = FlashSACConfig(learning_rate_init=RATE, learning_rate_peak=RATE, learning_rate_end=RATE)
        self.optimizer = FusedOptimizer(s, cfg, ema_tau=TAU, kinds=kinds)
        self.optimizer.timestep.fill_(100.0)


def _optimizer_run(state):
    state.optimizer.step()
    s = state.store
    return {"param": s.param, "target": s.target, "m1": s.m1, "m2": s.m2}


def _optimizer_exact(case, seed):
    s = _Optimizer(case, seed).store
    grad = s.grad.double()
    out = {"param": s.param.double(), "target": s.target.double(), "m1": s.m1.double(), "m2": s.m2.double()}
    for name in s.shapes:
        p, t, m1, m2, g = (s.view(b, name) for b in (out["param"], out["target"], out["m1"], out["m2"], grad))
        m1.mul_(0.9).add_(0.1 * g)
        m2.mul_(0.999).add_(0.001 * g * g)
        step = 101
        p.sub_(RATE / (1 - 0.9**step) * m1 / ((m2 / (1 - 0.999**step)).sqrt() + 1e-8))
        if name.endswith("weight"):
            p.div_(p.norm(dim=-1, keepdim=True).clamp_min(1e-8))
        t.mul_(1 - TAU).add_(TAU * p)
    return out


def _optimizer_work(case):
    count = sum(math.prod(shape) for shape in _optimizer_shapes(case).values())
    return dict(bytes=36.0 * count, flops=20.0 * count)


# ---------------------------------------------------------------------------
_KINDS = {
    "update": (_update_prepare, _update_run, None, _update_work),
    "ppo_update": (_ppo_update_prepare, _ppo_update_run, None, _ppo_update_work),
    "critic": (_Critic, _critic_run, _critic_exact, _critic_work),
    "mlp": (_Mlp, _mlp_run, _mlp_exact, _mlp_work),
    "act": (_act_prepare, _act_run, _act_exact, _actor_work),
    "collect": (_collect_prepare, _collect_run, _collect_exact, _collect_work),
    "rollout": (_rollout_prepare, _rollout_run, _rollout_exact, _rollout_work),
    "td": (_td_prepare, _td_run, _td_exact, _td_work),
    "optimizer": (_Optimizer, _optimizer_run, _optimizer_exact, _optimizer_work),
}


def prepare(case, seed):
    kind = case["kind"]
    return kind, _KINDS[kind][0](case, seed)


def run(state):
    kind, held = state
    return _KINDS[kind][1](held)


def work(case):
    return _KINDS[case["kind"]][3](case)


def exact(case, seed):
    """None for whole updates: their second step starts from Adam's first, which maps a gradient within
    rounding of zero to a change of a whole learning rate."""
    function = _KINDS[case["kind"]][2]
    return None if function is None else function(case, seed)


# About four times what separates two correct implementations of the same precision, measured between the
# fp32 matrix instruction and the three-piece bf16 products, between row orders of the batch, and between
# numbers of K splits.  In whole networks a rounding decides which ReLU inputs near zero pass, and in whole
# updates the sign of Adam's first steps; in bf16 the rounding midpoints add to it.
_TOLERANCES = {
    "mlp": {"rel": 1e-5, "max": 5e-5},
    "act": {"rel": 5e-6, "max": 5e-5},
    "collect": {"rel": 5e-6, "max": 5e-5},
    "rollout": {"rel": 5e-6, "max": 5e-5},
    "td": {"rel": 1.5e-5, "max": 1e-3},
    "optimizer": {"rel": 2e-7, "max": 1e-6},
    "ppo_update": {"rel": 0.03, "max": 0.1},
}


def tolerance(case):
    if case["kind"] == "update":
        return {"rel": 0.025, "max": 0.99} if case["amp"] else {"rel": 2e-3, "max": 0.1}
    if case["kind"] == "critic":
        return {"rel": 0.03, "max": 0.99} if case["bf16"] else {"rel": 0.016, "max": 0.99}
    return _TOLERANCES[case["kind"]]
