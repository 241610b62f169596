"""The one-launch actor against a float64 eval-mode actor and against the layer-by-layer path."""

import pytest
import torch

from robolearn_amd import kernels as K
from robolearn_amd.config import FlashSACConfig
from robolearn_amd.flashsac import FlashSAC

pytestmark = pytest.mark.gpu


# widths at and off the 16-wide blocks and chunks, the smallest and largest the launch takes; rows at the edges of
# the 16-row workgroups
@pytest.mark.parametrize("obs_dim,action_dim,hidden,blocks", [(1, 1, 4, 0), (4, 1, 128, 1), (17, 6, 20, 3),
                                                              (600, 65, 132, 1), (123, 37, 256, 1), (33, 128, 256, 1)])
@pytest.mark.parametrize("rows", [1, 15, 17, 300])
def test_one_launch_actor_matches_float64(gpu, obs_dim, action_dim, hidden, blocks, rows):
    """2e-6 of the actions' scale: fp32 sums of up to 1024 terms through 2 + 2 blocks layers, each within sqrt(1024)
    2^-24, below a normalization that keeps values near one."""
    print(f"case actor obs={obs_dim} act={action_dim} hidden={hidden} blocks={blocks} rows={rows}", flush=True)
    cfg = FlashSACConfig(seed=3, actor_hidden_dim=hidden, actor_num_blocks=blocks, critic_hidden_dim=32,
                         critic_num_blocks=1, sample_batch_size=16, buffer_max_length=64, buffer_min_length=16)
    agent = FlashSAC(obs_dim, action_dim, num_envs=rows, cfg=cfg)
    g = torch.Generator(device=gpu).manual_seed(rows)
    for name, value in list(agent.actor_running.views.items()) + list(agent.actor_p.items()):
        if name.endswith("running_var"):
            value.copy_(0.5 + torch.rand(value.shape, generator=g, device=gpu))
        elif name.endswith("running_mean") or name.endswith("bias"):
            value.copy_(0.2 * torch.randn(value.shape, generator=g, device=gpu))
    # rows with a pitch, as a slice of wider (asymmetric) observations
    observations = torch.randn(rows, obs_dim + 3, generator=g, device=gpu)
    assert K.actor_act_fits(rows, obs_dim, hidden, blocks, action_dim)
    p = {k: v.double() for k, v in agent.actor_p.items()}
    s = {k: v.double() for k, v in agent.actor_running.views.items()}

    def norm(u, name):
        u = (u - s[name + ".running_mean"]) * torch.rsqrt(s[name + ".running_var"] + 1e-5)
        return u * p[name + ".weight"] + p[name + ".bias"]

    x = norm(observations[:, :obs_dim].double(), "embedder.norm") @ p["embedder.w.w.weight"].t()
    for i in range(blocks):
        r = torch.relu(norm(x @ p[f"encoder.{i}.w1.w.weight"].t(), f"encoder.{i}.norm1"))
        x = x + torch.relu(norm(r @ p[f"encoder.{i}.w2.w.weight"].t(), f"encoder.{i}.norm2"))
    z = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * p["post_norm.weight"]
    mean = z @ p["predictor.mean_w.w.weight"].t() + p["predictor.mean_bias"]
    std = torch.exp(-10 + 6 * (1 + torch.tanh(z @ p["predictor.std_w.w.weight"].t() + p["predictor.std_bias"])))
    for training in (False, True):
        got = agent.act(observations, training=training)
        expected = torch.tanh(mean + (std * agent.exploration_noise.double() if training else 0.0))
        torch.testing.assert_close(got.double(), expected, rtol=0, atol=2e-6 * max(1.0, float(std.max())))
    layered = {}
    fits, K.actor_act_fits = K.actor_act_fits, lambda *sizes: False
    try:
        layered = agent.act(observations, training=False)
    finally:
        K.actor_act_fits = fits
    torch.testing.assert_close(agent.act(observations, training=False), layered, rtol=0, atol=4e-6)


# [rows, columns] observations of every stride that .contiguous() may hand on as it is or has to copy
VIEWS = {
    "packed": lambda x: x,
    "transposed": lambda x: x.t().contiguous().t(),
    "every other row": lambda x: x.repeat_interleave(2, 0)[::2],
    "every other column": lambda x: x.repeat_interleave(2, 1)[:, ::2],
    "one row for all": lambda x: x[:1].expand(x.shape[0], -1),
    "one value for all": lambda x: x[:1, :1].expand(x.shape),
}


@pytest.mark.parametrize("view", VIEWS)
@pytest.mark.parametrize("rows,obs_dim,columns", [(1, 1, 1), (1, 1, 3), (1, 5, 5), (7, 1, 1), (7, 1, 4), (7, 5, 5), (7, 5, 8)])
def test_observation_strides(gpu, rows, obs_dim, columns, view):
    """act() on views of any strides gives what it gives on packed rows, with the same exploration draws."""
    print(f"case actor strides rows={rows} obs={obs_dim} columns={columns} view={view}", flush=True)
    cfg = FlashSACConfig(seed=5, actor_hidden_dim=32, actor_num_blocks=1, critic_hidden_dim=32, critic_num_blocks=1,
                         sample_batch_size=16, buffer_max_length=64, buffer_min_length=16)
    agent, packed = (FlashSAC(obs_dim, 2, num_envs=rows, cfg=cfg) for _ in range(2))
    x = VIEWS[view](torch.randn(rows, columns, generator=torch.Generator(device=gpu).manual_seed(rows), device=gpu))
    same = torch.empty(rows, columns, device=gpu).copy_(x)
    for training in (False, True, True):
        assert torch.equal(agent.act(x, training=training), packed.act(same, training=training))
    assert int(agent.exploration_step) == int(packed.exploration_step)


def test_refused_observations_draw_no_noise(gpu):
    cfg = FlashSACConfig(seed=5, actor_hidden_dim=32, actor_num_blocks=1, critic_hidden_dim=32, critic_num_blocks=1,
                         sample_batch_size=16, buffer_max_length=64, buffer_min_length=16)
    agent = FlashSAC(3, 2, num_envs=4, cfg=cfg)
    for shape in ((4,), (4, 2), (3, 3), (4, 3, 1)):
        with pytest.raises(ValueError):
            agent.act(torch.zeros(shape, device=gpu), training=True)
    assert int(agent.exploration_step) == 0
    # overlapping rows are refused where a copy is not made for the caller
    rows = torch.zeros(1, 3, device=gpu).expand(4, 3)
    with pytest.raises(ValueError):
        K.actor_act(rows, agent._act_parameters, None, torch.empty(4, 2, device=gpu), obs_dim=3, hidden=32, blocks=1,
                    action_dim=2)


# the largest observations, action counts and block counts of the launch, and either side of its two instances
@pytest.mark.parametrize("obs_dim,action_dim,hidden,blocks", [(1024, 80, 256, 0), (1024, 2, 128, 1), (48, 5, 64, 8),
                                                              (512, 64, 128, 1), (513, 64, 128, 1), (9, 3, 129, 2)])
@pytest.mark.parametrize("rows", [1, 33])
def test_one_launch_actor_at_its_limits(gpu, obs_dim, action_dim, hidden, blocks, rows):
    test_one_launch_actor_matches_float64(gpu, obs_dim, action_dim, hidden, blocks, rows)
