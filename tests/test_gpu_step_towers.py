"""The rollout step's joined launches (ppo_step_towers_f32,
ppo_head_sample_categorical_f32, ppo_gru_fwd_step_x_f32) against the oracle's
forward and draw and against the layer-by-layer launches, over the networks they
accept and at the edges of their tiles.

Tolerances as in test_gpu_step.py: values and log-probabilities 1e-5 relative
(atol 1e-5), categorical actions exact where the oracle's margin exceeds 1e-4,
Gaussian actions 1e-5 of |sigma eps| + |mean| (the draw) plus 1e-5 (the mean's
forward in float32).
"""
import numpy as np
import pytest
import torch

from boonta_amd import networks as nn, recipes
from boonta_amd.algorithms.ppo import PPO, flat_state_of
from boonta_amd.random import key as make_key
from boonta_amd.algorithms.recurrent_ppo import RecurrentPPO
from boonta_amd.rollout import RecurrentStepExecutor, StepExecutor
from boonta_amd.types import Timestep
from oracle import nets, sample
from test_gpu_step import check_categorical, dev, key_dev, stream

pytestmark = pytest.mark.gpu

CASES = [
    # rows, obs, row padding, width, depth, LayerNorm, activation, distribution, outputs, temperature
    (1, 3, 0, 64, 1, False, "tanh", "categorical", 2, 1.0),
    (15, 4, 0, 64, 2, False, "tanh", "categorical", 16, 0.0),
    (17, 5, 3, 64, 8, False, "relu", "gaussian", 1, 1.0),
    (16, 16, 0, 128, 2, False, "relu", "gaussian", 16, 0.5),
    (300, 65, 1, 128, 3, False, "tanh", "categorical", 7, 0.7),
    (300, 87, 0, 256, 2, False, "tanh", "gaussian", 8, 1.0),
    (33, 600, 0, 256, 1, False, None, "categorical", 3, 1.0),
    (4096, 87, 0, 256, 4, True, "silu", "gaussian", 8, 1.0),
    (31, 64, 0, 256, 1, True, "relu", "categorical", 15, 1.0),
    (47, 129, 0, 256, 2, True, "tanh", "gaussian", 12, 0.3),
    (2, 8, 0, 256, 8, True, None, "categorical", 4, 1.0),
]


@pytest.mark.parametrize("rows,D,pad,width,depth,ln,act,dist,A,temperature", CASES)
def test_towers_step(rows, D, pad, width, depth, ln, act, dist, A, temperature):
    def torso():
        out = []
        for _ in range(depth):
            out += [nn.Dense(width)] + ([nn.LayerNorm()] if ln else [])
            out += [{"tanh": nn.tanh, "relu": nn.relu, "silu": nn.silu}[act]] if act else []
        return out
    if dist == "gaussian":
        actor = nn.Gaussian(nn.Sequential(torso() + [nn.SpreadScale(A)]))
    else:
        actor = nn.Categorical(nn.Sequential(torso() + [nn.Dense(A)]))
    net = nn.Network(feature_extractor=nn.FeatureExtractor(nn.Identity()),
                     head=nn.ActorCritic(actor=actor, critic=nn.Sequential(torso() + [nn.Dense(1)])))
    params = net.init(rows + D, D)["params"]
    plan = net.plan(D)
    obs = np.random.default_rng(D + A).standard_normal((rows, D)).astype(np.float32)
    head, value, _ = nets.forward(params, plan, obs)
    alg = PPO(cfg=recipes.make(2).cfg, network=net, optimizer=recipes.make(2).optimizer, use_graph=False)
    state = alg.init_from_params({"params": params}, D)
    o = torch.full((rows, D + pad), float("nan"), device="cuda")
    o[:, :D] = dev(obs)
    key = make_key(rows + 3 * A)
    out = {}
    for fused in (True, False):
        ex = StepExecutor(alg.program(D), flat_state_of(state), rows, fused=fused)
        assert (ex.towers is not None) == fused
        ex.KEY.copy_(key_dev(key))
        a = (torch.full((rows,), -1, dtype=torch.int32, device="cuda") if dist == "categorical"
             else torch.full((rows, A), float("nan"), device="cuda"))
        lp = torch.full((rows,), float("nan"), device="cuda")
        v = torch.full((rows,), float("nan"), device="cuda")
        ex.issue(stream(), o.data_ptr(), D + pad, temperature, a.data_ptr(), lp.data_ptr(), v.data_ptr())
        torch.cuda.synchronize()
        out[fused] = (a.cpu().numpy(), lp.cpu().numpy(), v.cpu().numpy())
    a, lp, v = out[True]
    np.testing.assert_allclose(v, value, rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(v, out[False][2], rtol=1e-5, atol=1e-5)
    if dist == "categorical":
        check_categorical(a, lp, head, key, temperature, 1e-4, 1e-5)
        return
    raw = nets_leaf(params, plan["dist"]["scale"])
    a_or, lp_or, eps = sample.gaussian_sample(head, raw, key, temperature)
    sig = temperature * (sample.softplus(np.broadcast_to(raw, head.shape)) + 1e-3)
    bound = 1e-5 * (np.abs(sig * eps) + np.abs(head)) + 1e-5
    np.testing.assert_array_less(np.abs(a - a_or), bound)
    np.testing.assert_allclose(lp, lp_or, rtol=1e-5, atol=1e-5)
    # the same draw as the sampling launch's, from the same formulas
    np.testing.assert_allclose(lp, out[False][1], rtol=1e-6, atol=1e-6)


def nets_leaf(tree, path):
    for k in path:
        tree = tree[k]
    return tree


@pytest.mark.parametrize("rows,width,depth,A,temperature", [(1, 32, 1, 2, 1.0), (16, 96, 2, 15, 0.0), (31, 200, 1, 7, 1.0),
                                                            (300, 512, 3, 14, 0.7), (17, 16, 1, 1, 1.0)])
def test_shared_head_and_draw_in_one_launch(rows, width, depth, A, temperature):
    """ppo_head_sample_categorical_f32 behind a trunk the one-launch step does
    not take: against the oracle, at widths whose 16-deep chunks leave waves
    idle or with a remainder (200 is no multiple of 16: the head GEMM's path)."""
    D = 24
    trunk = [f for _ in range(depth) for f in (nn.Dense(width), nn.tanh)]
    net = nn.Network(feature_extractor=nn.FeatureExtractor(nn.Sequential(trunk)),
                     head=nn.ActorCritic(actor=nn.Categorical(nn.Dense(A)), critic=nn.Dense(1)))
    params = net.init(rows + A, D)["params"]
    obs = np.random.default_rng(width).standard_normal((rows, D)).astype(np.float32)
    head, value, _ = nets.forward(params, net.plan(D), obs)
    alg = PPO(cfg=recipes.make(2).cfg, network=net, optimizer=recipes.make(2).optimizer, use_graph=False)
    state = alg.init_from_params({"params": params}, D)
    ex = StepExecutor(alg.program(D), flat_state_of(state), rows)
    assert not ex.fused and ex.head_samples == (width % 16 == 0)
    key = make_key(width + rows)
    _, _, action, aux = alg.step(state, None, key, Timestep(obs=dev(obs)), temperature)
    torch.cuda.synchronize()
    np.testing.assert_allclose(aux["value"].cpu().numpy(), value, rtol=1e-5, atol=1e-5)
    check_categorical(action.cpu().numpy(), aux["log_prob"].cpu().numpy(), head, key, temperature, 1e-4, 1e-5)


@pytest.mark.parametrize("rows,H,I,A", [(1, 64, 64, 2), (17, 128, 128, 15), (33, 256, 256, 8), (300, 256, 64, 3),
                                        (16, 512, 512, 4), (40, 64, 192, 5), (40, 64, 96, 16), (1000, 256, 256, 3),
                                        (2040, 256, 256, 4), (4090, 128, 128, 5), (500, 512, 64, 2)])
def test_recurrent_step_forms_the_projections(rows, H, I, A):
    """ppo_gru_fwd_step_x_f32 against the oracle and the projection GEMM's path,
    with rows reset, at equal and unequal widths (96: not its multiple of 64) and
    with one, two and four row tiles per workgroup."""
    D = 20
    net = nn.Network(feature_extractor=nn.FeatureExtractor(nn.Sequential([nn.Dense(I), nn.relu])),
                     torso=nn.RNN(nn.GRUCell(H)),
                     head=nn.ActorCritic(actor=nn.Categorical(nn.Dense(A)), critic=nn.Dense(1)))
    params = net.init(rows + H, D)["params"]
    rng = np.random.default_rng(H + I)
    obs = rng.standard_normal((rows, D)).astype(np.float32)
    carry = np.tanh(rng.standard_normal((rows, H))).astype(np.float32)
    term, trunc = rng.random(rows) < 0.2, rng.random(rows) < 0.1
    head, value, final, _ = nets.recurrent_forward(params, net.plan(D), obs[:, None, :], (term | trunc)[:, None], carry)
    alg = RecurrentPPO(cfg=recipes.make(4).cfg, network=net, optimizer=recipes.make(4).optimizer, use_graph=False)
    state = alg.init_from_params({"params": params}, D)
    key = make_key(H + rows)
    out = {}
    for fused in (True, False):
        ex = RecurrentStepExecutor(alg.program(D), flat_state_of(state), rows, fused=fused)
        assert ex.input_proj == (fused and I % 64 == 0) and ex.head_samples == (fused and A < 16)
        ex.KEY.copy_(key_dev(key))
        o, c, t1, t2 = dev(obs), dev(carry), dev(term), dev(trunc)
        c2 = torch.full((rows, H), float("nan"), device="cuda")
        a = torch.full((rows,), -1, dtype=torch.int32, device="cuda")
        lp, v = torch.full((rows,), float("nan"), device="cuda"), torch.full((rows,), float("nan"), device="cuda")
        ex.issue(stream(), o.data_ptr(), D, c.data_ptr(), t1.data_ptr(), t2.data_ptr(), 1.0, c2.data_ptr(), a.data_ptr(),
                 lp.data_ptr(), v.data_ptr())
        torch.cuda.synchronize()
        np.testing.assert_allclose(c2.cpu().numpy(), final, rtol=1e-5, atol=1e-5)
        np.testing.assert_allclose(v.cpu().numpy(), value[:, 0], rtol=1e-5, atol=1e-5)
        check_categorical(a.cpu().numpy(), lp.cpu().numpy(), head[:, 0], key, 1.0, 1e-4, 1e-5)
        out[fused] = c2.cpu().numpy()
    np.testing.assert_allclose(out[True], out[False], rtol=1e-5, atol=1e-5)


def test_device_keys_of_every_layout_draw_alike():
    """A step reads a contiguous device key in place; a strided one and a host
    key go through the executor's buffer."""
    net = nn.Network(feature_extractor=nn.FeatureExtractor(nn.Sequential([nn.Dense(64), nn.tanh])),
                     head=nn.ActorCritic(actor=nn.Categorical(nn.Dense(4)), critic=nn.Dense(1)))
    alg = PPO(cfg=recipes.make(2).cfg, network=net, optimizer=recipes.make(2).optimizer, use_graph=False)
    state = alg.init_from_params({"params": net.init(1, 6)["params"]}, 6)
    obs = torch.randn(200, 6, generator=torch.Generator().manual_seed(1)).cuda()
    key = make_key(9)
    strided = torch.zeros(2, 3, dtype=torch.int32, device="cuda")
    strided[:, 1] = key_dev(key)
    acts = [alg.step(state, None, k, Timestep(obs=obs))[2].cpu() for k in (key, key_dev(key), strided[:, 1])]
    assert torch.equal(acts[0], acts[1]) and torch.equal(acts[0], acts[2])
    with pytest.raises(ValueError):
        alg.step(state, None, torch.zeros(2, dtype=torch.int64, device="cuda"), Timestep(obs=obs))
