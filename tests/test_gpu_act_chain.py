"""An actor / critic pair of plain Dense -> activation towers in one launch
per step (forward, heads + loss, torso backward): the first minibatch's
gradient and the parameters after a whole update against the same update layer
by layer, over widths, depths, activations, both distributions, input widths
the vector loads cannot take and ragged last tiles.

Bar: the two paths form the same fp32 sums in other orders: gradients within
rel-L2 2e-5 of the layer-by-layer path's, parameters after the update within
1e-3 of that update's change (Adam turns the rounding of a near-zero gradient
into a step of its own size), logs to 1e-4."""
import numpy as np
import pytest
import torch

from boonta_amd import networks as nn
from boonta_amd import optim
from boonta_amd.algorithms.ppo import PPO, PPOConfig, flat_state_of
from boonta_amd.learner import MLPExecutor
from boonta_amd.random import key as make_key
from boonta_amd.types import Timestep, Transition

pytestmark = pytest.mark.gpu


class _PerLayer(MLPExecutor):
    CHAIN_ACT = False


class _PerLayerPPO(PPO):
    executor_class = _PerLayer


def algorithm(cls, width, depth, act, gaussian, A, M, use_graph):
    def torso():
        out = []
        for _ in range(depth):
            out += [nn.Dense(width)] + ([act] if act is not None else [])
        return out
    actor = (nn.Gaussian(nn.Sequential(torso() + [nn.SpreadScale(A)])) if gaussian
             else nn.Categorical(nn.Sequential(torso() + [nn.Dense(A)])))
    net = nn.Network(feature_extractor=nn.FeatureExtractor(nn.Identity()),
                     head=nn.ActorCritic(actor=actor, critic=nn.Sequential(torso() + [nn.Dense(1)])))
    cfg = PPOConfig(num_minibatches=M, update_epochs=2, clip_coefficient=0.2, clip_value_loss=True,
                    entropy_coefficient=0.01, value_coefficient=0.5, gamma=0.99, gae_lambda=0.95,
                    normalize_advantage=False)
    return cls(cfg=cfg, network=net, optimizer=optim.chain(optim.clip_by_global_norm(0.5), optim.adam(3e-4)),
               use_graph=use_graph)


def transition(T, N, D, gaussian, A):
    g = torch.Generator(device="cuda").manual_seed(T * N + D)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    obs = r(T + 1, N, D)
    action = r(T, N, A) if gaussian else torch.randint(0, A, (T, N), device="cuda", generator=g).to(torch.int32)
    lp = -0.5 * (action * action).sum(-1) - 0.92 * A if gaussian else torch.full((T, N), -float(np.log(A)), device="cuda")
    done = torch.rand(T, N, device="cuda", generator=g) < 0.05
    return Transition(first=Timestep(obs=obs[:-1]),
                      second=Timestep(obs=obs[1:], action=action, reward=r(T, N), terminated=done,
                                      truncated=torch.zeros_like(done)),
                      aux={"log_prob": lp.contiguous(), "value": 0.1 * r(T, N)})


@pytest.mark.parametrize("width, depth, act, gaussian, A, D, T, N, M, use_graph", [
    (64, 2, nn.tanh, False, 2, 4, 16, 8, 4, True),        # 32-row minibatches
    (64, 1, nn.relu, False, 14, 3, 8, 5, 2, False),       # 20 rows: a ragged second tile
    (128, 3, nn.relu, True, 4, 17, 16, 33, 2, True),      # 264 rows, an odd input width
    (256, 2, nn.tanh, True, 8, 87, 16, 128, 1, True),
    (256, 4, nn.tanh, False, 6, 130, 8, 75, 3, False),
    (128, 2, None, False, 5, 64, 8, 16, 1, False)])       # no activation
def test_one_launch_step_matches_the_layer_by_layer_update(width, depth, act, gaussian, A, D, T, N, M, use_graph):
    tr = transition(T, N, D, gaussian, A)
    out = []
    for cls in (PPO, _PerLayerPPO):
        alg = algorithm(cls, width, depth, act, gaussian, A, M, use_graph)
        params = alg.network.init(3, D)
        state = alg.init_from_params(params, D)
        p0 = flat_state_of(state).P.cpu().numpy().copy()
        ex = alg.executor(state, T, N, D)
        assert ex.chain_act == (cls is PPO)
        ex.bind(alg._inputs(tr, D)[0])
        ex.KEY.copy_(torch.tensor([0, 5], dtype=torch.int32))
        ex.issue(torch.cuda.current_stream().cuda_stream, max_steps=1)
        torch.cuda.synchronize()
        grad = flat_state_of(state).G.cpu().numpy().copy()
        state = alg.init_from_params(params, D)
        ex = alg.executor(state, T, N, D)
        alg.update(state, make_key(9), tr)
        torch.cuda.synchronize()
        out.append((grad, flat_state_of(state).P.cpu().numpy().copy() - p0, ex.LOGS.cpu().numpy().copy()))
    (g1, d1, l1), (g0, d0, l0) = out
    rel = lambda a, b: float(np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b))
    assert rel(g1, g0) <= 2e-5
    assert rel(d1, d0) <= 1e-3
    np.testing.assert_allclose(l1, l0, rtol=1e-4, atol=1e-5)


def test_recorded_act_chain_arguments_match_the_signature(monkeypatch):
    """(the launch's argument list, recorded over device memory without running it)"""
    from boonta_amd import _lib
    alg = algorithm(PPO, 64, 2, nn.tanh, False, 3, 2, True)
    state = alg.init_from_params(alg.network.init(0, 5), 5)
    ex = alg.executor(state, 8, 8, 5)
    ex.bind(alg._inputs(transition(8, 8, 5, False, 3), 5)[0])
    calls = [a for n, a in ex.record() if n == "ppo_mlp_act_fwd_head_loss_bwd_f32"]
    assert len(calls) == 4 and all(len(a) == len(_lib.SIGNATURES["ppo_mlp_act_fwd_head_loss_bwd_f32"][1]) for a in calls)
