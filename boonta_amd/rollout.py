"""The rollout-side ``PPO.step`` on MI355X kernels (boonta/algorithms/ppo.py:57-74).

``StepExecutor`` binds an MLP program to a number of environments and issues,
on one stream:

    network forward on timestep.obs [rows, obs]     network.py:18-49 (shared
        trunk or separate actor / critic towers, as in the learner)
    head GEMMs -> logits or mean, and the value column
    sample_and_log_prob(seed=key)                   distributions.py:8-57
        (``ppo_sample_categorical_f32`` / ``ppo_sample_gaussian_f32``)

``RecurrentStepExecutor`` is the same for ``RecurrentPPO.step``
(recurrent_ppo.py:71-96): trunk forward, the GRU input projection, one GRU
step from the given carry with the carry reset to zeros where the timestep is
done (reset_carry, networks/blocks/rnn.py:11-16,43-46), the heads on the new
carry, and the sampling launch.

The forward reuses the learner's kernels (``ForwardChain``) and reads the
same flat parameter buffer, so a step issued after an update sees the updated
parameters without a copy.
"""
from __future__ import annotations

import ctypes

import torch

from . import _lib
from .learner import (A_ROW, B_KN, EPI_BIAS_ACT, LayerBufs, DenseSpec, FlatState, ForwardChain, Program, _act, _p,
                      forward_bufs,
                      split_forward_bufs)


def _head_samples(program: Program, lib) -> bool:
    """Whether ppo_head_sample_categorical_f32 takes the program's shared head:
    on a trunk's float32 features (the executor's own, 16-byte rows) at every
    number of rows."""
    h = program.head_a
    return (not program.bf16 and program.shared_head and bool(program.trunk) and program.dist["kind"] == "categorical"
            and program.head_out == program.dist["num"] and program.head_out + 1 <= lib.ppo_step_towers_max_outputs()
            and h.fin % 16 == 0)


class StepExecutor(ForwardChain):
    """PPO.step for a fixed number of environments (rows).

    A float32 shared-trunk MLP of 256-wide Dense layers with one activation
    and a categorical head of at most 15 logits (the discrete Anakin network)
    steps in one launch, ``ppo_step_mlp_categorical_f32``, and float32 actor
    and critic towers of one shape (Dense layers of 64, 128 or 256 features, or
    256 with LayerNorm; at most 16 actor outputs) in ``ppo_step_towers_f32``;
    ``fused=False`` issues the layer-by-layer GEMMs and the sampling launch
    instead."""

    def __init__(self, program: Program, flat: FlatState, rows: int, fused: bool = True):
        if program.gru is not None:
            raise TypeError("a recurrent program steps through RecurrentPPO")
        super().__init__(program, flat)
        lib = _lib.load()
        if program.action_dim > lib.ppo_sample_max_outputs():
            raise NotImplementedError(f"an action dimension above {lib.ppo_sample_max_outputs()} is not compiled")
        dev = flat.device
        self.rows = rows
        self.trunk = [forward_bufs(s, rows, dev) for s in program.trunk]
        self.actor = [forward_bufs(s, rows, dev) for s in program.actor_layers]
        self.critic = [forward_bufs(s, rows, dev) for s in program.critic_layers]
        for group in (self.trunk, self.actor, self.critic):
            if group:
                split_forward_bufs(group[0], rows, dev, self.bf16)
        f32 = dict(dtype=torch.float32, device=dev)
        ha, hc = program.head_a, program.head_c
        if program.shared_head:
            self.HEAD = torch.zeros(rows, ha.w.ld, **f32)
        else:
            self.HA = torch.zeros(rows, ha.w.ld, **f32)
            self.HC = torch.zeros(rows, hc.w.ld, **f32)
        self.KEY = torch.zeros(2, dtype=torch.int32, device=dev)
        self.fused = fused and self._fusable(lib)
        self.head_samples = fused and _head_samples(program, lib)
        self.trunk_tables = self._trunk_tables() if self.fused else None
        self.towers = self._tower_tables() if fused and self._towers_fusable(lib) else None

    def _fusable(self, lib) -> bool:
        """Whether the one-launch step kernel covers this program."""
        prog = self.prog
        trunk = prog.trunk
        if (self.bf16 or not prog.shared_head or prog.dist["kind"] != "categorical" or not trunk
                or len(trunk) > lib.ppo_step_mlp_max_layers() or trunk[0].dense.fin > lib.ppo_step_mlp_max_obs()):
            return False
        if len({s.act for s in trunk}) != 1 or any(s.ln is not None for s in trunk):
            return False
        if any(s.fout != 256 or s.ld != 256 or (i > 0 and s.dense.fin != 256) for i, s in enumerate(trunk)):
            return False
        h = prog.head_a
        return h.fin == 256 and h.w.ld <= 16 and prog.head_out == prog.dist["num"] and prog.head_out + 1 <= h.w.ld

    def _trunk_tables(self) -> dict:
        """Host arrays of ppo_step_mlp_categorical_f32's parameter pointers."""
        prog, view, h = self.prog, self.flat.view, self.prog.head_a
        n = len(prog.trunk)
        keep = ((ctypes.c_void_p * n)(*[view(s.dense.w) for s in prog.trunk]),
                (ctypes.c_int64 * n)(*[s.ld for s in prog.trunk]),
                (ctypes.c_void_p * n)(*[view(s.dense.b) if s.dense.b is not None else None for s in prog.trunk]))
        return {"keep": keep, "args": (n, *map(ctypes.addressof, keep), _act(prog.trunk[0].act), view(h.w), h.w.ld)}

    def _towers_fusable(self, lib) -> bool:
        """Whether the paired towers' one-launch step covers this program, and
        its number of rows: it replaces two launches per layer and three after (4
        x 256 LayerNorm + SiLU, 4096 rows: 125 -> 64 us).  The layers' GEMMs
        overtake its 16-row chains on fp32 MFMA as the rows' products grow beside
        the launches saved, sooner where the input's rows take no 16-byte loads.
        Us, this launch / layer by layer: plain towers, 3 x 256 on 300 inputs,
        9000 rows 136 / 165, 12288 156 / 149; 2 x 256 on 87, 16384 109 / 120; 1 x
        256 on 600, 4096 52 / 67, on 1000, 7000 159 / 117; 1 x 128 on 600, 4096
        36 / 60, 16384 157 / 81, on 159, 10580 70 / 52; 4 x 64 on 98, 52037 154 /
        154.  With LayerNorm, whose layers run 16-row tiles as well, only through
        a wide input: 4 x 256 on 87, 65536 rows 937 / 1144; 1 x 256 on 916, 2994
        75 / 87, on 1500, 16384 456 / 406, on 489, 7020 157 / 129, on 109,
        48756 239 / 190; 2 x 256 on 2044, 11341 500 / 563, on 2010, 856 292 / 220.
        Over 83 drawn shapes the choice is within 14 % of the better."""
        prog = self.prog
        A, C = prog.actor_layers, prog.critic_layers
        if (self.bf16 or prog.shared_head or not A or len(A) != len(C) or len(A) > lib.ppo_step_towers_max_layers()
                or A[0].dense.fin * A[0].fout > 2 ** 31 - 1):
            return False
        s0 = A[0]
        F, ln = s0.fout, s0.ln is not None
        if (F not in ((256,) if ln else (64, 128, 256))
                or s0.act not in ("relu", "tanh", None) + (("silu",) if ln else ())):
            return False
        for layers in (A, C):
            for i, s in enumerate(layers):
                if (s.fout != F or s.ld != F or s.dense.w.ld != F or s.act != s0.act or (s.ln is not None) != ln
                        or s.dense.fin != (A[0].dense.fin if i == 0 else F) or (ln and s.ln["eps"] != s0.ln["eps"])):
                    return False
        K0 = s0.dense.fin
        L, aligned = len(A), K0 % 4 == 0
        if ln:
            wide = K0 * F > (280_000 if aligned else 60_000 if self.rows <= 16384 else 20_000) * L
            if wide and (self.rows > 2048 or not aligned):
                return False
        else:
            macs = self.rows * F * ((1.0 if aligned else 1.5) * K0 + (L - 1) * F)  # of one tower
            if macs > ((0.5 + 0.5 * L) if F == 256 else (0.32 + 0.4 * (L - 1))) * 1e9:
                return False
        ha, hc = prog.head_a, prog.head_c
        gaussian = prog.dist["kind"] != "categorical"
        if gaussian and (prog.scale_region is None or prog.dist["dim"] != prog.head_out):
            return False
        if not gaussian and prog.dist["num"] != prog.head_out:
            return False
        # (the launch loads parameters as 16-byte vectors)
        base = self.flat.P.data_ptr()
        regions = [r for layers in (A, C) for s in layers
                   for r in (s.dense.w, s.dense.b, *((s.ln["scale"], s.ln["bias"]) if ln else ())) if r is not None]
        return (ha.fin == F and hc.fin == F and hc.fout == 1 and prog.head_out <= lib.ppo_step_towers_max_outputs()
                and all((base + 4 * r.offset) % 16 == 0 for r in regions))

    def _tower_tables(self) -> dict:
        """Host arrays of ppo_step_towers_f32's parameter pointers (kept: the
        flat buffers live as long as this executor)."""
        prog, view = self.prog, self.flat.view
        layers = prog.actor_layers + prog.critic_layers
        heads = (prog.head_a, prog.head_c)
        vp = lambda xs: (ctypes.c_void_p * len(xs))(*xs)
        ln = layers[0].ln
        keep = {"W": vp([view(s.dense.w) for s in layers]),
                "b": vp([view(s.dense.b) if s.dense.b is not None else None for s in layers]),
                "g": vp([view(s.ln["scale"]) for s in layers]) if ln else None,
                "be": vp([view(s.ln["bias"]) for s in layers]) if ln else None,
                "hw": vp([view(h.w) for h in heads]), "ldh": (ctypes.c_int64 * 2)(*[h.w.ld for h in heads]),
                "hb": vp([view(h.b) if h.b is not None else None for h in heads])}
        s0 = layers[0]
        t = {k: None if v is None else ctypes.addressof(v) for k, v in keep.items()}
        t.update(keep=keep, args=(len(prog.actor_layers), s0.fout, t["W"], t["b"], t["g"], t["be"],
                                  float(ln["eps"]) if ln else 0.0, _act(s0.act), t["hw"], t["ldh"], t["hb"],
                                  prog.head_out, view(prog.scale_region) if prog.scale_region is not None else None))
        return t

    def _head(self, st, x, ldx, h: DenseSpec, out: torch.Tensor):
        """Head Dense on the last features (bias added, no activation)."""
        self._gemm(st, A_ROW, B_KN, x, ldx, None, self.flat.view(h.w), h.w.ld, _p(out), h.w.ld, self.rows,
                   h.w.ld, h.fin, 1, 0, EPI_BIAS_ACT, self.flat.view(h.b) if h.b is not None else None, 0, None,
                   None, 0, None, -1)

    def issue(self, st: int, obs: int, ldo: int, temperature: float, action: int, log_prob: int, value: int,
              key: int | None = None):
        """Enqueues one step on stream handle ``st``: obs is a device pointer
        to [rows, ldo] float32; action [rows] int32 (categorical) or [rows, D]
        float32 (Gaussian), log_prob and value [rows] float32; key a device
        pointer to uint32[2] key data (default: this executor's KEY buffer)."""
        key = _p(self.KEY) if key is None else key
        prog = self.prog
        rows = self.rows
        if self.fused:
            h, t = prog.head_a, self.trunk_tables
            self._call("ppo_step_mlp_categorical_f32", st, obs, ldo, rows, prog.trunk[0].dense.fin, *t["args"],
                       self.flat.view(h.b) if h.b is not None else None, prog.dist["num"], key, float(temperature),
                       action, log_prob, value)
            return
        if self.towers is not None:
            self._call("ppo_step_towers_f32", st, obs, ldo, rows, prog.actor_layers[0].dense.fin, *self.towers["args"],
                       key, float(temperature), action, log_prob, value)
            return
        if prog.shared_head:
            x, ldx, _ = self._fwd_layers(st, self.trunk, obs, ldo, None, rows)
            if self.head_samples:
                h = prog.head_a
                self._call("ppo_head_sample_categorical_f32", st, x, ldx, rows, h.fin, self.flat.view(h.w), h.w.ld,
                           self.flat.view(h.b) if h.b is not None else None, prog.head_out, key, float(temperature),
                           action, log_prob, value)
                return
            self._head(st, x, ldx, prog.head_a, self.HEAD)
            head, ldh = self.HEAD, self.HEAD.shape[1]
            vsrc, ldv = _p(self.HEAD) + 4 * prog.head_out, ldh
        else:
            xa, lda, _ = self._fwd_layers(st, self.actor, obs, ldo, None, rows)
            self._head(st, xa, lda, prog.head_a, self.HA)
            xc, ldc, _ = self._fwd_layers(st, self.critic, obs, ldo, None, rows)
            self._head(st, xc, ldc, prog.head_c, self.HC)
            head, ldh = self.HA, self.HA.shape[1]
            vsrc, ldv = _p(self.HC), self.HC.shape[1]
        dist = prog.dist
        if dist["kind"] == "categorical":
            self._call("ppo_sample_categorical_f32", st, _p(head), ldh, rows, dist["num"], vsrc, ldv, key,
                       float(temperature), action, log_prob, value)
        else:
            D = dist["dim"]
            if prog.scale_region is not None:
                scale, lds = self.flat.view(prog.scale_region), 0
            else:
                scale, lds = _p(head) + 4 * D, ldh
            self._call("ppo_sample_gaussian_f32", st, _p(head), ldh, scale, lds, rows, D, vsrc, ldv, key,
                       float(temperature), action, D, log_prob, value)

    def record(self, *issue_args) -> list:
        """The launch sequence of one step as (entry point, args) without
        running it (used by the benchmark to time single launches)."""
        calls = []
        self._call = lambda name, *args: calls.append((name, args))
        try:
            self.issue(0, *issue_args)
        finally:
            self._call = _lib.call
        return calls


class RecurrentStepExecutor(ForwardChain):
    """RecurrentPPO.step for a fixed number of environments (rows): the
    network of ``Network(feature_extractor=<MLP>, torso=RNN(GRUCell(H)),
    head=ActorCritic(Dense, Dense))`` one time step at a time: the trunk's
    launches, one for the GRU step with its input projections (a trunk width that
    is a multiple of 64), one for the head and the draw (at most 15 logits);
    ``fused=False`` issues the projection GEMM, the head GEMM and the sampling
    launch instead (128 -> 256 -> GRU 256, 1024 envs: 42 -> 28
    us a step, a key copy left out besides)."""

    def __init__(self, program: Program, flat: FlatState, rows: int, fused: bool | None = None):
        # (None: fused where the parameters are on the device, not where launches
        # are recorded over host memory)
        fused = flat.P.is_cuda if fused is None else fused
        if program.gru is None:
            raise TypeError("RecurrentStepExecutor needs a program with a GRU torso")
        if not program.shared_head or not program.trunk:
            raise NotImplementedError("the recurrent step compiles an MLP feature extractor, the GRU and plain "
                                      "Dense heads")
        if program.dist["kind"] != "categorical":
            raise NotImplementedError("the recurrent step compiles a categorical head")
        super().__init__(program, flat)
        lib = _lib.load()
        if program.action_dim > lib.ppo_sample_max_outputs():
            raise NotImplementedError(f"an action dimension above {lib.ppo_sample_max_outputs()} is not compiled")
        dev = flat.device
        H = program.gru.H
        f32 = dict(dtype=torch.float32, device=dev)
        self.rows = rows
        self.trunk: list[LayerBufs] = [forward_bufs(s, rows, dev) for s in program.trunk]
        # (ahead of the projection GEMM and the step apart at every size timed but
        # wide inputs of many sequences: 1024 -> 256, 4096 120 / 115 us, 16384 404 /
        # 369; 512 -> 64, 4096 30 / 38, 16384 78 / 71; 2048 -> 128 107 / 119, 373 /
        # 325; 256 -> 512, 16384 480 / 551)
        self.input_proj = (fused and program.gru.fin % 64 == 0
                           and not (program.gru.fin >= 4 * H and rows > 4096))
        self.head_samples = fused and _head_samples(program, lib)
        if not self.input_proj:
            self.XI = torch.zeros(rows, 3 * H, **f32)
        if not self.head_samples:
            self.HEAD = torch.zeros(rows, program.head_a.w.ld, **f32)
        self.KEY = torch.zeros(2, dtype=torch.int32, device=dev)

    def issue(self, st: int, obs: int, ldo: int, carry: int, terminated: int | None, truncated: int | None,
              temperature: float, carry_out: int, action: int, log_prob: int, value: int, key: int | None = None):
        """Enqueues one step: obs [rows, ldo] and carry [rows, H] float32 in,
        terminated / truncated [rows] bool (or None: no reset); the new carry
        [rows, H], action [rows] int32, log_prob and value [rows] out."""
        key = _p(self.KEY) if key is None else key
        prog = self.prog
        g = prog.gru
        H, I = g.H, g.fin
        rows = self.rows
        x, ldx, _ = self._fwd_layers(st, self.trunk, obs, ldo, None, rows)
        if self.input_proj:
            self._call("ppo_gru_fwd_step_x_f32", st, x, ldx, I, self.flat.view(g.wi), 3 * H, self.flat.view(g.bi),
                       carry, H, terminated, truncated, self.flat.view(g.wh), 3 * H, self.flat.view(g.bhn), carry_out,
                       H, rows, H)
        else:
            self._gemm(st, A_ROW, B_KN, x, ldx, None, self.flat.view(g.wi), 3 * H, _p(self.XI), 3 * H, rows, 3 * H, I,
                       1, 0, EPI_BIAS_ACT, self.flat.view(g.bi), 0, None, None, 0, None, -1)
            self._call("ppo_gru_fwd_step_f32", st, _p(self.XI), 3 * H, carry, H, None, terminated, truncated, None,
                       self.flat.view(g.wh), 3 * H, self.flat.view(g.bhn), carry_out, H, None, H, None, 4 * H, rows, H)
        h = prog.head_a
        if self.head_samples:
            self._call("ppo_head_sample_categorical_f32", st, carry_out, H, rows, H, self.flat.view(h.w), h.w.ld,
                       self.flat.view(h.b) if h.b is not None else None, prog.head_out, key, float(temperature),
                       action, log_prob, value)
            return
        self._gemm(st, A_ROW, B_KN, carry_out, H, None, self.flat.view(h.w), h.w.ld, _p(self.HEAD), h.w.ld, rows,
                   h.w.ld, h.fin, 1, 0, EPI_BIAS_ACT, self.flat.view(h.b) if h.b is not None else None, 0, None,
                   None, 0, None, -1)
        ldh = self.HEAD.shape[1]
        self._call("ppo_sample_categorical_f32", st, _p(self.HEAD), ldh, rows, prog.dist["num"],
                   _p(self.HEAD) + 4 * prog.head_out, ldh, key, float(temperature), action, log_prob, value)

    def record(self, *issue_args) -> list:
        calls = []
        self._call = lambda name, *args: calls.append((name, args))
        try:
            self.issue(0, *issue_args)
        finally:
            self._call = _lib.call
        return calls
