"""Performance cases: the work a user of this library has it do, through its
public entry points (the ``mdnav`` package and the C ABI behind it).

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same
ranges.  ``prepare(case, seed)`` makes what a program holds before the call
(simulator, trainer, policy, rollout rows), ``run(state)`` does one pass and
returns what it computes, ``work(case)`` counts the bytes and operations the
pass cannot do without, ``tolerance(case)`` bounds how far another correct
implementation of the same precision may be, and ``exact(case, seed)`` gives
the result in 64 bits where plain tensor code can form it.

The kinds of case:

* ``train``     one training iteration: rollout of every environment, then the
                PPO update (the small 64-unit policy);
* ``evaluate``  one deterministic evaluation: reset, roll out, read the runs;
* ``wide``      one training iteration with the wide bf16 policy in the loop;
* ``update``    the PPO update alone on rollout rows the program uploaded;
* ``forward``   the policy over a batch of host observations;
* ``normalize`` advantage normalisation of device memory on a stream.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "metal-drone-nav_amd"))

from mdnav import (LargePPOTrainer, PPOTrainer, Sim, abi, formats, native, ops, task_runtime,  # noqa: E402
                   task_settings)

LOG_TWO_PI = math.log(2.0 * math.pi)


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the reference's CPU training shape: 512 envs x 64 ticks, its own
        # schedule of 256-row minibatches
        dict(name="train_cpu_shape", kind="train", envs=512, ticks=64, family=1, obs=181, memory=0, delay=0, tasks=0,
             epochs=2, minibatch=256),
        # the benchmark's default workload: 8,192 envs x 128 ticks in static
        # boxes, one epoch of four minibatches
        dict(name="train_headline", kind="train", envs=8192, ticks=128, family=1, obs=181, memory=0, delay=0,
             tasks=0, epochs=1, minibatch=262144),
        # the reference's own benchmark schedule: 8,192 x 32, two epochs of
        # 256-row minibatches (2,048 optimiser steps)
        dict(name="train_reference_schedule", kind="train", envs=8192, ticks=32, family=1, obs=181, memory=0,
             delay=0, tasks=0, epochs=2, minibatch=256),
        # the guided actor with the geometry-memory hint, the benchmark's
        # --geometry-memory mode with a shorter rollout
        dict(name="train_guided_memory", kind="train", envs=8192, ticks=32, family=1, obs=184, memory=1, delay=0,
             tasks=0, epochs=1, minibatch=65536),
        # the reference's task training loop: 128 envs x 32 ticks of clutter
        # tasks with per-episode plants, guided actor with memory
        dict(name="train_tasks", kind="train", envs=128, ticks=32, family=12, obs=184, memory=1, delay=0, tasks=1,
             epochs=2, minibatch=256),
        # the moving-threat rehearsal with 100 ms sensor and command delays at
        # an odd size: a fleet that fills the GPU only in part, a ragged last
        # minibatch
        dict(name="train_threats_ragged", kind="train", envs=3001, ticks=50, family=13, obs=181, memory=0, delay=2,
             tasks=0, epochs=2, minibatch=40000),
        # the periodic evaluation of a training run: 128 episodes of the
        # trained guided policy (mode 17, geometry memory), 200 ticks
        dict(name="evaluate_guided", kind="evaluate", envs=128, ticks=200, family=3),
        # the capacity actor (184-5120-4) in the loop with its update
        dict(name="wide_train", kind="wide", envs=4096, ticks=32, hidden=5120, epochs=4, minibatch=32768),
        # the update alone, small policy, from rollout rows of another
        # simulator: ragged minibatches
        dict(name="update_ragged", kind="update", envs=1000, ticks=37, obs=184, hidden=64, epochs=2, minibatch=4096),
        # the update alone, capacity actor at its production minibatch
        dict(name="update_wide", kind="update", envs=2048, ticks=32, obs=184, hidden=5120, epochs=4,
             minibatch=32768),
        # the deployed policy over a batch of recorded observations (host arrays)
        dict(name="forward_batch", kind="forward", batch=4096, obs=184, hidden=64),
        # normalisation inside another program's step (device memory, its
        # stream): the smallest call
        dict(name="normalize_small", kind="normalize", count=128 * 32),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "evaluate", "wide", "update", "update", "forward", "normalize"])
    if kind == "train":
        tasks = int(rng.random() < 0.25)
        if tasks:
            return dict(kind=kind, envs=_log(rng, 32, 512), ticks=rng.randint(8, 32), family=12, obs=184, memory=1,
                        delay=0, tasks=1, epochs=2, minibatch=256)
        obs = rng.choice([181, 181, 184])
        memory = int(obs == 184 and rng.random() < 0.5)
        family = rng.choice([1, 1, 12, 13, abi.FAMILY_C3_MIX])
        delay = 2 if family in (13, abi.FAMILY_C3_MIX) else rng.choice([0, 0, 1])
        envs = _log(rng, 64, 8192)
        small = rng.random() < 0.4  # the reference's schedule, up to 1,024 steps
        most = 131072 if small or memory else 400000
        ticks = max(4, min(rng.randint(8, 128), most // envs))
        minibatch = 256 if small else -(-envs * ticks // rng.randint(2, 5))
        return dict(kind=kind, envs=envs, ticks=ticks, family=family, obs=obs, memory=memory, delay=delay, tasks=0,
                    epochs=2 if small else 1, minibatch=minibatch)
    if kind == "evaluate":
        return dict(kind=kind, envs=_log(rng, 32, 512), ticks=rng.randint(60, 200), family=rng.choice([0, 3, 5, 7]))
    if kind == "wide":
        envs = _log(rng, 256, 4096)
        return dict(kind=kind, envs=envs, ticks=rng.randint(6, 32), hidden=128 * _log(rng, 4, 40),
                    epochs=rng.randint(1, 4), minibatch=_log(rng, 4096, 32768))
    if kind == "update":
        hidden = rng.choice([64, 64, 64, 128 * _log(rng, 4, 40)])
        envs = _log(rng, 64, 2048)
        if hidden == 64:
            minibatch = rng.choice([256, _log(rng, 300, 65536)])
            most = 60000 if minibatch < 1024 else 200000
        else:
            minibatch, most = _log(rng, 2048, 32768), 65536
        ticks = max(8, min(rng.randint(8, 128), most // envs))
        return dict(kind=kind, envs=envs, ticks=ticks, obs=rng.choice([181, 184]), hidden=hidden,
                    epochs=rng.randint(1, 4), minibatch=minibatch)
    if kind == "forward":
        hidden = rng.choice([64, 64, 64, 128 * _log(rng, 1, 16)])
        return dict(kind=kind, batch=_log(rng, 1, 16384 if hidden == 64 else 1024), obs=rng.choice([181, 184]),
                    hidden=hidden)
    return dict(kind=kind, count=_log(rng, 1000, 1 << 22))


# ---------------------------------------------------------------- preparation
def _config(case, seed):
    kw = dict(n=case["envs"], family=case["family"], seed=1 + seed % 1000003, speed=1.0, distance=3.0)
    if case["tasks"]:  # the reference's task training settings
        kw.update(mode=22, speed=1.5, distance=8.0, max_steps=400, entropy_coef=0.001, learning_rate=0.0001)
    elif case["family"] != 1:
        kw.update(speed=1.5, distance=4.0)
    kw.update(sensor_delay=case["delay"], command_delay=case["delay"], geometry_memory=case["memory"])
    return abi.default_config(**kw)


def _jitter(values, rng):
    """A policy some way into training: the initialisation, each weight off by a few per cent."""
    return (values * (1.0 + 0.05 * rng.standard_normal(values.size))).astype(np.float32)


def _rows(case, seed, actor, critic):
    """Rollout rows as a simulator records them: pooled ranges in (0, 1] with
    the previous frame close to the current one, body-frame context, actions
    sampled around the policy's means, values near the critic's, episode ends
    in about 2 % of the rows."""
    n, t, d, h = case["envs"], case["ticks"], case["obs"], case["hidden"]
    rows = n * t
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    def uniform(*shape):
        return torch.rand(*shape, generator=g, device="cuda")

    obs = torch.empty(rows, d, device="cuda")
    obs[:, :80] = (0.05 + 1.2 * uniform(rows, 80) ** 2).clamp(max=1.0)
    obs[:, 80:160] = (obs[:, :80] + 0.02 * normal(rows, 80)).clamp(0.0, 1.0)
    obs[:, 160:d] = (0.4 * normal(rows, d - 160)).clamp(-1.5, 1.5)
    co = 0.5 * normal(rows, 32)
    co[:, 30:] = 0.0
    a, c = torch.from_numpy(actor).cuda().double(), torch.from_numpy(critic).cuda().double()
    means, values = torch.empty(rows, 4, device="cuda"), torch.empty(rows, device="cuda")
    for lo in range(0, rows, 16384):
        hi = min(rows, lo + 16384)
        means[lo:hi] = _actor(a, obs[lo:hi].double(), h)[0].float()
        values[lo:hi] = _critic(c, co[lo:hi].double(), h)[0].float()
    noise = normal(rows, 4)
    log_std = a[-4:].float()
    out = dict(obs=obs, critic_obs=co, actions=means + noise * log_std.exp(),
               logp=(-0.5 * (noise * noise + 2.0 * log_std + LOG_TWO_PI)).sum(1) + 0.02 * normal(rows),
               values=values + 0.05 * normal(rows), next_values=values + 0.1 * normal(rows),
               rewards=-0.01 + 0.05 * normal(rows))
    ends = uniform(rows)
    out["terminated"] = (ends < 0.015).to(torch.uint8)
    out["truncated"] = ((ends >= 0.015) & (ends < 0.02)).to(torch.uint8)
    out["rewards"] -= 10.0 * (ends < 0.012).float()
    return out


def _update_policy(case, seed):
    """Actor and critic vectors of an update case at the initialisation's scales."""
    rng = np.random.default_rng(seed)
    d, h = case["obs"], case["hidden"]
    wide = math.sqrt(64.0 / h)
    actor = np.concatenate([0.04 * rng.standard_normal(h * d), 0.01 * rng.standard_normal(h),
                            0.05 * wide * rng.standard_normal(4 * h), 0.01 * rng.standard_normal(4),
                            -1.0 + 0.1 * rng.standard_normal(4)]).astype(np.float32)
    critic = np.concatenate([0.15 * rng.standard_normal(32 * h), 0.01 * rng.standard_normal(h),
                             0.1 * wide * rng.standard_normal(h), [0.05]]).astype(np.float32)
    return actor, critic


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "train":
        sim = Sim(_config(case, seed), case["ticks"], actor_obs=case["obs"])
        if case["tasks"]:
            sim.set_runtime(task_runtime(1.0))
            sim.set_tasks(task_settings(2, case["family"]))
            sim.reset()
        sim.set("actor", _jitter(sim.get("actor"), rng))
        sim.set("critic", _jitter(sim.get("critic"), rng))
        return dict(kind=kind, sim=sim, ppo=PPOTrainer(sim, case["epochs"], case["minibatch"]), tasks=case["tasks"],
                    done=0)
    if kind == "evaluate":
        weights = formats.read_navigation_policy(os.path.join(ROOT, "tests", "golden", "navigation.bin"))[1]
        cfg = abi.default_config(n=case["envs"], family=case["family"], mode=17, eval=1, seed=1 + seed % 1000003,
                                 speed=1.5, distance=4.0, max_steps=case["ticks"], geometry_memory=1)
        sim = Sim(cfg, 32, actor_obs=184)
        sim.set("actor", weights)
        return dict(kind=kind, sim=sim, ticks=case["ticks"])
    if kind == "wide":
        cfg = abi.default_config(n=case["envs"], family=1, speed=1.0, distance=3.0, seed=1 + seed % 1000003)
        sim = Sim(cfg, case["ticks"], actor_obs=184)
        lp = LargePPOTrainer(sim, case["hidden"], case["epochs"], case["minibatch"])
        lp.set("actor", _jitter(lp.get("actor"), rng))
        lp.set("critic", _jitter(lp.get("critic"), rng))
        return dict(kind=kind, sim=sim, lp=lp, done=0)
    if kind == "update":
        cfg = abi.default_config(n=case["envs"], family=1, speed=1.0, distance=3.0)
        sim = Sim(cfg, case["ticks"], actor_obs=case["obs"])
        actor, critic = _update_policy(case, seed)
        small = case["hidden"] == 64
        if small:
            trainer = PPOTrainer(sim, case["epochs"], case["minibatch"])
            holder = sim
        else:
            trainer = holder = LargePPOTrainer(sim, case["hidden"], case["epochs"], case["minibatch"])
        holder.set("actor", actor)
        holder.set("critic", critic)
        for name, values in _rows(case, seed, actor, critic).items():
            sim.set(name, values.cpu().numpy())
        return dict(kind=kind, sim=sim, trainer=trainer, holder=holder, small=small, done=0)
    if kind == "forward":
        params, obs = _forward_inputs(case, seed)
        return dict(kind=kind, params=params, obs=obs, hidden=case["hidden"])
    advantages = torch.from_numpy(_advantages(case, seed)).cuda()
    return dict(kind=kind, advantages=advantages)


def _forward_inputs(case, seed):
    rng = np.random.default_rng(seed)
    params = _update_policy(case, seed)[0]
    obs = np.clip(0.4 * rng.standard_normal((case["batch"], case["obs"])), -1.5, 1.5).astype(np.float32)
    obs[:, :160] = np.abs(obs[:, :160]).clip(0.0, 1.0)
    return params, obs


def _advantages(case, seed):
    rng = np.random.default_rng(seed)
    return (0.3 + 2.0 * rng.standard_normal(case["count"])).astype(np.float32)


# ---------------------------------------------------------------- one pass
EVAL_FIELDS = ("successes", "collisions", "timeouts", "elapsed", "path", "final_progress", "success_time",
               "peak_speed", "min_clearance")


def run(state):
    kind = state["kind"]
    if kind == "train":
        sim, ppo = state["sim"], state["ppo"]
        sim.collect()
        if state["tasks"]:  # the task training loop rejects bad draws before the update
            sim.validate_rollout()
        ppo.rollout_update(state["done"])
        state["done"] += 1
        return dict(actor=sim.get("actor"), critic=sim.get("critic"), metrics=ppo.metric_mean())
    if kind == "evaluate":
        sim = state["sim"]
        sim.reset()
        sim.collect(state["ticks"])
        runs = sim.get("runs")
        return {f: runs[f] for f in EVAL_FIELDS}
    if kind == "wide":
        sim, lp = state["sim"], state["lp"]
        lp.collect()
        lp.rollout_update(state["done"])
        state["done"] += 1
        return dict(actor=lp.get("actor"), critic=lp.get("critic"), metrics=lp.metric_mean())
    if kind == "update":
        sim, holder = state["sim"], state["holder"]
        state["trainer"].rollout_update(state["done"])
        state["done"] += 1
        out = dict(actor=holder.get("actor"), critic=holder.get("critic"), advantages=sim.get("advantages"))
        if state["small"]:
            out.update(actor_m=sim.get("actor_m"), critic_m=sim.get("critic_m"), returns=sim.get("returns"))
        return out
    if kind == "forward":
        hidden, means = ops.actor_forward(state["params"], state["obs"], state["hidden"])
        return dict(hidden=hidden, means=means)
    a = state["advantages"]
    native.check(native.lib().mdn_op_normalize_noalloc(ctypes.c_void_p(a.data_ptr()), a.numel(),
                                                       ctypes.c_float(1.0e-8),
                                                       ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return a


# ---------------------------------------------------------------- what a pass cannot do without
# Per env-step: the environment step (5 substeps of RAPTOR and RK4, clearance,
# a 320-ray depth frame over 8 boxes and the room, the observation) 117 kFLOP,
# the critic at s and s' 8.7 kFLOP, state and rollout rows 4.34 KB; the
# geometry-prior hint 10.8 kFLOP; the geometry memory 640 points x 85 sweeps x
# ~10 FLOP.
ENV_FLOP, CRITIC_FLOP, ENV_BYTES, HINT_FLOP, MEMORY_FLOP = 117e3, 8.7e3, 4.34e3, 10.8e3, 640 * 45 + 85 * 650 * 10


def _update_work(rows, epochs, d, h):
    params = d * h + 5 * h + 8 + 32 * h + 2 * h + 1
    # forward, weight gradients and hidden deltas per row; each epoch reads
    # every row, GAE and normalisation read and write theirs once
    return dict(flops=epochs * rows * (4.0 * params + 10.0 * h), bytes=epochs * rows * 4.0 * (d + 32 + 8) + 38.0 * rows)


def work(case):
    kind = case["kind"]
    if kind == "train":
        rows, d = case["envs"] * case["ticks"], case["obs"]
        w = _update_work(rows, case["epochs"], d, 64)
        flop = ENV_FLOP + CRITIC_FLOP + 2.0 * (d * 64 + 4 * 64)
        if d == 184:
            flop += MEMORY_FLOP if case["memory"] else HINT_FLOP
        return dict(flops=w["flops"] + rows * flop, bytes=w["bytes"] + rows * ENV_BYTES)
    if kind == "evaluate":
        rows = case["envs"] * case["ticks"]
        return dict(flops=rows * (ENV_FLOP + CRITIC_FLOP + MEMORY_FLOP + 24e3), bytes=rows * ENV_BYTES)
    if kind == "wide":
        rows, h = case["envs"] * case["ticks"], case["hidden"]
        w = _update_work(rows, case["epochs"], 184, h)
        forward = 2.0 * (184 * h + 4 * h + 33 * h)
        return dict(flops=w["flops"] + rows * (ENV_FLOP + HINT_FLOP + forward), bytes=w["bytes"] + rows * ENV_BYTES)
    if kind == "update":
        return _update_work(case["envs"] * case["ticks"], case["epochs"], case["obs"], case["hidden"])
    if kind == "forward":
        b, d, h = case["batch"], case["obs"], case["hidden"]
        return dict(flops=2.0 * b * h * (d + 4), bytes=4.0 * (b * (d + h + 4) + h * (d + 5) + 8))
    return dict(flops=6.0 * case["count"], bytes=8.0 * case["count"])


def _steps(case):
    """Optimiser steps of one pass."""
    rows = case["envs"] * case["ticks"]
    return case["epochs"] * -(-rows // min(case["minibatch"], rows))


def tolerance(case):
    """About four times what the same pass shows when every weight is moved by
    one unit in its last place (a stand-in for sums in another order)."""
    kind = case["kind"]
    if kind == "train":
        # Adam divides each gradient by its own size, so a weight whose
        # gradient is all rounding moves by the learning rate either way:
        # 5e-6 (at worst 1e-4) after a few steps, 2e-3 after 512, 9e-3 after 2,048
        return dict(rel=4e-4, max=0.05) if _steps(case) < 100 else dict(rel=0.03, max=0.35)
    if kind == "evaluate":  # 5e-7 while no episode's outcome flips
        return dict(rel=1e-5, max=1e-4, differ=0.01)
    if kind == "wide":  # bf16 products in the loop: 8e-4
        return dict(rel=4e-3, max=0.1)
    if kind == "update":
        if case["hidden"] != 64:  # bf16 products: 6e-4 from the 64-bit result
            return dict(rel=2e-3, max=0.1)
        return dict(rel=4e-5, max=2e-3) if _steps(case) < 100 else dict(rel=0.02, max=0.2)
    if kind == "forward":  # 2.4e-7 from the 64-bit result
        return dict(rel=1e-6, max=1e-5)
    return dict(rel=5e-7, max=2e-6)


# ---------------------------------------------------------------- 64-bit results
def _actor(p, x, h):
    d = x.shape[1]
    w1, b1 = p[:h * d].reshape(h, d), p[h * d:h * d + h]
    w2, b2 = p[h * d + h:h * d + 5 * h].reshape(4, h), p[h * d + 5 * h:h * d + 5 * h + 4]
    hid = torch.tanh(x @ w1.T + b1)
    mean = hid @ w2.T + b2
    if d == 184:  # the guided actor's hint joins the first three means
        mean = mean + torch.nn.functional.pad(x[:, d - 3:], (0, 1))
    return mean, hid


def _critic(p, x, h):
    w1, b1 = p[:32 * h].reshape(h, 32), p[32 * h:33 * h]
    hid = torch.tanh(x @ w1.T + b1)
    return hid @ p[33 * h:34 * h] + p[34 * h], hid


def _below(words, n):
    """A uniform integer below n from a stream of 32-bit words: the low bits, rejecting."""
    if n <= 1:
        return 0
    mask = (1 << (n - 1).bit_length()) - 1
    while True:
        u = next(words) & mask
        if u < n:
            return u


def _schedule(rows, minibatch, epochs, index):
    """The order of an update's minibatches: contiguous blocks, shuffled
    before the first epoch and again before the second."""
    starts = list(range(0, rows, minibatch))
    twister = np.random.RandomState((0x9e3779b9 + index * 0x85ebca6b) & 0xffffffff)

    def stream():
        while True:
            yield int(twister.randint(0, 1 << 32, dtype=np.uint64))

    words = stream()
    order = []
    for e in range(epochs):
        if e < 2:
            for k in range(len(starts) - 1):
                i = _below(words, len(starts) - k)
                starts[k], starts[k + i] = starts[k + i], starts[k]
        order += starts
    return order


def _adam(p, g, m, v, step, lr):
    g = g * min(1.0, 0.5 / math.sqrt(float((g * g).sum()) + 1e-20))
    m.mul_(0.9).add_(0.1 * g)
    v.mul_(0.999).add_(0.001 * g * g)
    p.sub_(lr * (m / (1.0 - 0.9 ** step)) / ((v / (1.0 - 0.999 ** step)).sqrt() + 1e-8))


def _exact_update(case, seed):
    n, t, d, h = case["envs"], case["ticks"], case["obs"], case["hidden"]
    rows = n * t
    minibatch = min(case["minibatch"], rows)
    actor, critic = _update_policy(case, seed)
    r = {k: x.double() for k, x in _rows(case, seed, actor, critic).items()}
    a, c = torch.from_numpy(actor).cuda().double(), torch.from_numpy(critic).cuda().double()
    am, av, cm, cv = torch.zeros_like(a), torch.zeros_like(a), torch.zeros_like(c), torch.zeros_like(c)
    # generalised advantage estimation, gamma 0.99, lambda 0.95
    shape = {k: r[k].reshape(t, n) for k in ("rewards", "values", "next_values", "terminated", "truncated")}
    adv, carry = torch.zeros(t, n, dtype=torch.float64, device="cuda"), 0.0
    for k in range(t - 1, -1, -1):
        alive = 1.0 - shape["terminated"][k]
        delta = shape["rewards"][k] + 0.99 * shape["next_values"][k] * alive - shape["values"][k]
        carry = delta + 0.99 * 0.95 * alive * (1.0 - shape["truncated"][k]) * carry
        adv[k] = carry
    returns = (adv + shape["values"]).reshape(-1)
    adv = adv.reshape(-1)
    adv = (adv - adv.mean()) / torch.sqrt(adv.var(unbiased=False) + 1e-8)
    at, ct = h * d, 32 * h
    ls0 = at + 5 * h + 4
    for step, lo in enumerate(_schedule(rows, minibatch, case["epochs"], 0), 1):
        hi = min(rows, lo + minibatch)
        b = hi - lo
        x, co, act = r["obs"][lo:hi], r["critic_obs"][lo:hi], r["actions"][lo:hi]
        mean, ha = _actor(a, x, h)
        value, hc = _critic(c, co, h)
        ls = a[ls0:ls0 + 4]
        z = (act - mean) * torch.exp(-ls)
        logp = (-0.5 * (z * z + 2.0 * ls + LOG_TWO_PI)).sum(1)
        ratio = torch.exp((logp - r["logp"][lo:hi]).clamp(-20.0, 20.0))
        ad = adv[lo:hi]
        live = torch.where(ad >= 0, ratio <= 1.2, ratio >= 0.8)
        dlogp = torch.where(live, -ratio * ad, torch.zeros_like(ad)) / b
        dmean = dlogp[:, None] * z * torch.exp(-ls)
        dls = (dlogp[:, None] * (z * z - 1.0)).sum(0) - 0.005
        da = (dmean @ a[at + h:at + 5 * h].reshape(4, h)) * (1.0 - ha * ha)
        ga = torch.cat([(da.T @ x).reshape(-1), da.sum(0), (dmean.T @ ha).reshape(-1), dmean.sum(0), dls])
        dv = 0.5 * (value - returns[lo:hi]) / b
        dc = dv[:, None] * c[ct + h:ct + 2 * h] * (1.0 - hc * hc)
        gc = torch.cat([(dc.T @ co).reshape(-1), dc.sum(0), dv @ hc, dv.sum()[None]])
        _adam(a, ga, am, av, step, 0.0003)
        _adam(c, gc, cm, cv, step, 0.0003)
        a[ls0:ls0 + 4].clamp_(-2.0, 0.5)
    out = dict(actor=a, critic=c, advantages=adv)
    if h == 64:
        out.update(actor_m=am, critic_m=cm, returns=returns)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "update":
        return _exact_update(case, seed)
    if kind == "forward":
        params, obs = _forward_inputs(case, seed)
        mean, hid = _actor(torch.from_numpy(params).double(), torch.from_numpy(obs).double(), case["hidden"])
        return dict(hidden=hid, means=mean)
    if kind == "normalize":
        a = _advantages(case, seed).astype(np.float64)
        return (a - a.mean()) / np.sqrt(a.var() + 1e-8)
    return None  # a simulated trajectory has no plain counterpart
