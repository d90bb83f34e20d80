"""The rollout instances of fleets above 4,096 envs (32 envs per workgroup),
which the smaller fleets of the other tests do not reach: every ring size, actor
width and kind of plant, fused, one launch per tick and with the wide policy's
means, against the oracle at tolerance 0.  The same with a small fleet where the
other tests leave an instance out."""
import sys

import numpy as np
import pytest

from gpu_compare import ENV_BUFFERS, ROW_BUFFERS, compare, config
from mdnav import LargePPOTrainer, Sim
from oracle_lib import OracleTrainer, crazyflie, raptor_fixture

pytestmark = pytest.mark.gpu

N = 4100


def say(*args):
    print(*args, flush=True)
    sys.stdout.flush()


def _plant(kind):
    p = crazyflie().copy()
    if kind == "heavier":  # standard structure, not the Crazyflie
        p["mass"] = np.float32(p["mass"] * np.float32(1.1))
    elif kind == "tilted":  # general derivative
        p["rotor_thrust_directions"][:3] = np.array([0.05, 0.0, 0.99875], np.float32)
    return p


def _pair(cfg, ticks, obs, plant):
    weights, p = raptor_fixture()[0], _plant(plant)
    sim = Sim(cfg, ticks, raptor=weights, physics=p, actor_obs=obs)
    ora = OracleTrainer(cfg, ticks, weights, physics=p)
    if obs != 181:
        ora.set_actor_obs(obs)
    return sim, ora


def _rollout(cfg, ticks, obs, plant="crazyflie"):
    sim, ora = _pair(cfg, ticks, obs, plant)
    for name in ("actor", "critic"):
        ora.set(name, sim.get(name))
    for count in (ticks, ticks - 1):
        sim.collect(count)
        sim.sync()
        ora.collect(count)
        bad = compare(sim, ora, ENV_BUFFERS + ROW_BUFFERS)
        assert not bad, bad
    assert ora.get("runs")["episodes"].sum() > 0


@pytest.mark.parametrize("plant", ["crazyflie", "heavier", "tilted"])
@pytest.mark.parametrize("obs,delay,memory", [(181, 0, 0), (181, 2, 0), (181, 6, 0), (184, 0, 0), (184, 2, 0),
                                              (184, 6, 0), (184, 0, 1)])
def test_rollout(obs, delay, memory, plant):
    say("case: fleet of", N, "inputs", obs, "delay", delay, "memory", memory, "plant", plant)
    cfg = config(n=N, family=13 if delay else 1, seed=21, speed=1.5, distance=4.0, max_steps=4, sensor_delay=delay,
                 command_delay=delay, geometry_memory=memory)
    _rollout(cfg, 6, obs, plant)


@pytest.mark.parametrize("obs", [181, 184])
@pytest.mark.parametrize("variant", ["eval", "noise", "period2", "wind", "deployed"])
def test_variants(variant, obs):
    kw = dict(n=N, family=1, seed=22, speed=1.0, distance=3.0, max_steps=4)
    if variant == "eval":
        kw.update(eval=1)
    elif variant == "noise":
        kw.update(depth_noise=0.05, dropout=0.1)
    elif variant == "period2":
        kw.update(sensor_period=2, sensor_delay=1, command_delay=1)
    elif variant == "wind":
        kw.update(wind=0.5, family=6)
    elif variant == "deployed":  # the deployed map of the guided actor
        kw.update(mode=22, family=3)
    say("case: fleet of", N, "inputs", obs, "variant", variant)
    _rollout(config(**kw), 6, obs)


@pytest.mark.parametrize("n,plant", [(N, "crazyflie"), (N, "heavier"), (48, "crazyflie")])
@pytest.mark.parametrize("obs", [181, 184])
@pytest.mark.parametrize("delay", [0, 2, 6])
def test_wide_policy(delay, obs, n, plant):
    """The split launches around the wide policy; its means go to the oracle."""
    hidden, ticks = 128, 6
    say("case: wide closed loop, fleet of", n, "inputs", obs, "delay", delay, "plant", plant)
    cfg = config(n=n, family=13 if delay else 1, seed=23, speed=1.5, distance=4.0, max_steps=4, sensor_delay=delay,
                 command_delay=delay, geometry_memory=int(obs == 184 and delay == 2))
    sim, ora = _pair(cfg, ticks, obs, plant)
    lp = LargePPOTrainer(sim, hidden, epochs=1, minibatch=8192)
    ora.set_hidden(hidden)
    for _ in range(2):
        lp.collect()
        sim.sync()
        ora.set_ext_means(lp.means())
        ora.collect()
        ora.set_ext_means(None)
        bad = compare(sim, ora, ENV_BUFFERS + [b for b in ROW_BUFFERS if b not in ("values", "next_values")])
        assert not bad, bad
    assert ora.get("runs")["episodes"].sum() > 0
