"""Plants whose forces or torques overflow within a physics step, against the
oracle.  Such a plant is the Crazyflie in units so small that its thrusts lie
near the largest float: the same flight, until a stage of the step overflows.
A step that overflows anywhere is rejected (the env collides), whichever form
of the derivative the device takes for it."""
import sys

import numpy as np
import pytest

from gpu_compare import ENV_BUFFERS, ROW_BUFFERS, config, make_pair
from mdnav import Sim, ops, task_runtime
from oracle_lib import OracleTrainer, crazyflie, oracle, ptr, raptor_fixture

pytestmark = pytest.mark.gpu

# Scale of the plant's force and inertia units: the four rotors together reach
# 0.44 N at full speed and 0.31 N in hover, so the total thrust overflows
# (3.4e38) above 7.7e38 at full speed and above 1.1e39 in hover.  Turning at w,
# the gyroscopic torque w x I w overflows at a scale of about 1e43 / w^2.
SCALES = [3e38, 6e38, 7e38, 7.3e38, 7.6e38, 7.8e38, 1e39]


def say(*args):
    print(*args, flush=True)
    sys.stdout.flush()


def scaled(scale):
    p = crazyflie()
    for f, k in (("rotor_thrust_coefficients", scale), ("inertia", scale), ("mass", scale),
                 ("inertia_inverse", 1.0 / scale)):
        p[f] = (p[f].astype(np.float64) * k).astype(np.float32)
    return p


def same(gpu, ora, names):
    """Equal values, NaN equal to NaN."""
    bad = []
    for name in names:
        a, b = gpu.get(name), ora.get(name)
        for f in a.dtype.names or [None]:
            x, y = (a, b) if f is None else (a[f], b[f])
            if x.dtype.names is None and not np.array_equal(x, y, equal_nan=x.dtype.kind == "f"):
                bad.append((name, f))
    return bad


def states(n, seed):
    rng = np.random.default_rng(seed)
    s = np.zeros(n, [("position", "<f4", 3), ("orientation_wxyz", "<f4", 4), ("linear_velocity", "<f4", 3),
                     ("angular_velocity_body", "<f4", 3), ("rpm", "<f4", 4)])
    s["position"] = rng.normal(0, 2, (n, 3))
    q = rng.normal(size=(n, 4))
    s["orientation_wxyz"] = q / np.linalg.norm(q, axis=1)[:, None]
    s["linear_velocity"] = rng.normal(0, 2, (n, 3))
    s["angular_velocity_body"] = rng.normal(0, 1, (n, 3)) * 10.0 ** rng.uniform(0, 4, (n, 1))
    s["rpm"] = rng.uniform(0.5, 1.0, (n, 4))
    return s


@pytest.mark.parametrize("scale", SCALES)
def test_step_overflow(scale):
    say("case: physics step, force unit", scale)
    n, p = 4096, scaled(scale)
    s = states(n, 1)
    rng = np.random.default_rng(2)
    action, wind = rng.uniform(-1, 1, (n, 4)).astype(np.float32), np.zeros((n, 3), np.float32)
    want = np.zeros_like(s)
    oracle().orc_physics_step_batch(ptr(s), ptr(action), ptr(wind), ptr(p), ptr(want), n)
    got = ops.physics_step(s, action, wind, p)
    for f in s.dtype.names:
        assert np.array_equal(got[f], want[f], equal_nan=True), f
    # steps of which only the last stage overflowed are among them
    late = np.isfinite(want["orientation_wxyz"]).all(1) & np.isnan(want["linear_velocity"]).any(1)
    assert late.any() and np.isfinite(want["linear_velocity"]).all(1).any()


def _fly(sim, ora, ticks, n, rates=2.7):
    rng = np.random.default_rng(n)
    spin = (rng.normal(0, 1, (n, 3)) * 10.0 ** rng.uniform(0, rates, (n, 1))).astype(np.float32)
    s = sim.get("states")
    s["angular_velocity_body"] = spin
    rejected = 0
    for x in (sim, ora):
        x.set("states", s)
    for _ in range(ticks):
        before = ora.get("runs")["collisions"].sum()
        sim.collect(1)
        sim.sync()
        ora.collect(1)
        rejected += ora.get("runs")["collisions"].sum() - before
        bad = same(sim, ora, ENV_BUFFERS + ROW_BUFFERS)
        assert not bad, bad
    assert 0 < rejected


@pytest.mark.parametrize("scale", SCALES[:5])
@pytest.mark.parametrize("n", [48, 4100])
def test_fleet_plant_overflow(n, scale):
    """The launch's plant, in the small-fleet and the large-fleet rollout."""
    say("case: fleet of", n, "force unit", scale)
    cfg = config(n=n, family=1, seed=4, speed=1.0, distance=3.0, max_steps=400)
    weights = raptor_fixture()[0]
    p = scaled(scale)
    sim, ora = Sim(cfg, 1, raptor=weights, physics=p), OracleTrainer(cfg, 1, weights, physics=p)
    _fly(sim, ora, 4, n)


@pytest.mark.parametrize("obs,delay", [(181, 0), (181, 2), (184, 0)])
@pytest.mark.parametrize("n", [48, 4100])
def test_fleet_state_overflow(n, obs, delay):
    """The Crazyflie turning at up to 1e6 rad/s, where its torques overflow
    from about 1e4 on."""
    say("case: fleet of", n, "inputs", obs, "delay", delay, "high body rates")
    cfg = config(n=n, family=1, seed=4, speed=1.0, distance=3.0, max_steps=400, sensor_delay=delay)
    sim, _, ora = make_pair(cfg, 1, actor_obs=obs)
    for name in ("actor", "critic"):
        ora.set(name, sim.get(name))
    _fly(sim, ora, 4, n, rates=6)


@pytest.mark.parametrize("n", [48, 1500])
def test_episode_plant_overflow(n):
    """Plants uploaded per env, overflowing or not, side by side in a wavefront."""
    say("case: uploaded plants of several force units, fleet of", n)
    cfg = config(n=n, family=1, seed=4, speed=1.0, distance=3.0, max_steps=400)
    sim, _, ora = make_pair(cfg, 1)
    for x in (sim, ora):
        x.set_runtime(task_runtime(1.0))
        x.set("actor", sim.get("actor"))
        x.set("critic", sim.get("critic"))
        x.reset()
    plants = sim.get("environment_physics")
    for e in range(n):
        plants[e] = scaled((1.0, *SCALES)[e % (1 + len(SCALES))])
    for x in (sim, ora):
        x.set("environment_physics", plants)
    _fly(sim, ora, 4, n)
