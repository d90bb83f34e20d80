"""The sizes at which a kernel or its split of the work changes, against the
oracle at tolerance 0: fleets around the small-fleet rollout's envs per
wavefront (1,024 envs each) and its limit (4,096), with every ring size, the
guided actor and per-episode plants; minibatches around the few-chunk limit;
advantage normalisation around a chunk, a group and the one-workgroup limit;
the geometry memory either side of its wide workgroups."""
import ctypes
import sys

import numpy as np
import pytest

from gpu_compare import ENV_BUFFERS, ROW_BUFFERS, compare, config, make_pair
from mdnav import LargePPOTrainer, Sim, native, ops, task_runtime, task_settings
from oracle_lib import oracle, ptr

pytestmark = pytest.mark.gpu


def say(*args):
    print(*args, flush=True)
    sys.stdout.flush()


def _collect_both(sim, ora, ticks, extra=()):
    ora.set("actor", sim.get("actor"))
    ora.set("critic", sim.get("critic"))
    sim.reset()
    ora.reset()
    for count in (ticks, ticks - 1):
        sim.collect(count)
        sim.sync()
        ora.collect(count)
        bad = compare(sim, ora, ENV_BUFFERS + ROW_BUFFERS + list(extra))
        assert not bad, bad


@pytest.mark.parametrize("n", [1, 3, 5, 1024, 1025, 2048, 2049, 3071, 3073, 4096, 4097])
def test_fleet_sizes(n):
    say("case: fleet of", n)
    sim, _, ora = make_pair(config(n=n, family=1, seed=n, max_steps=3, speed=1.0, distance=3.0), 5)
    _collect_both(sim, ora, 5)


@pytest.mark.parametrize("n", [37, 1030, 4100])
@pytest.mark.parametrize("delay", [2, 6])
@pytest.mark.parametrize("obs,memory", [(181, 0), (184, 0), (184, 1)])
def test_fleet_ring_sizes(n, delay, obs, memory):
    say("case: fleet of", n, "sensor delay", delay, "inputs", obs, "memory", memory)
    cfg = config(n=n, family=13, seed=5, max_steps=6, sensor_delay=delay, command_delay=delay, speed=1.5, distance=4.0,
                 geometry_memory=memory)
    sim, _, ora = make_pair(cfg, 10, actor_obs=obs)
    _collect_both(sim, ora, 10)


@pytest.mark.parametrize("n,delay,obs", [(1, 0, 184), (1026, 0, 184), (130, 2, 181), (130, 6, 184), (4099, 0, 181)])
def test_fleet_plants_and_tasks(n, delay, obs):
    say("case: per-episode plants and tasks, fleet of", n, "sensor delay", delay, "inputs", obs)
    cfg = config(n=n, family=12, seed=9, sensor_delay=delay, geometry_memory=int(obs == 184), speed=1.5, distance=8.0,
                 max_steps=400)
    sim, _, ora = make_pair(cfg, 6, actor_obs=obs)
    rt, t = task_runtime(1.0), task_settings(2, 12)
    t["config"]["max_nav_steps"] = 4
    for x in (sim, ora):
        x.set_runtime(rt)
        x.set_tasks(t)
    _collect_both(sim, ora, 6, ["environment_physics", "task_states"])


def test_fleet_plants_of_any_structure():
    """Per-episode plants the host uploads: standard structure in some
    wavefronts (the specialised derivative), a tilted rotor, an off-diagonal
    inertia or a -0 in others (the general one)."""
    say("case: uploaded plants, standard and not")
    cfg = config(n=48, family=1, seed=4, speed=1.0, distance=3.0, max_steps=400)
    sim, _, ora = make_pair(cfg, 6)
    rt = task_runtime(1.0)
    for x in (sim, ora):
        x.set_runtime(rt)
        x.set("actor", sim.get("actor"))
        x.set("critic", sim.get("critic"))
        x.reset()
    plants = sim.get("environment_physics")
    plants["rotor_thrust_directions"][5, 3:6] = [0.1, 0.0, 0.99]
    plants["inertia"][11, 1] = 1e-7
    plants["rotor_positions"][17, 2] = -0.0
    plants["gravity_world"][23, 0] = 0.5
    plants["rotor_torque_directions"][29, 2] = 0.9
    for x in (sim, ora):
        x.set("environment_physics", plants)
        x.collect(6)
    sim.sync()
    bad = compare(sim, ora, ENV_BUFFERS + ROW_BUFFERS + ["environment_physics"])
    assert not bad, bad


@pytest.mark.parametrize("n", [2048, 2049])
def test_memory_workgroups(n):
    say("case: geometry memory, fleet of", n)
    cfg = config(n=n, family=12, seed=11, speed=1.5, distance=4.0, geometry_memory=1)
    sim, _, ora = make_pair(cfg, 9, actor_obs=184)
    _collect_both(sim, ora, 9)


@pytest.mark.parametrize("dt", [0.05, 5.0, 500.0, 5e3, 5e5])
def test_memory_point_radius(dt):
    """Remembered points of every age: a point's sphere grows by 0.15 m a
    second, so a slow sensor gives spheres of kilometres around points near
    the body, and their contacts start at along = 0 to the last bit."""
    say("case: geometry memory, sensor interval", dt)
    n, period = 512, int(round(dt / 0.05))
    cfg = config(n=n, family=1, seed=13, speed=1.0, distance=3.0, geometry_memory=1, sensor_period=period,
                 max_steps=1 << 30)
    sim, _, ora = make_pair(cfg, 1, actor_obs=184)
    ora.set("actor", sim.get("actor"))
    ora.set("critic", sim.get("critic"))
    sim.reset()
    ora.reset()
    rng = np.random.default_rng(13)
    runs, poses = sim.get("runs"), sim.get("poses").reshape(n, 8, 12)
    runs["steps"] = 7 * period + (1 if period > 1 else 0)  # eight frames held, none due unless every tick has one
    sensors = np.full((n, 8, 320), 12.0, np.float32)
    frame, pixel = rng.integers(0, 7, n), rng.integers(0, 320, n)
    sensors[np.arange(n), frame, pixel] = rng.uniform(0.011, 0.05, n)  # one hit per env, centimetres away
    poses[:, :, :3] = sim.get("states")["position"][:, None] + rng.uniform(-0.03, 0.03, (n, 8, 3))
    poses[:, :, 3:] = np.eye(3, dtype=np.float32).reshape(9)
    for x in (sim, ora):
        x.set("runs", runs)
        x.set("sensors", sensors)
        x.set("poses", poses)
        x.collect(1)
    sim.sync()
    bad = compare(sim, ora, ENV_BUFFERS + ROW_BUFFERS)
    assert not bad, bad


@pytest.mark.parametrize("obs", [181, 184])
@pytest.mark.parametrize("n,T,minibatch", [(257, 1, 257), (64, 8, 512), (100, 83, 4150), (2048, 10, 20480),
                                           (20481, 1, 20481)])
def test_few_chunk_minibatches(obs, n, T, minibatch):
    """One chunk more than the single-chunk path, two chunks, an odd last
    chunk in two minibatches, the most chunks of the few-chunk path and one
    more (the chunk kernel); the update is the oracle's bit for bit."""
    say("case: update of %d x %d rows, minibatches of %d, %d inputs" % (n, T, minibatch, obs))
    sim, ppo, ora = make_pair(config(n=n, family=1, seed=3, max_steps=7), T, epochs=2, minibatch=minibatch,
                              actor_obs=obs)
    rng = np.random.default_rng(n)
    for name in ("actor", "critic"):
        w = sim.get(name)
        w *= (1.0 + 0.1 * rng.standard_normal(w.size)).astype(np.float32)
        sim.set(name, w)
        ora.set(name, w)
    sim.collect()
    ora.collect()
    for it in range(2):
        ppo.rollout_update(it)
        ora.gae()
        ora.normalize()
        ora.update(it)
    names = ["actor", "critic", "actor_m", "actor_v", "critic_m", "critic_v", "advantages", "returns", "metric_rows",
             "grad_norm_rows"]
    bad = compare(sim, ora, names)
    assert not bad, bad
    assert np.array_equal(ppo.metric_mean(), ora.metric_mean())
    # the rollout's transposed first layers follow the update
    sim.collect()
    ora.collect()
    bad = compare(sim, ora, ENV_BUFFERS + ROW_BUFFERS)
    assert not bad, bad


@pytest.mark.parametrize("updates", [1, 15, 256, 257, 530])
def test_metric_mean_rows(updates):
    say("case: metric mean over", updates, "updates")
    sim, ppo, ora = make_pair(config(n=updates, family=1, seed=3), 3, epochs=1, minibatch=3)
    sim.collect()
    ppo.rollout_update(0)
    rows = sim.get("metric_rows").reshape(updates, 4)
    want = np.zeros(4, np.float32)
    for r in rows:
        want = want + r
    assert np.array_equal(ppo.metric_mean(), want / np.float32(updates))


@pytest.mark.parametrize("count", [1, 2, 255, 256, 257, 4097, 16383, 16384, 16385, 32767, 32768, 32769, 65537])
def test_normalize_sizes(count):
    from test_zz_no_alloc import hip_runtime
    say("case: normalise", count, "values")
    rng = np.random.default_rng(count)
    x = rng.normal(3, 5, count).astype(np.float32)
    want = x.copy()
    oracle().orc_normalize_advantages(ptr(want), count, np.float32(1e-8))
    assert np.array_equal(ops.normalize(x), want)
    # device memory at every 4-byte alignment, with values before and after left alone
    hip = hip_runtime()
    for offset in (0, 1, 2, 3):
        host = np.full(count + 8, 7.0, np.float32)
        host[offset:offset + count] = x
        dev = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(dev), host.nbytes) == 0
        assert hip.hipMemcpy(dev, ptr(host), host.nbytes, 1) == 0
        native.check(native.lib().mdn_op_normalize_noalloc(ctypes.c_void_p(dev.value + 4 * offset), count, 1e-8, None))
        assert hip.hipMemcpy(ptr(host), dev, host.nbytes, 2) == 0
        assert hip.hipFree(dev) == 0
        assert np.array_equal(host[offset:offset + count], want), offset
        assert np.all(host[:offset] == 7.0) and np.all(host[offset + count:] == 7.0)


def _order(rows, minibatch, epochs, rollout):
    out = np.zeros(-(-rows // minibatch) * epochs, np.uint32)
    oracle().orc_minibatch_schedule(rows, minibatch, epochs, rollout, ptr(out))
    return out.tolist()


@pytest.mark.parametrize("hidden", [128, 384])
@pytest.mark.parametrize("n,minibatch", [(50, 500), (50, 260), (61, 200)])
def test_wide_epochs(n, minibatch, hidden):
    """The wide update keeps its prepared rows from the first epoch on: three
    epochs equal three one-epoch updates in the same orders bit for bit (one
    minibatch, two and four, ragged last ones), and so does a second update on
    other rows."""
    say("case: wide update of", n, "x 10 rows, minibatches of", minibatch, "hidden", hidden)
    T, epochs = 10, 3
    cfg = config(n=n, family=1, seed=7, max_steps=6)
    sims = [Sim(cfg, T, actor_obs=184) for _ in range(2)]
    a, b = LargePPOTrainer(sims[0], hidden, epochs, minibatch), LargePPOTrainer(sims[1], hidden, 1, minibatch)
    per = -(-n * T // minibatch)
    for rollout in range(2):
        a.collect()
        b.collect()
        a.rollout_update(rollout)
        order = _order(n * T, minibatch, epochs, rollout)
        for e in range(epochs):
            want = order[per * e:per * (e + 1)]
            b.rollout_update(next(r for r in range(10000) if _order(n * T, minibatch, 1, r) == want))
        assert a.optimizer_step == b.optimizer_step == per * epochs * (rollout + 1)
        for name in ("actor", "critic", "actor_m", "actor_v", "critic_m", "critic_v"):
            assert np.array_equal(a.get(name), b.get(name)), (rollout, name)


@pytest.mark.parametrize("n,minibatch", [(20, 50), (5, 20), (13, 63), (24, 60)])
def test_wide_epochs_in_turn(n, minibatch):
    """The same with one minibatch's buffers serving every minibatch in turn:
    rows whose padding to 128 would take more than they do are not kept."""
    test_wide_epochs(n, minibatch, 128)


def test_wide_small_minibatch_memory():
    """Rows of tiny minibatches are not kept padded: 65,536 of them in pairs
    would take 3.8 GB, the trainer's other buffers a few MB."""
    from test_zz_no_alloc import hip_runtime
    say("case: wide trainer, 65,536 rows in minibatches of 2")
    hip = hip_runtime()
    hip.hipMemGetInfo.argtypes = [ctypes.POINTER(ctypes.c_size_t)] * 2
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    sim = Sim(config(n=4096, family=1, seed=7), 16, actor_obs=184)
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    before = free.value
    p = LargePPOTrainer(sim, 128, 3, 2)
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    assert before - free.value < 256 << 20, before - free.value
    p.close()


def _mlp(d, h, b, seed, special):
    rng = np.random.default_rng(seed)
    w = rng.normal(0, 0.3, h * d + h + 4 * h + 8).astype(np.float32)
    x = rng.uniform(-1, 1, (b, d)).astype(np.float32)
    if special:  # signed zeros, subnormals, infinities and NaN in inputs and weights
        x.flat[::7] = -0.0
        x.flat[3::11] = 1e-41
        w[5::13] = -0.0
        w[2::17] = 3e-42
        if b > 2:
            x[1, d // 2] = np.inf
            x[2, d - 1] = np.nan
    return w, x


@pytest.mark.parametrize("d,h,b", [(3, 7, 5), (181, 64, 17), (184, 64, 16), (200, 130, 20)])
def test_forward_subnormal_sums(d, h, b):
    """Inputs and weights so small that every product, partial sum and
    activation is subnormal: none is flushed to zero."""
    say("case: forward,", b, "rows", d, "inputs", h, "units, subnormal sums")
    w, x = _mlp(d, h, b, d, 0)
    w[:h * d + h] *= np.float32(1e-20)
    w[h * d:h * d + h] *= np.float32(1e-20)
    x *= np.float32(1e-20)
    ho, mo = np.zeros((b, h), np.float32), np.zeros((b, 4), np.float32)
    oracle().orc_actor_forward_batch(ptr(w), ptr(x), d, h, b, ptr(ho), ptr(mo))
    tiny = np.finfo(np.float32).tiny
    assert np.all(np.abs(ho) < tiny) and np.count_nonzero(ho) > ho.size // 2
    hid, mean = ops.actor_forward(w, x, hidden_dim=h)
    assert np.array_equal(hid, ho) and np.array_equal(mean, mo)


@pytest.mark.parametrize("special", [0, 1])
@pytest.mark.parametrize("d,h,b", [(1, 1, 1), (2, 5, 3), (4, 64, 16), (181, 64, 17), (184, 63, 33), (191, 65, 15),
                                   (193, 128, 31), (192, 256, 16), (385, 257, 20), (824, 320, 18), (1024, 512, 1)])
def test_forward_sizes(d, h, b, special):
    say("case: forward,", b, "rows", d, "inputs", h, "units, special", special)
    w, x = _mlp(d, h, b, d + h + b, special)
    ho, mo = np.zeros((b, h), np.float32), np.zeros((b, 4), np.float32)
    oracle().orc_actor_forward_batch(ptr(w), ptr(x), d, h, b, ptr(ho), ptr(mo))
    if d == 824:  # the oracle adds the hint at 184 inputs only
        mo[:, :3] += x[:, -3:]
    hid, mean = ops.actor_forward(w, x, hidden_dim=h)
    assert np.array_equal(hid, ho, equal_nan=True) and np.array_equal(mean, mo, equal_nan=True)
    if d in (184, 824):
        return  # a critic has no hint to add
    # a critic whose output row is the actor's first
    c = np.concatenate([w[:h * d + 2 * h], w[h * d + 5 * h:h * d + 5 * h + 1]])
    hid, value = ops.critic_forward(c, x, hidden_dim=h)
    assert np.array_equal(hid, ho, equal_nan=True) and np.array_equal(value, mo[:, 0], equal_nan=True)
