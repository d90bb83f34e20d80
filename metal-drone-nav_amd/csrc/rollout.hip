// rollout.hip — resets, per-episode work, the rollout instances for fleets
// that fill the GPU (rollout_small.hip has the others), their launchers and
// the RAPTOR fixture.
#include "rollout_kernel.h"

namespace nav {

// First reset of every env (sim_reset kernel, sim.metal:142-144): one
// thread per env, writes straight to the global buffers.
__global__ __launch_bounds__(64) void reset_kernel(RolloutArgs a) {
    const uint32_t n = blockIdx.x * 64 + threadIdx.x;
    const uint32_t N = a.cfg.n;
    if (n >= N) return;
    State s;
    Run r;
    load_run(a.run, N, n, r);
    uint32_t rng = 0, family = 0, seed = 0;
    reset_draw(a.cfg, n, true, rng, family, seed);
    float* world = a.world + size_t(n) * WORLD_WORDS;
    WorldGen wg{world};
    wg.generate(seed, family, a.cfg.distance);
    reset_apply(a.cfg, a.phys, a.raptor, n, true, rng, world, s, r);
    store_state(a.state, N, n, s, 0, 1);
    store_run(a.run, N, n, r, 0, 1);
    for (uint32_t j = 0; j < 8 * PIX; j++) a.sensors[size_t(n) * 8 * PIX + j] = 12.0f;
    for (uint32_t j = 0; j < 32; j++) a.commands[size_t(n) * 32 + j] = 0.0f;
    for (uint32_t j = 0; j < 96; j++) a.poses[size_t(n) * 96 + j] = 0.0f;
}

// Per-episode work of the envs whose episode just began, one thread per env:
// the episode's plant (sim.metal:62-69, with its hover rpm 70-81), its
// challenge-bank world (sim.metal:95-121) and its navigation task
// (sim.metal:122-141: world, start state, yaw, reference point, desired
// velocity, initial distance, wind), in the reference's order.  Runs after the reset
// kernel (first: every env) and after each launch that may reset envs (an
// env with steps == 0 was reset by it; an evaluation never restarts one).
// One wavefront per env: every lane computes the same values (and stores
// the same words), except the task generator's segment clearances, whose
// samples the lanes share.  The workgroup is that one wavefront, so the
// plant, its draw, the task state and the witness path live in its LDS.
__global__ __launch_bounds__(64) void episode_kernel(EpisodeArgs a) {
    const uint32_t n = blockIdx.x;
    const uint32_t N = a.cfg.n;
    if (n >= N) return;  // uniform over the wavefront
    Run r;
    load_run(a.run, N, n, r);
    if (!a.first && r.steps != 0u) return;
    State s;
    load_state(a.state, N, n, s);
    // the plant and its draw live in the wavefront's LDS (88 words each, the
    // same values from every lane), not in registers
    __shared__ MdnPhysicsParams s_ep, s_varied;
    MdnPhysicsParams& ep = s_ep;
    ep = a.phys;
    if (a.runtime.enabled != 0u && a.runtime.domain_amplitude > 0.0f) {
        const uint32_t rng = dom_seed(a.runtime, a.cfg.seed, n, a.first ? 0u : r.episodes);
        if (dom_sample(a.phys, rng, a.runtime.domain_amplitude, a.runtime.domain_range, s_varied)) ep = s_varied;
        else ep.mass = nan_f();  // rejected draw: the host's validation reports it
    }
    a.env_phys[n] = ep;
    if (a.runtime.enabled != 0u) {
        const float target = ep.mass * 9.81f / 4;
        for (int q = 0; q < 4; q++) {
            const float c0 = ep.rotor_thrust_coefficients[3 * q], c1 = ep.rotor_thrust_coefficients[3 * q + 1],
                        c2 = ep.rotor_thrust_coefficients[3 * q + 2];
            const float disc = c1 * c1 - 4 * c2 * (c0 - target);
            s.rpm[q] = disc >= 0.0f ? clamp_f((-c1 + sqrt_f(disc)) / (2 * c2), ep.action_min, ep.action_max)
                                    : ep.action_max;
        }
    }
    float* world = a.world + size_t(n) * WORLD_WORDS;
    if (a.bank.enabled != 0u) {  // sim.metal:95-121
        if (a.bank.bank_count != 0u && a.slot < a.bank.schedule_stride) {
            const uint32_t level = a.bank_schedule[size_t(n) * a.bank.schedule_stride + a.slot];
            bool apply = true;
            if (level == MDN_BANK_REHEARSAL) {  // alternating static / moving-threat rehearsal
                uint32_t rng = r.rng;
                const uint32_t family = training_family(n % 2 == 0 ? 12u : 13u, rng);
                const uint32_t seed = xs(rng);
                WorldGen{world}.generate(seed, family, 4.0f);
                r.rng = rng;
            } else if (level < a.bank.bank_count) {
                const float* src = a.bank_worlds + size_t(level) * WORLD_WORDS;
                for (uint32_t i = 0; i < WORLD_WORDS; i++) world[i] = src[i];
            } else {
                apply = false;
            }
            if (apply) {
                world[166] = clean_env(a.cfg, n) ? 0.0f : a.cfg.wind;
                world[167] = 0.0f;
                world[168] = 0.0f;
                const float gx = world[163], gy = world[164], gz = world[165] - 1.5f;
                r.initial_distance = sqrt_f(gx * gx + gy * gy + gz * gz);
                const uint32_t wfam = float_bits(world[162]);
                if (wfam == 10u || wfam == 11u) {
                    s.v[0] = a.cfg.speed;
                    r.desired_vel[0] = a.cfg.speed;
                    r.prev_nav[0] = 1.0f;
                }
                a.bank_active[n] = level;
            }
        }
    } else {
        a.bank_active[n] = MDN_BANK_REHEARSAL;
    }
    __shared__ MdnTaskState s_task;  // in LDS like the plant
    MdnTaskState& t = s_task;
    uint32_t* tw = reinterpret_cast<uint32_t*>(&t);
    for (uint32_t i = 0; i < sizeof(MdnTaskState) / 4; i++) tw[i] = 0u;
    if (a.task.enabled != 0u) {
        uint32_t rng = a.cfg.seed ^ ((n + 1u) * 0x27d4eb2du) ^ ((r.episodes + 1u) * 0x165667b1u);
        task_generate(world, t, rng, a.task.config);
        if (t.valid != 0u) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                s.p[k] = t.start_position[k];
                s.v[k] = t.start_velocity_world[k];
                s.w[k] = 0.0f;
            }
            float sh, ch;
            sincos_f(t.start_yaw_rad * 0.5f, &sh, &ch);
            s.q[0] = ch; s.q[1] = 0.0f; s.q[2] = 0.0f; s.q[3] = sh;
            r.yaw = t.start_yaw_rad;
            r.initial_distance = t.initial_distance_m;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                r.ref_pos[k] = s.p[k];
                r.desired_vel[k] = s.v[k];
            }
            world[166] = clean_env(a.cfg, n) ? 0.0f : a.cfg.wind;
            world[167] = 0.0f;
            world[168] = 0.0f;
        }
    }
    a.task_states[n] = t;
    store_state(a.state, N, n, s, 0, 1);
    store_run(a.run, N, n, r, 0, 1);
}

// navigation_training::validate_rollout (navigation_training.hpp:27-35): the
// lowest env whose task is not valid and ready (out[0]) and the lowest whose
// plant mass is not finite and positive (out[1]); 0xffffffff when none.  The
// caller fills out with 0xffffffff first.
__global__ __launch_bounds__(256) void validate_kernel(const MdnTaskState* __restrict__ tasks,
                                                       const MdnPhysicsParams* __restrict__ phys, uint32_t n,
                                                       uint32_t* __restrict__ out) {
    const uint32_t e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const MdnTaskState& t = tasks[e];
    if (!(t.valid != 0u && t.generation_status == MDN_TASK_READY)) atomicMin(out, e);
    const float m = phys[e].mass;
    if (!(isfinite_f(m) && m > 0.0f)) atomicMin(out + 1, e);
}

}  // namespace nav

// ---------------------------------------------------------------- launchers
extern "C" {

hipError_t nav_launch_validate(const MdnTaskState* tasks, const MdnPhysicsParams* phys, uint32_t n, uint32_t* out,
                               hipStream_t stream) {
    hipError_t e = hipMemsetAsync(out, 0xff, 8, stream);
    if (e != hipSuccess || n == 0) return e;
    hipLaunchKernelGGL(nav::validate_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, tasks, phys, n, out);
    return hipGetLastError();
}

hipError_t nav_launch_episode(const nav::EpisodeArgs* a, hipStream_t stream) {
    if (a->cfg.n == 0) return hipSuccess;
    hipLaunchKernelGGL(nav::episode_kernel, dim3(a->cfg.n), dim3(64), 0, stream, *a);
    return hipGetLastError();
}

hipError_t nav_launch_reset(const nav::RolloutArgs* a, hipStream_t stream) {
    const uint32_t blocks = (a->cfg.n + 63) / 64;
    hipLaunchKernelGGL(nav::reset_kernel, dim3(blocks), dim3(64), 0, stream, *a);
    return hipGetLastError();
}

// Lanes per env G and pooled ring slots K are compile-time; K = sensor_delay+2
// rounded up to 2, 4 or 8.
// The 8-lane cases run four wavefronts per workgroup with the weights in LDS
// (32 envs, one workgroup per CU); with 4 or 8 slots the pooled ring lives in
// HBM (a.pool_ring), except in the small-fleet instances.  16 and 4 lanes per
// env run one wavefront per workgroup with the weights in L1/L2.
// Split ticks (a->ext_means set) and 184-input actors are built for 8 lanes
// per env only.
// 8-lane fleets of at most nav::SMALL_FLEET envs, and every launch with
// per-episode plants or tasks, take the small-fleet instances
// (rollout_small.hip).
hipError_t nav_launch_rollout(const nav::RolloutArgs* a, int lanes_per_env, int ring_slots, uint32_t actor_obs,
                              hipStream_t stream) {
    const bool dyn = a->env_phys != nullptr;
    if (lanes_per_env == 8 && (dyn || a->cfg.n <= nav::SMALL_FLEET))
        return nav_launch_rollout_small(a, ring_slots, actor_obs, stream);
    if (dyn) return hipErrorInvalidValue;  // per-episode plants run 8 lanes per env
    constexpr uint32_t P = MDN_ACTOR_OBS_POOLED, H = MDN_ACTOR_OBS_PRIOR;
    // the Crazyflie plant as compile-time constants (the common plant of the
    // 8-lane instances with two ring slots, fused or split)
    const bool cf = std::memcmp(&a->phys, &mdn::kCrazyflie, sizeof(MdnPhysicsParams)) == 0;
#define NAV_ROLLOUT_CASE(COND, G, K, W, X, D, CF)                                                              \
    if (COND && lanes_per_env == G && ring_slots == K && (a->ext_means != nullptr) == X && actor_obs == D) {   \
        const uint32_t blocks = (a->cfg.n + 64 * W / G - 1) / (64 * W / G);                                    \
        hipLaunchKernelGGL((nav::rollout_kernel<G, K, W, X, D, false, CF>), dim3(blocks), dim3(64 * W), 0,     \
                           stream, *a);                                                                        \
        return hipGetLastError();                                                                              \
    }
    NAV_ROLLOUT_CASE(cf, 8, 2, 4, false, P, true) NAV_ROLLOUT_CASE(cf, 8, 4, 4, false, P, true)
    NAV_ROLLOUT_CASE(cf, 8, 2, 4, false, H, true)
    NAV_ROLLOUT_CASE(cf, 8, 2, 4, true, P, true) NAV_ROLLOUT_CASE(cf, 8, 2, 4, true, H, true)
    NAV_ROLLOUT_CASE(true, 8, 2, 4, false, P, false) NAV_ROLLOUT_CASE(true, 8, 4, 4, false, P, false)
    NAV_ROLLOUT_CASE(true, 8, 8, 4, false, P, false)
    NAV_ROLLOUT_CASE(true, 16, 2, 1, false, P, false) NAV_ROLLOUT_CASE(true, 16, 4, 1, false, P, false)
    NAV_ROLLOUT_CASE(true, 16, 8, 1, false, P, false)
    NAV_ROLLOUT_CASE(true, 4, 2, 1, false, P, false) NAV_ROLLOUT_CASE(true, 4, 4, 1, false, P, false)
    NAV_ROLLOUT_CASE(true, 4, 8, 1, false, P, false)
    NAV_ROLLOUT_CASE(true, 8, 2, 4, true, P, false) NAV_ROLLOUT_CASE(true, 8, 4, 4, true, P, false)
    NAV_ROLLOUT_CASE(true, 8, 8, 4, true, P, false)
    NAV_ROLLOUT_CASE(true, 8, 2, 4, false, H, false) NAV_ROLLOUT_CASE(true, 8, 4, 4, false, H, false)
    NAV_ROLLOUT_CASE(true, 8, 8, 4, false, H, false)
    NAV_ROLLOUT_CASE(true, 8, 2, 4, true, H, false) NAV_ROLLOUT_CASE(true, 8, 4, 4, true, H, false)
    NAV_ROLLOUT_CASE(true, 8, 8, 4, true, H, false)
#undef NAV_ROLLOUT_CASE
    return hipErrorInvalidValue;
}

}  // extern "C"

// ---------------------------------------------------------------- RAPTOR fixture
namespace nav {
// Each lane group runs RAPTOR from the initial hidden state over obs[steps][22]
// with the production group step (raptor_fixture, main.mm:74-77).
template <int G>
__global__ __launch_bounds__(64) void raptor_fixture_kernel(const float* __restrict__ RW, const float* __restrict__ obs,
                                                            uint32_t steps, uint32_t copies, float* __restrict__ actions,
                                                            float* __restrict__ hidden_out) {
    constexpr int E = 64 / G, U = 16 / G;
    __shared__ float s_x[E][17];
    __shared__ float s_h[E][17];
    const uint32_t lane = threadIdx.x % G, grp = threadIdx.x / G;
    const uint32_t copy = blockIdx.x * E + grp;
    const bool live = copy < copies;
    float hidden[16], hu[U];
#pragma unroll
    for (int j = 0; j < 16; j++) hidden[j] = RW[2000 + j];
#pragma unroll
    for (int j = 0; j < U; j++) hu[j] = RW[2000 + lane + G * j];
    for (uint32_t t = 0; t < steps; t++) {
        float mo[22];
#pragma unroll
        for (int j = 0; j < 22; j++) mo[j] = obs[t * 22 + j];
        float act[4];
        raptor_group<G>(RW, mo, hidden, hu, s_x[grp], s_h[grp], lane, live, act);
        if (live && lane == 0) {
            // the fixture reports the raw network output (raptor.hpp:51),
            // recomputed here without the clip
#pragma unroll
            for (int q = 0; q < 4; q++) {
                float val = RW[2080 + q];
#pragma unroll
                for (int col = 0; col < 16; col++) val = fma_f(RW[2016 + q * 16 + col], hidden[col], val);
                actions[(size_t(copy) * steps + t) * 4 + q] = val;
            }
        }
    }
    if (live && lane == 0)
        for (int j = 0; j < 16; j++) hidden_out[size_t(copy) * 16 + j] = hidden[j];
}
}  // namespace nav

extern "C" hipError_t nav_launch_raptor_fixture(const float* RW, const float* obs, uint32_t steps, uint32_t copies,
                                                float* actions, float* hidden, int lanes_per_env, hipStream_t st) {
    const uint32_t per = 64 / lanes_per_env;
    const dim3 grid((copies + per - 1) / per);
    if (lanes_per_env == 4) hipLaunchKernelGGL(nav::raptor_fixture_kernel<4>, grid, dim3(64), 0, st, RW, obs, steps, copies, actions, hidden);
    else if (lanes_per_env == 8) hipLaunchKernelGGL(nav::raptor_fixture_kernel<8>, grid, dim3(64), 0, st, RW, obs, steps, copies, actions, hidden);
    else if (lanes_per_env == 16) hipLaunchKernelGGL(nav::raptor_fixture_kernel<16>, grid, dim3(64), 0, st, RW, obs, steps, copies, actions, hidden);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
