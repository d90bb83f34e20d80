// rollout_small.hip — the rollout instances for fleets too small to give
// every wavefront of the GPU eight envs, and for per-episode plants and tasks.
#include "rollout_kernel.h"

// An 8-lane env step is one latency chain per wavefront, and its depth frames
// are cast one env after the other over the wavefront's 64 lanes.  A fleet of
// n <= 4 x 1,024 envs therefore holds ceil(n / 1,024) envs per wavefront (four
// wavefronts on each of the 256 CUs) instead of eight: fewer frames per
// wavefront and one matrix-core tile per layer and wavefront instead of two.
extern "C" hipError_t nav_launch_rollout_small(const nav::RolloutArgs* args, int ring_slots,
                                               uint32_t actor_obs, hipStream_t stream) {
    constexpr uint32_t P = MDN_ACTOR_OBS_POOLED, H = MDN_ACTOR_OBS_PRIOR, WAVES = 4, CUS = 256;
    nav::RolloutArgs a = *args;
    a.epw = (a.cfg.n + WAVES * CUS - 1) / (WAVES * CUS);
    a.epw = a.epw < 1 ? 1 : (a.epw > 4 ? 4 : a.epw);
    const uint32_t per = WAVES * a.epw, blocks = (a.cfg.n + per - 1) / per;
    const bool dyn = a.env_phys != nullptr, ext = a.ext_means != nullptr;
    const bool cf = !dyn && std::memcmp(&a.phys, &mdn::kCrazyflie, sizeof(MdnPhysicsParams)) == 0;
#define NAV_ROLLOUT_CASE(COND, K, X, D, DYN, CF)                                                               \
    if (COND && ring_slots == K && ext == X && actor_obs == D && dyn == DYN) {                                 \
        hipLaunchKernelGGL((nav::rollout_kernel<8, K, 4, X, D, DYN, CF, true>), dim3(blocks), dim3(256), 0,    \
                           stream, a);                                                                         \
        return hipGetLastError();                                                                              \
    }
    // the Crazyflie plant as compile-time constants
    NAV_ROLLOUT_CASE(cf, 2, false, P, false, true) NAV_ROLLOUT_CASE(cf, 4, false, P, false, true)
    NAV_ROLLOUT_CASE(cf, 2, false, H, false, true)
    NAV_ROLLOUT_CASE(cf, 2, true, P, false, true) NAV_ROLLOUT_CASE(cf, 2, true, H, false, true)
    // any plant
    NAV_ROLLOUT_CASE(true, 2, false, P, false, false) NAV_ROLLOUT_CASE(true, 4, false, P, false, false)
    NAV_ROLLOUT_CASE(true, 8, false, P, false, false) NAV_ROLLOUT_CASE(true, 2, false, H, false, false)
    NAV_ROLLOUT_CASE(true, 4, false, H, false, false) NAV_ROLLOUT_CASE(true, 8, false, H, false, false)
    NAV_ROLLOUT_CASE(true, 2, true, P, false, false) NAV_ROLLOUT_CASE(true, 4, true, P, false, false)
    NAV_ROLLOUT_CASE(true, 8, true, P, false, false) NAV_ROLLOUT_CASE(true, 2, true, H, false, false)
    NAV_ROLLOUT_CASE(true, 4, true, H, false, false) NAV_ROLLOUT_CASE(true, 8, true, H, false, false)
    // per-episode plants and navigation tasks
    NAV_ROLLOUT_CASE(true, 2, false, P, true, false) NAV_ROLLOUT_CASE(true, 4, false, P, true, false)
    NAV_ROLLOUT_CASE(true, 8, false, P, true, false) NAV_ROLLOUT_CASE(true, 2, false, H, true, false)
    NAV_ROLLOUT_CASE(true, 4, false, H, true, false) NAV_ROLLOUT_CASE(true, 8, false, H, true, false)
#undef NAV_ROLLOUT_CASE
    return hipErrorInvalidValue;
}
