// memory.hip — the geometry-memory hint of the 184-input actor
// (guidance.hpp:100-194 nav_memory_clearance / nav_guidance_memory, as the CPU
// reference calls it: cpu_reference.hpp:353-375; the reference's GPU splits it
// into memory.metal:9-153 + sim.metal:226).
//
// One workgroup per env, run between the env kernel's observation of a tick
// and the launch that acts on it:
//   1. the env's up to 8 x 80 remembered range hits become body-frame points,
//      built once instead of once per candidate direction.  Only points that
//      some sweep could touch are kept (compacted into LDS): a contact needs
//      along <= 3 + radius and |p|^2 - along^2 < radius^2, so a point with
//      |p|^2 above (3 + radius)^2 + radius^2 (with a 0.1 % margin for
//      rounding) is never one, whatever the sweep.  The kept points are
//      grouped nearest first in quarter-metre shells;
//   2. each of the 85 candidate sweeps is scanned by PARTS threads, which take
//      every PARTS-th kept point (every lane of a part reads the same point:
//      LDS broadcast) with one trip count for the whole workgroup; the nearest
//      contacts are combined with a min, which is exact in any order, so the
//      order of the points does not change the result.  A contact needs along
//      > c = sqrt(|p|^2 - radius^2), and it lowers the sweep's nearest contact
//      so far only if along - radius < nearest; with margins for rounding both
//      are comparisons of one three-fma chain, and only a point that passes
//      them (for some lane of the wavefront) is evaluated exactly.  Near
//      points first lower the running nearest contact early, so most later
//      points fail the second;
//   3. the 85 candidates are scored and reduced with the sequential scan's
//      rule (maximum score, first candidate on ties), and three lanes write
//      the hint to the row's last three inputs.
// What bounds it: VALU issue for fleets that fill the GPU (8,192 envs in box
// worlds: 119 us a tick, from 143 when every pair was tested with the exact
// operations), the
// chain of dependent loads and LDS round trips for small ones (128 envs: 20
// us, from 38): every load that depends on no other is issued at the start,
// the goal's cell and the risk are formed while the ranges arrive, and points
// are read four at a time.  Finding the contacts on the matrix cores instead
// (one k-step tests 16 points x 16 sweeps) and evaluating listed pairs was
// slower (150-190 us for 8,192 envs): the lists cost more than the tests saved.
// Every value is computed with the operations and order of the oracle's
// restatement, so the hint is bit-identical to it.
#include <hip/hip_runtime.h>

#include "kernel_args.h"
#include "mdnav_math.h"
#include "mdnav_types.h"

namespace mem {
using namespace mdn;

constexpr uint32_t OBS = MDN_ACTOR_OBS_PRIOR;
constexpr uint32_t POINTS = 640, CANDIDATES = 85, SHELLS = 16;

__device__ __forceinline__ float fbits(uint32_t u) { return __builtin_bit_cast(float, u); }
// Correctly rounded square root of a positive normal x >= 2^-96: the
// hardware estimate and the one-ulp correction of the compiler's own
// correctly rounded sqrt lowering, without its scaling of tiny inputs and its
// zero / infinity fix-up, neither of which applies in that range (the
// instruction sequence is otherwise the same, so the results are equal).
__device__ __forceinline__ float sqrt_pos(float x) {
    const float s = __builtin_amdgcn_sqrtf(x);
    const uint32_t b = __builtin_bit_cast(uint32_t, s);
    const float dn = fbits(b - 1u), up = fbits(b + 1u);
    float r = __builtin_fmaf(-dn, s, x) <= 0.0f ? dn : s;
    r = __builtin_fmaf(-up, s, x) > 0.0f ? up : r;
    return r;
}
// distance shell of a kept point by |p|^2: quarter metres (the order of the
// points does not change the result)
__device__ __forceinline__ uint32_t shell_of(float p2) {
    return min(uint32_t(4.0f * __builtin_amdgcn_sqrtf(p2)), SHELLS - 1);
}
__device__ __forceinline__ float div_r(float x, double r) { return float(double(x) * r); }

// The 8 x 10 pooled grid with a border: cell (row, col) at (row + 1) * GRID + col + 1.
constexpr uint32_t GRID = 12, GRID_WORDS = 10 * GRID;
__device__ __forceinline__ uint32_t grid_at(uint32_t row, uint32_t col) { return (row + 1) * GRID + col + 1; }
// guidance.hpp:27-34 over the current ranges (already x 12; border 12, the scan's start)
__device__ __forceinline__ float min3x3(const float* cur, uint32_t at) {
    float nearest = 12.0f;
#pragma unroll
    for (int k = 0; k < 9; k++) nearest = fmin_f(nearest, cur[int(at) + (k / 3 - 1) * int(GRID) + k % 3 - 1]);
    return nearest;
}
// guidance.hpp:55-63 over the per-cell risk contributions (0 or min(0.2 u, 1); border 0)
__device__ __forceinline__ float max3x3(const float* v, uint32_t at) {
    float risk = 0.0f;
#pragma unroll
    for (int k = 0; k < 9; k++) risk = fmax_f(risk, v[int(at) + (k / 3 - 1) * int(GRID) + k % 3 - 1]);
    return risk;
}

// arg-max over a wavefront with the first index winning ties.  The larger of
// two pairs does not depend on their order, so within a row the lanes meet by
// quad swaps and mirrors (DPP); the two levels across rows shuffle.
__device__ __forceinline__ void arg_max(float& v, uint32_t& idx, float ov, uint32_t oi) {
    if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
}
template <int CTRL>
__device__ __forceinline__ void dpp_arg_max(float& v, uint32_t& idx) {
    const float ov = fbits(uint32_t(__builtin_amdgcn_update_dpp(0, int(__builtin_bit_cast(uint32_t, v)), CTRL, 0xF, 0xF, false)));
    const uint32_t oi = uint32_t(__builtin_amdgcn_update_dpp(0, int(idx), CTRL, 0xF, 0xF, false));
    arg_max(v, idx, ov, oi);
}
__device__ __forceinline__ void wave_argmax(float& v, uint32_t& idx) {
    dpp_arg_max<0xB1>(v, idx);   // quad_perm [1,0,3,2]
    dpp_arg_max<0x4E>(v, idx);   // quad_perm [2,3,0,1]
    dpp_arg_max<0x141>(v, idx);  // row_half_mirror
    dpp_arg_max<0x140>(v, idx);  // row_mirror
#pragma unroll
    for (int off = 16; off < 64; off <<= 1) arg_max(v, idx, __shfl_xor(v, off, 64), __shfl_xor(idx, off, 64));
}

// Eight wavefronts per env for fleets of at most WIDE_ENVS (latency: more
// parts, fewer points per thread; us a tick with eight and four: 20 and 30 at
// 128 envs, 46 and 49 at 2,048), four for larger ones (issue: the loads and
// barriers that every wavefront repeats; 74 and 74 at 4,096, 126 and 119 at
// 8,192).
constexpr uint32_t WIDE_ENVS = 2048;
template <uint32_t WAVES>
__global__ __launch_bounds__(64 * WAVES) void memory_hint_kernel(nav::MemoryArgs a) {
    constexpr uint32_t THREADS = 64 * WAVES;
    constexpr uint32_t PARTS = THREADS / CANDIDATES;
    // points: (x, y, z, -low) and (c - low, radius); sweeps
    __shared__ float4 pts[POINTS + 4 * PARTS], sweep[CANDIDATES];
    __shared__ float2 lim[POINTS + 4 * PARTS];
    __shared__ float part_near[PARTS][CANDIDATES];
    __shared__ float poses[96];
    __shared__ float cur[GRID_WORDS], risk_v[GRID_WORDS];
    __shared__ float cand_score[2], cand_free[CANDIDATES];
    __shared__ uint32_t cand_idx[2], goal_cell_s[2];
    __shared__ float goal_al_s[2];
    __shared__ uint32_t shell_count[SHELLS];
    const uint32_t n = blockIdx.x, t = threadIdx.x, wv = t / 64, lane = t % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(wv);  // uniform trip counts
    const uint32_t* hd = a.head + size_t(n) * nav::MEM_HEAD_WORDS;
    float* og = a.obs + size_t(n) * OBS;
    const float* ctx = og + 160;
    // every load that depends on no other, before the first use
    uint32_t head[nav::MEM_HEAD_WORDS];
#pragma unroll
    for (uint32_t j = 0; j < nav::MEM_HEAD_WORDS; j++) head[j] = hd[j];
    const float gin[3] = {ctx[0], ctx[1], ctx[2]};
    const float vel[3] = {ctx[4] * 4.0f, ctx[5] * 4.0f, ctx[6] * 4.0f};
    const uint32_t cell_t = t < 80 ? t : 0;
    const float ray_t[3] = {a.cells[3 * cell_t], a.cells[3 * cell_t + 1], a.cells[3 * cell_t + 2]};
    const float now_t = og[cell_t], old_t = og[80 + cell_t];
    const float pose_t = a.poses[size_t(n) * 96 + (t < 96 ? t : 0)];
    if (head[nav::MEM_HEAD_OBSERVED] == 0u) return;  // uniform over the workgroup
    const float distance = fbits(head[nav::MEM_HEAD_DISTANCE]);
    const float gnorm = sqrt_f(gin[0] * gin[0] + gin[1] * gin[1] + gin[2] * gin[2]);
    if (gnorm < 1e-6f || distance < 0.05f) {
        if (t < 3) og[OBS - 3 + t] = 0.0f;
        return;
    }
    // the ranges of this thread's up to three remembered cells: the cell's
    // 2x2 pixels, each row pair one 8-byte load (the column is even)
    constexpr uint32_t PER = (POINTS + THREADS - 1) / THREADS;
    const uint32_t latest = head[nav::MEM_HEAD_FRAME], valid = head[nav::MEM_HEAD_VALID];
    float2 r01[PER], r23[PER];
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) {
        const uint32_t j = k * THREADS + t, back = j / 80, cell = j % 80;
        const uint32_t frame = (latest + 8u - back) % 8u;
        const bool on = j < POINTS && back < valid;
        const float* px = a.sensors + (size_t(n) * 8 + (on ? frame : 0u)) * 320 +
                          (on ? (cell / 10) * 40 + (cell % 10) * 2 : 0u);
        r01[k] = *reinterpret_cast<const float2*>(px);
        r23[k] = *reinterpret_cast<const float2*>(px + 20);
    }
    // what only the two wavefronts of the candidates use
    const float sensor_dt = a.sensor_dt;
    float goal[3] = {0.0f, 0.0f, 0.0f}, stop_margin = 0.0f;
    if (wave < 2) {
#pragma unroll
        for (int j = 0; j < 3; j++) goal[j] = gin[j] / gnorm;
        const float speed = sqrt_f(vel[0] * vel[0] + vel[1] * vel[1] + vel[2] * vel[2]);
        stop_margin = 0.28f + speed * fmax_f(sensor_dt, 0.0f) + 0.25f * speed * speed;
    }
    float pose[12];
#pragma unroll
    for (int j = 0; j < 12; j++) pose[j] = fbits(head[nav::MEM_HEAD_POSE + j]);

    // candidate direction of thread t (guidance.hpp:164-166): the 80 cells,
    // the goal, up, down, left and right
    float dir[3] = {ray_t[0], ray_t[1], ray_t[2]};
    if (t == 80) {
        dir[0] = goal[0]; dir[1] = goal[1]; dir[2] = goal[2];
    } else if (t > 80) {
        dir[0] = 0.0f;
        dir[1] = t >= 83 ? (t == 83 ? 1.0f : -1.0f) : 0.0f;
        dir[2] = t < 83 ? (t == 81 ? 1.0f : -1.0f) : 0.0f;
    }
    if (t < 96) poses[t] = pose_t;
    if (t < SHELLS) shell_count[t] = 0;
    if (t < CANDIDATES) {  // the sweeps
        float sw[3] = {1.2f * dir[0] + 0.35f * vel[0], 1.2f * dir[1] + 0.35f * vel[1],
                       1.2f * dir[2] + 0.35f * vel[2]};
        const float sn = sqrt_f(sw[0] * sw[0] + sw[1] * sw[1] + sw[2] * sw[2]);
#pragma unroll
        for (int j = 0; j < 3; j++) sw[j] /= fmax_f(sn, 1e-6f);
        sweep[t] = make_float4(sw[0], sw[1], sw[2], 1.0f);
    }
    // per-cell current range x 12 and closing-speed risk contribution
    if (t < GRID_WORDS) {
        const uint32_t row = t / GRID, col = t % GRID;
        if (row == 0 || row == 9 || col == 0 || col == GRID - 1) {
            cur[t] = 12.0f;
            risk_v[t] = 0.0f;
        }
    }
    if (t < 80) {
        const float now = now_t * 12.0f, old = old_t * 12.0f;
        const uint32_t at = grid_at(t / 10, t % 10);
        cur[at] = now;
        const float unexpected =
            div_r(old - now, a.inv_sensor_dt) - (vel[0] * ray_t[0] + vel[1] * ray_t[1] + vel[2] * ray_t[2]);
        const bool hit = (sensor_dt > 1e-4f) & (old < 11.9f) & (now < 11.9f) & (unexpected > 0.5f);
        risk_v[at] = hit ? fmin_f(0.20f * unexpected, 1.0f) : 0.0f;
    }
    // goal cell: the cell ray best aligned with the goal (first on ties), wave 0 and 1
    if (t < 128) {
        float al = -1e20f;
        uint32_t c = 80;
        if (t < 80) {
            al = ray_t[0] * goal[0] + ray_t[1] * goal[1] + ray_t[2] * goal[2];
            if (!(al == al)) al = -INFINITY;  // the scan never selects a NaN
            c = t;
        }
        wave_argmax(al, c);
        if ((t & 63) == 0) { goal_al_s[wv] = al; goal_cell_s[wv] = c; }
    }
    __syncthreads();
    // 1. remembered points (guidance.hpp:113-139 up to the sweep test)
    float4 held[PER];
    float2 held_rad[PER];
    uint32_t shell[PER];
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) {
        const uint32_t j = k * THREADS + t, back = j / 80, cell = j % 80;
        shell[k] = SHELLS;
        if (j < POINTS && back < valid) {
            const float* old_pose = poses + ((latest + 8u - back) % 8u) * 12;
            const uint32_t px = (cell / 10) * 40 + (cell % 10) * 2;
            const float others[3] = {r01[k].y, r23[k].x, r23[k].y};
            const uint32_t pixels[3] = {px + 1, px + 20, px + 21};
            uint32_t hit = px;
            float range = r01[k].x;
#pragma unroll
            for (int q = 0; q < 3; q++)
                if (others[q] < range) { range = others[q]; hit = pixels[q]; }
            if (!(range <= 0.01f || range >= 11.9f)) {
                const float* ray = a.pix_rays + 3 * hit;
                const float wx = old_pose[3] * ray[0] + old_pose[4] * ray[1] + old_pose[5] * ray[2];
                const float wy = old_pose[6] * ray[0] + old_pose[7] * ray[1] + old_pose[8] * ray[2];
                const float wz = old_pose[9] * ray[0] + old_pose[10] * ray[1] + old_pose[11] * ray[2];
                const float dx = old_pose[0] + range * wx - pose[0];
                const float dy = old_pose[1] + range * wy - pose[1];
                const float dz = old_pose[2] + range * wz - pose[2];
                const float x = pose[3] * dx + pose[6] * dy + pose[9] * dz;
                const float y = pose[4] * dx + pose[7] * dy + pose[10] * dz;
                const float z = pose[5] * dx + pose[8] * dy + pose[11] * dz;
                // nav_memory_point_radius with the capture-age term off
                const float age = fmax_f(float(back) * fmax_f(sensor_dt, 0.0f), 0.0f) + 0.0f;
                const float radius = 0.20f + 0.015f * range + 0.15f * age;
                const float p2 = x * x + y * y + z * z, lx = 3.0f + radius, ly = radius * radius;
                // A contact has along^2 > |p|^2 - radius^2 up to the rounding
                // of |p|^2, radius^2, along^2 and their difference, below
                // 5e-7 |p|^2 together; its value is at least along - radius
                // (1 + 2^-22); and the fma chain differs from the exact along -
                // radius by less than 5e-7 (1 + |p| + radius).  The margin is
                // several times these, and the root's own error.  (The radius
                // counts with points minutes old: 0.15 m a second.)
                const float margin = 2e-6f * (8.0f + p2 + radius), c2 = p2 - ly - margin;
                const float c = (c2 > 0.0f ? __builtin_amdgcn_sqrtf(c2) * 0.999999f : 0.0f) - margin;
                const float low = radius * 1.0001f + margin;
                held[k] = make_float4(x, y, z, -low);
                held_rad[k] = make_float2(c - low - margin, radius);
                if (p2 <= 1.001f * (lx * lx + ly)) shell[k] = shell_of(p2);
            }
        }
    }
    // places in the shells, in whatever order the points reserve them
    uint32_t rank[PER];
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) rank[k] = shell[k] < SHELLS ? atomicAdd(&shell_count[shell[k]], 1u) : 0u;
    __syncthreads();
    const uint32_t count = lane < SHELLS ? shell_count[lane] : 0u;
    uint32_t upto = count;  // inclusive prefix over the shells (one row of lanes)
    upto += uint32_t(__builtin_amdgcn_update_dpp(0, int(upto), 0x111, 0xF, 0xF, true));  // row_shr:1
    upto += uint32_t(__builtin_amdgcn_update_dpp(0, int(upto), 0x112, 0xF, 0xF, true));
    upto += uint32_t(__builtin_amdgcn_update_dpp(0, int(upto), 0x114, 0xF, 0xF, true));
    upto += uint32_t(__builtin_amdgcn_update_dpp(0, int(upto), 0x118, 0xF, 0xF, true));
    const uint32_t kept = __builtin_amdgcn_readlane(upto, SHELLS - 1), below = upto - count;
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) {
        const uint32_t at = rank[k] + __shfl(below, int(shell[k] % SHELLS), 64);
        if (shell[k] < SHELLS) {
            pts[at] = held[k];
            lim[at] = held_rad[k];
        }
    }
    if (t < 4 * PARTS) {  // padding that no sweep reaches
        pts[kept + t] = make_float4(0.0f, 0.0f, 0.0f, 1e9f);
        lim[kept + t] = make_float2(1e9f, 1.0f);
    }
    __syncthreads();

    // 2. swept-sphere clearance of every candidate (guidance.hpp:134-139),
    // each by PARTS threads that take every PARTS-th point, four at a time
    const uint32_t rounds = __builtin_amdgcn_readfirstlane((kept + 4 * PARTS - 1) / (4 * PARTS));
    if (t < PARTS * CANDIDATES) {
        const uint32_t c = t % CANDIDATES, part = t / CANDIDATES;
        const float4 sw = sweep[c];
        float near = 3.0f;
        for (uint32_t i = 0; i < rounds; i++) {
            float4 q[4];
            float2 k[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                q[j] = pts[(4 * i + j) * PARTS + part];
                k[j] = lim[(4 * i + j) * PARTS + part];
            }
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                const float u = fma_f(q[j].x, sw.x, fma_f(q[j].y, sw.y, fma_f(q[j].z, sw.z, q[j].w)));
                if ((u > k[j].x) & (u < near)) {
                    const float radius = k[j].y, r2 = radius * radius;
                    const float p2 = q[j].x * q[j].x + q[j].y * q[j].y + q[j].z * q[j].z;
                    const float along = q[j].x * sw.x + q[j].y * sw.y + q[j].z * sw.z;
                    const float lateral2 = __builtin_fmaxf(p2 - along * along, 0.0f);
                    const bool hit = (along > 0.0f) & (along <= 3.0f + radius) & (lateral2 < r2);
                    const float v = __builtin_fmaxf(along - sqrt_pos(r2 - lateral2), 0.0f);
                    near = hit ? __builtin_fminf(near, v) : near;
                }
            }
        }
        part_near[part][c] = near;
    }
    __syncthreads();

    // 3. candidate scores (guidance.hpp:167-183) and the best candidate
    if (wave >= 2) return;
    uint32_t gcell = goal_cell_s[0];
    if (goal_al_s[1] > goal_al_s[0] || (goal_al_s[1] == goal_al_s[0] && goal_cell_s[1] < gcell)) gcell = goal_cell_s[1];
    const float gsel = goal_al_s[1] > goal_al_s[0] || (goal_al_s[1] == goal_al_s[0] && goal_cell_s[1] < goal_cell_s[0])
                           ? goal_al_s[1] : goal_al_s[0];
    // scan's fallback without any finite alignment: cell (0, 0)
    const uint32_t goal_row = gsel > -1e20f ? gcell / 10 : 0, goal_col = gsel > -1e20f ? gcell % 10 : 0;

    const float desired_speed = fmin_f(1.6f, sqrt_f(4.0f * fmax_f(distance - 0.28f, 0.0f)));
    float score = -1e20f;
    uint32_t ci = CANDIDATES;
    if (t < CANDIDATES) {
        const uint32_t at = t < 80 ? grid_at(t / 10, t % 10) : grid_at(goal_row, goal_col);
        float free = part_near[0][t];
#pragma unroll
        for (uint32_t q = 1; q < PARTS; q++) free = fmin_f(free, part_near[q][t]);
        const float observed = min3x3(cur, at);
        if (t < 81) free = fmin_f(free, observed);
        const float temporal_risk = max3x3(risk_v, at);
        free = fmax_f(free - temporal_risk, 0.0f);
        const float alignment = dir[0] * goal[0] + dir[1] * goal[1] + dir[2] * goal[2];
        const float required = stop_margin + 0.15f + desired_speed * desired_speed * .25f;
        score = 1.4f * alignment + 0.20f * fmin_f(free, 3.0f) - (free < required ? 3.0f * (required - free) / required : 0.0f);
        if (!(score == score)) score = -INFINITY;  // the scan never selects a NaN
        ci = t;
        cand_free[t] = free;
        // the direction for the lanes that write the hint (the sweep is no longer read)
        sweep[t] = make_float4(dir[0], dir[1], dir[2], 0.0f);
    }
    wave_argmax(score, ci);
    if (lane == 0) { cand_score[wv] = score; cand_idx[wv] = ci; }
    __syncthreads();
    if (t < 3) {
        uint32_t best = cand_idx[0];
        if (cand_score[1] > cand_score[0] || (cand_score[1] == cand_score[0] && cand_idx[1] < best)) best = cand_idx[1];
        const bool any = (cand_score[0] > -1e20f) | (cand_score[1] > -1e20f);
        float best_dir = t == 0 ? 1.0f : 0.0f, best_free = 0.0f;
        if (any) {
            best_dir = reinterpret_cast<const float*>(&sweep[best])[t];
            best_free = cand_free[best];
        }
        const float tan_v = a.tan_v;
        const bool goal_in_fov = goal[0] > 0.0f && fabs_f(goal[1]) <= goal[0] && fabs_f(goal[2]) <= tan_v * goal[0];
        const float after_stop = fmax_f(best_free - stop_margin - 0.15f, 0.0f);
        float command_speed = fmin_f(desired_speed, sqrt_f(4.0f * after_stop));
        if (!goal_in_fov) command_speed = fmin_f(command_speed, 0.25f);
        const float fraction = fmin_f(0.8f, command_speed * 0.5f);
        const float x = fraction * best_dir;
        og[OBS - 3 + t] = 0.5f * log_f((1.0f + x) / (1.0f - x));
    }
}

}  // namespace mem

extern "C" hipError_t nav_launch_memory_hint(const nav::MemoryArgs* a, hipStream_t st) {
    if (a->n == 0) return hipSuccess;
    if (a->n > mem::WIDE_ENVS)
        hipLaunchKernelGGL(mem::memory_hint_kernel<4>, dim3(a->n), dim3(256), 0, st, *a);
    else
        hipLaunchKernelGGL(mem::memory_hint_kernel<8>, dim3(a->n), dim3(512), 0, st, *a);
    return hipGetLastError();
}
