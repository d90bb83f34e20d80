// fixed_ppo.hip — the reference's fixed-shape PPO operators (ppo.hpp:65-181,
// 310-324) as batched kernels over caller arrays: actor and critic forward,
// Gaussian log-probability, per-sample clipped-surrogate loss and derivatives,
// and Adam.  They back the mdn_op_* entry points that stand in for the header
// functions a host harness calls (fixed_ppo::actor_forward, ...); the training
// path uses the fused kernels of ppo.hip and large.hip.
//
// The arithmetic is the canonical form the rest of the library and the CPU
// oracle share: dot products are fma chains from the bias with inputs in
// ascending order, tanh/exp are this project's own (mdnav_math.h), divisions
// and square roots are correctly rounded.
#include <hip/hip_runtime.h>

#include "kernel_args.h"
#include "mdnav_math.h"
#include "mdnav_types.h"

namespace fppo {
using namespace mdn;

constexpr float LOG_TWO_PI = 1.8378770664093453f;
constexpr uint32_t MAX_IN = 1024, MAX_HIDDEN = 8192;

// First layer of 16 rows x 64 hidden units per workgroup on the matrix cores:
// each of the four wavefronts owns 16 units, and one 16x16x4 step is the same
// chain of fused multiply-adds, bias first and inputs ascending, as the scalar
// form.  Layouts (ppo.hpp:35-45): W1[H][D] at 0, b1[H], W2[O][H], b2[O]; the
// actor (O = 4) then has log_std[4], the critic (O = 1) nothing.
//
// Bound by latency: a batch of 4,096 rows is one workgroup per CU, so a tile
// loads its 80 rows of up to 192 inputs (60 loads a lane, coalesced, all in
// flight together) and then runs 46 dependent steps.  LDS rows are 196 words
// apart: the 16 rows x 4 inputs that a step reads lie in 64 different banks.
// Inputs beyond D multiply 0 by -0, which changes no partial sum.  184 -> 64
// -> 4 with the output chains: 9.7 us at 4,096 rows, 6.8 at one (one workgroup
// per row with scalar chains over uncoalesced weight rows: 29.6 and 13.3).
//
// O > 0: the whole hidden layer is this tile (H <= 64) and its output chains
// run here.  O = 0: wider layers; output_kernel follows.
constexpr uint32_t ROWS = 16, UNITS = 64, SLAB = 192, STRIDE = SLAB + 4, HSTRIDE = UNITS + 4;
using f32x4 = float __attribute__((ext_vector_type(4)));

template <uint32_t O>
__global__ __launch_bounds__(256) void hidden_kernel(const float* __restrict__ w, const float* __restrict__ x,
                                                     uint32_t D, uint32_t H, uint32_t prior, uint64_t B,
                                                     float* __restrict__ hidden, float* __restrict__ out) {
    __shared__ float s_w[UNITS * STRIDE];
    __shared__ float s_x[ROWS * STRIDE];
    __shared__ __align__(16) float s_h[O ? ROWS * HSTRIDE : 4];
    __shared__ __align__(16) float s_w2[O ? O * HSTRIDE : 4];
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint64_t row0 = uint64_t(blockIdx.x) * ROWS;
    const uint32_t unit0 = blockIdx.y * UNITS;
    const float* b1 = w + size_t(H) * D;
    const uint32_t unit = unit0 + wave * 16 + (lane & 15);
    const float bias = unit < H ? b1[unit] : 0.0f;
    if constexpr (O != 0) {
        if (t < O * UNITS) {
            const uint32_t o = t / UNITS, h = t % UNITS;
            s_w2[o * HSTRIDE + h] = h < H ? b1[H + size_t(o) * H + h] : -0.0f;
        }
    }
    f32x4 acc = {bias, bias, bias, bias};
    for (uint32_t k0 = 0; k0 < D; k0 += SLAB) {
        const uint32_t kn = D - k0 < SLAB ? D - k0 : SLAB;
        float rw[UNITS / 4][SLAB / 64], rx[ROWS / 4][SLAB / 64];
#pragma unroll
        for (uint32_t r = 0; r < UNITS / 4; r++) {
            const uint32_t u = unit0 + wave + 4 * r;
#pragma unroll
            for (uint32_t c = 0; c < SLAB / 64; c++) {
                const uint32_t k = lane + 64 * c;
                rw[r][c] = u < H && k < kn ? w[size_t(u) * D + k0 + k] : -0.0f;
            }
        }
#pragma unroll
        for (uint32_t r = 0; r < ROWS / 4; r++) {
            const uint64_t row = row0 + wave + 4 * r;
#pragma unroll
            for (uint32_t c = 0; c < SLAB / 64; c++) {
                const uint32_t k = lane + 64 * c;
                rx[r][c] = row < B && k < kn ? x[row * D + k0 + k] : 0.0f;
            }
        }
        if (k0) __syncthreads();  // the last slab has been read
#pragma unroll
        for (uint32_t c = 0; c < SLAB / 64; c++) {
#pragma unroll
            for (uint32_t r = 0; r < UNITS / 4; r++) s_w[(wave + 4 * r) * STRIDE + lane + 64 * c] = rw[r][c];
#pragma unroll
            for (uint32_t r = 0; r < ROWS / 4; r++) s_x[(wave + 4 * r) * STRIDE + lane + 64 * c] = rx[r][c];
        }
        __syncthreads();
        const float* fx = s_x + (lane & 15) * STRIDE + (lane >> 4);
        const float* fw = s_w + (wave * 16 + (lane & 15)) * STRIDE + (lane >> 4);
#pragma unroll 8
        for (uint32_t k = 0; k < kn; k += 4) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fx[k], fw[k], acc, 0, 0, 0);
    }
#pragma unroll
    for (uint32_t r = 0; r < 4; r++) {
        const float z = acc[r];
        const float a = tanh_f(z);
        const uint32_t m = 4 * (lane >> 4) + r;
        if (unit < H && row0 + m < B) hidden[(row0 + m) * H + unit] = a;
        if constexpr (O != 0) s_h[m * HSTRIDE + wave * 16 + (lane & 15)] = unit < H ? a : 0.0f;
    }
    if constexpr (O != 0) {
        __syncthreads();
        const uint32_t m = t / O, o = t % O;
        if (m < ROWS && row0 + m < B) {
            float z = b1[H + size_t(O) * H + o];
            const f32x4* h4 = reinterpret_cast<const f32x4*>(s_h + m * HSTRIDE);
            const f32x4* v4 = reinterpret_cast<const f32x4*>(s_w2 + o * HSTRIDE);
#pragma unroll
            for (uint32_t q = 0; q < UNITS / 4; q++) {
                const f32x4 h = h4[q], v = v4[q];
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) z = fma_f(v[i], h[i], z);
            }
            // geometry prior (ppo.hpp:30-34, 77): the hint inputs join the first three means
            if (prior && o < 3) z += x[(row0 + m) * D + D - 3 + o];
            out[(row0 + m) * O + o] = z;
        }
    }
}

// Output chains over a hidden layer wider than one tile: one wavefront runs
// the 16 rows x O chains of a workgroup, all four bring the next 256 units of
// the rows and of W2 while it does.  Bound by the chain itself, about 6 cycles
// a unit.  184 -> 2,048 -> 4 at 1,024 rows: hidden layer 28.7 us, this 14.8
// (scalar chains: 238 together).  A layer of one tile stays with the fused
// form: a second launch costs more than its chain of 64.
constexpr uint32_t OUT_SLAB = 256, OUT_STRIDE = OUT_SLAB + 4;

template <uint32_t O>
__global__ __launch_bounds__(256) void output_kernel(const float* __restrict__ w, const float* __restrict__ x,
                                                     uint32_t D, uint32_t H, uint32_t prior, uint64_t B,
                                                     const float* __restrict__ hidden, float* __restrict__ out) {
    __shared__ __align__(16) float s_h[2][ROWS * OUT_STRIDE];
    __shared__ __align__(16) float s_v[2][O * OUT_STRIDE];
    const uint32_t t = threadIdx.x, m = t / O, o = t % O;
    const uint64_t row0 = uint64_t(blockIdx.x) * ROWS;
    const float* w2 = w + size_t(H) * D + H;
    const bool mine = m < ROWS && row0 + m < B;
    float rh[ROWS], rv[O];
    auto load = [&](uint32_t h0) {
        const bool in = h0 + t < H;
#pragma unroll
        for (uint32_t r = 0; r < ROWS; r++) rh[r] = in && row0 + r < B ? hidden[(row0 + r) * H + h0 + t] : 0.0f;
#pragma unroll
        for (uint32_t r = 0; r < O; r++) rv[r] = in ? w2[size_t(r) * H + h0 + t] : -0.0f;
    };
    load(0);
    float z = mine ? w2[size_t(O) * H + o] : 0.0f;
    for (uint32_t h0 = 0, b = 0; h0 < H; h0 += OUT_SLAB, b ^= 1) {
#pragma unroll
        for (uint32_t r = 0; r < ROWS; r++) s_h[b][r * OUT_STRIDE + t] = rh[r];
#pragma unroll
        for (uint32_t r = 0; r < O; r++) s_v[b][r * OUT_STRIDE + t] = rv[r];
        __syncthreads();  // also: every wavefront is past the slab before the last, whose buffer comes next
        if (h0 + OUT_SLAB < H) load(h0 + OUT_SLAB);
        if (mine) {
            const f32x4* h4 = reinterpret_cast<const f32x4*>(s_h[b] + m * OUT_STRIDE);
            const f32x4* v4 = reinterpret_cast<const f32x4*>(s_v[b] + o * OUT_STRIDE);
#pragma unroll 8
            for (uint32_t q = 0; q < OUT_SLAB / 4; q++) {
                const f32x4 h = h4[q], v = v4[q];
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) z = fma_f(v[i], h[i], z);
            }
        }
    }
    if (mine) {
        if (prior && o < 3) z += x[(row0 + m) * D + D - 3 + o];  // geometry prior (ppo.hpp:30-34, 77)
        out[(row0 + m) * O + o] = z;
    }
}

template <uint32_t O>
hipError_t launch_forward(const float* w, const float* x, uint32_t D, uint32_t H, uint32_t prior, uint64_t B,
                          float* hidden, float* out, hipStream_t st) {
    const dim3 tiles(uint32_t((B + ROWS - 1) / ROWS), (H + UNITS - 1) / UNITS);
    if (H <= UNITS) {
        hipLaunchKernelGGL(hidden_kernel<O>, tiles, dim3(256), 0, st, w, x, D, H, prior, B, hidden, out);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(hidden_kernel<0>, tiles, dim3(256), 0, st, w, x, D, H, prior, B, hidden, out);
    hipLaunchKernelGGL(output_kernel<O>, dim3(tiles.x), dim3(256), 0, st, w, x, D, H, prior, B, hidden, out);
    return hipGetLastError();
}

__device__ __forceinline__ float log_prob(const float* a, const float* m, const float* ls) {
    float r = 0.0f;
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
        const float inv_std = exp_f(-ls[q]);
        const float d = (a[q] - m[q]) * inv_std;
        r += -0.5f * (d * d + 2.0f * ls[q] + LOG_TWO_PI);
    }
    return r;
}

// ppo.hpp:95-103; log_std is shared ([4], stride 0) or per row ([B][4]).
__global__ __launch_bounds__(256) void log_prob_kernel(const float* __restrict__ act, const float* __restrict__ mean,
                                                       const float* __restrict__ log_std, uint32_t ls_stride,
                                                       uint64_t B, float* __restrict__ out) {
    const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= B) return;
    out[i] = log_prob(act + 4 * i, mean + 4 * i, log_std + ls_stride * i);
}

// ppo.hpp:144-181 per row: d_mean[4], d_log_std[4], d_value and the losses
// [policy, value, entropy, ratio].
__global__ __launch_bounds__(256) void loss_grad_kernel(fppo_loss_args a) {
    const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= a.b) return;
    const float* act = a.actions + 4 * i;
    const float* mean = a.means + 4 * i;
    const float* ls = a.log_std + a.ls_stride * i;
    const float adv = a.advantages[i];
    const float value = a.values[i], target = a.returns[i];
    const float logp = log_prob(act, mean, ls);
    const float raw = logp - a.old_logp[i];
    const float ratio = exp_f(clamp_f(raw, -20.0f, 20.0f));
    const float clipped = clamp_f(ratio, 1.0f - a.clip, 1.0f + a.clip);
    const float chosen = min_f(ratio * adv, clipped * adv);
    const bool in_range = raw >= -20.0f && raw <= 20.0f;
    const bool active = in_range && (adv >= 0.0f ? ratio <= 1.0f + a.clip : ratio >= 1.0f - a.clip);
    const float scale = 1.0f / max_f(a.batch_size, 1.0f);
    float entropy = 0.0f;
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
        const float inv_var = exp_f(-2.0f * ls[q]);
        const float diff = act[q] - mean[q];
        float dm = 0.0f, dl = 0.0f;
        if (active) {
            const float dlogp = -ratio * adv * scale;
            dm = dlogp * diff * inv_var;
            dl = dlogp * (diff * diff * inv_var - 1.0f);
        }
        dl -= a.ecoef * scale;
        entropy += -a.ecoef * (ls[q] + 0.5f * (1.0f + LOG_TWO_PI)) * scale;
        a.d_mean[4 * i + q] = dm;
        a.d_log_std[4 * i + q] = dl;
    }
    a.d_value[i] = a.vcoef * (value - target) * scale;
    a.losses[4 * i] = -chosen * scale;
    a.losses[4 * i + 1] = 0.5f * a.vcoef * (value - target) * (value - target) * scale;
    a.losses[4 * i + 2] = entropy;
    a.losses[4 * i + 3] = ratio;
}

// ppo.hpp:310-324 elementwise; c1, c2 = 1 - beta^step from the host.
__global__ __launch_bounds__(256) void adam_op_kernel(float* __restrict__ p, const float* __restrict__ g,
                                                      float* __restrict__ m, float* __restrict__ v, uint64_t n,
                                                      float lr, float b1, float b2, float eps, float wd, float c1,
                                                      float c2) {
    const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i] + wd * p[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrt_f(vi / c2) + eps);
}

}  // namespace fppo

extern "C" {

hipError_t fppo_launch_forward(const float* w, const float* x, uint32_t D, uint32_t H, uint32_t O, uint32_t prior,
                               uint64_t B, float* hidden, float* out, hipStream_t st) {
    if (B == 0) return hipSuccess;
    if (D == 0 || D > fppo::MAX_IN || H == 0 || H > fppo::MAX_HIDDEN || (O != 1 && O != 4) || !hidden ||
        B > 0x7fffffffull || (prior && D < 3))
        return hipErrorInvalidValue;
    return O == 4 ? fppo::launch_forward<4>(w, x, D, H, prior, B, hidden, out, st)
                  : fppo::launch_forward<1>(w, x, D, H, prior, B, hidden, out, st);
}

hipError_t fppo_launch_log_prob(const float* act, const float* mean, const float* log_std, uint32_t ls_stride,
                                uint64_t B, float* out, hipStream_t st) {
    if (B == 0) return hipSuccess;
    hipLaunchKernelGGL(fppo::log_prob_kernel, dim3(uint32_t((B + 255) / 256)), dim3(256), 0, st, act, mean, log_std,
                       ls_stride, B, out);
    return hipGetLastError();
}

hipError_t fppo_launch_loss_grad(const fppo_loss_args* a, hipStream_t st) {
    if (a->b == 0) return hipSuccess;
    hipLaunchKernelGGL(fppo::loss_grad_kernel, dim3(uint32_t((a->b + 255) / 256)), dim3(256), 0, st, *a);
    return hipGetLastError();
}

hipError_t fppo_launch_adam(float* p, const float* g, float* m, float* v, uint64_t n, float lr, float b1, float b2,
                            float eps, float wd, float c1, float c2, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(fppo::adam_op_kernel, dim3(uint32_t((n + 255) / 256)), dim3(256), 0, st, p, g, m, v, n, lr, b1,
                       b2, eps, wd, c1, c2);
    return hipGetLastError();
}

}  // extern "C"
