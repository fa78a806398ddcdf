// The GEMV's neighbours in a decode step that the reference's CUDA backend fuses around it:
//
//  RMS norm (+ residual add) -> Q8_K activation          crates/rnb-backend/cuda/cuda/kernels/quant_batch_and_ops.cuh:4031
//                                                         (rnb_rms_norm_f32) and :4275 (rnb_rms_norm_add_then_rms_norm_q8_1_f32;
//                                                         here the quantised form is rnb-cpu's Q8_K, not the CUDA backend's Q8_1)
//  router top-k + softmax over the selected logits        crates/rnb-llm/src/engine/models/shared_expert_moe/routing.rs:18-64
//
// Arithmetic of the norm is rnb-cpu's (crates/rnb-cpu/src/kernels/norm.rs:140-225): the mean square is accumulated in f64
// (rms_norm_into_f64, the default) and rms = f32(sqrt(mean + eps)); with the unit offset (scale = 1 + weight) in f32, as
// rms_norm_unit_offset_into_scalar does; out = (x / rms) * scale with one IEEE division and one multiplication.  The
// quantiser is the wave-level Q8_K routine of act_quant.h applied to those f32 values, so quantising the f32 output with
// rnb_hip_quantize_q8k gives the same bits.
#include "act_quant.h"
#include "device_utils.h"
#include "kernels.h"
#include <type_traits>

namespace rnb {

namespace {

constexpr int kNormMaxWaves = 16;
constexpr uint32_t kNormManyRows = 513;  // two workgroups of sixteen waves fit a compute unit: 512 rows at once

// sum over the wave on the DPP data path, in lane 63 (f64: its two halves move separately)
template <int kCtrl, int kRowMask>
__device__ __forceinline__ double dpp_add(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(u), kCtrl, kRowMask, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(u >> 32), kCtrl, kRowMask, 0xf, false);
    const unsigned long long t = static_cast<unsigned long long>(static_cast<uint32_t>(hi)) << 32 | static_cast<uint32_t>(lo);
    return v + __builtin_bit_cast(double, t);
}
__device__ __forceinline__ double row16_sum(double v) {  // every lane of an aligned 16 gets the sum
    v = dpp_add<0xB1, 0xf>(v);
    v = dpp_add<0x4E, 0xf>(v);
    v = dpp_add<0x141, 0xf>(v);
    return dpp_add<0x140, 0xf>(v);
}
__device__ __forceinline__ float row16_sum(float v) { return seg_sum<16>(v); }
__device__ __forceinline__ double wave_sum63(double v) { return dpp_add<0x143, 0xc>(dpp_add<0x142, 0xa>(row16_sum(v))); }
__device__ __forceinline__ float wave_sum63(float v) { return seg_sum<64>(v); }

// sum over the workgroup: every wave puts its sums into slots, every thread gets the total of the sixteen slots.  They hold
// zeros before (slots that nobody puts to stay zero) and one slot array serves one sum
template <typename T>
__device__ __forceinline__ void put_sum(T v, T *s_part, uint32_t slot) {
    const T total = wave_sum63(v);
    if ((threadIdx.x & 63) == 63) s_part[slot] = total;
}
template <typename T>
__device__ __forceinline__ T wg_sum(const T *s_part) {
    __syncthreads();
    return row16_sum(s_part[threadIdx.x & 15]);
}

// what the mean square is summed in: f64, or f32 for the unit-offset form
template <bool kUnit>
struct NormSum {
    typedef double type;
};
template <>
struct NormSum<true> {
    typedef float type;
};
template <bool kUnit>
__device__ __forceinline__ void add_squares(typename NormSum<kUnit>::type &acc, const float4 v) {
    typedef typename NormSum<kUnit>::type T;
    acc += static_cast<T>(v.x) * static_cast<T>(v.x);
    acc += static_cast<T>(v.y) * static_cast<T>(v.y);
    acc += static_cast<T>(v.z) * static_cast<T>(v.z);
    acc += static_cast<T>(v.w) * static_cast<T>(v.w);
}
template <bool kUnit>
__device__ __forceinline__ float rms_of(uint32_t nb, float eps, const typename NormSum<kUnit>::type *s_part) {
    const float n = static_cast<float>(nb) * 256.0f;
    if constexpr (kUnit)
        return sqrtf(wg_sum(s_part) / n + eps);
    else
        return static_cast<float>(sqrt(wg_sum(s_part) / static_cast<double>(n) + static_cast<double>(eps)));
}

template <bool kUnit>
__device__ __forceinline__ float4 unit_scale(float4 w) {
    if constexpr (kUnit) w = make_float4(1.0f + w.x, 1.0f + w.y, 1.0f + w.z, 1.0f + w.w);
    return w;
}

// One workgroup per token row; wave w owns the 256-element blocks w, w + waves, ... of the row, lane l the elements
// 4l .. 4l+3 of a block.  kAdd: residual += norm(input, post_weight) first, then the row that is normalised with `weight`
// is the new residual; else it is `input`.  out_f32 and the Q8_K outputs are optional (null).
//
// A row is a few KB, so the kernel is a chain of latencies: one round trip for everything it reads, a sum across the
// workgroup per norm, the quantiser.  Hence up to sixteen waves, so that the blocks of a row of up to 4096 elements run side
// by side, and kPer > 0: a wave's kPer blocks of the input, the residual and both weights are requested together in front
// of the first sum and stay in registers (rows of up to kPer * 16 blocks).  One row of 4096 with the residual add: 9.4 ->
// 5.2 us (6.1 -> 3.8 us without it, twelve rows 10.0 -> 5.8); with four waves that read the row again for every step each
// wave went through four blocks and four dependent round trips, and with loads behind `b < nb` (four dword loads and a
// branch each) sixteen waves took 7.6.  kPer == 0 is the form for longer rows: blocks are read again in each step.  It is also
// the form for many rows (kByBlock, four waves): rows of other workgroups hide a row's latencies then, and sixteen waves
// that wait for each other leave the chip less to do: 2048 rows of 1536 with the residual add 15.4 us with a wave per block
// against 13.2, of 4096 without it 19.4 against 17.7 (4096 x 640 rows 9.3 : 8.8; x 512 7.3 : 7.7; four waves with their
// blocks in registers 19.2 at 2048 rows).  Its blocks' sums are added as the wave per block adds them: a row's bits do not
// depend on the number of rows.
template <bool kAdd, bool kUnitPost, bool kUnit, int kPer, bool kByBlock>
__global__ void __launch_bounds__(kWave * kNormMaxWaves)
    rms_norm_kernel(const float *__restrict__ input, const float *__restrict__ post_weight, float post_eps,
                    float *__restrict__ residual, const float *__restrict__ weight, float eps, uint32_t nb,
                    float *__restrict__ out_f32, int8_t *__restrict__ qs, float *__restrict__ d_out,
                    int16_t *__restrict__ bsums, uint8_t *__restrict__ digits) {
    constexpr int kHeld = kPer > 0 ? kPer : 1;
    __shared__ typename NormSum<kUnitPost>::type s_post[kNormMaxWaves];
    __shared__ typename NormSum<kUnit>::type s_sum[kNormMaxWaves];
    const int lane = threadIdx.x & 63;
    const uint32_t wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const size_t row = blockIdx.x, hidden = static_cast<size_t>(nb) * 256;
    const float4 *x = reinterpret_cast<const float4 *>(input + row * hidden) + lane;
    const float4 *pw = reinterpret_cast<const float4 *>(post_weight) + lane, *nw = reinterpret_cast<const float4 *>(weight) + lane;
    float4 *res = kAdd ? reinterpret_cast<float4 *>(residual + row * hidden) + lane : nullptr;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);

    float4 v[kHeld], w[kHeld];
    [[maybe_unused]] float4 r[kHeld], p[kHeld];
    if constexpr (kPer > 0) {
#pragma unroll
        for (int i = 0; i < kPer; i++) {
            const uint32_t b = wave + i * waves;
            const size_t at = static_cast<size_t>(min(b, nb - 1)) * 64;  // a load in a branch would be four of one dword
            v[i] = x[at];
            if constexpr (kAdd) {
                r[i] = res[at];
                p[i] = pw[at];
            }
            w[i] = nw[at];
        }
#pragma unroll
        for (int i = 1; i < kPer; i++)
            if (wave + i * waves >= nb) v[i] = zero;  // not in the sums (kPer == 1: a wave per block)
    }
    if (threadIdx.x < kNormMaxWaves) {
        if constexpr (kAdd) s_post[threadIdx.x] = 0;
        s_sum[threadIdx.x] = 0;
    }
    __syncthreads();

    // squares of a block: into the wave's sum, or (kByBlock) a sum and a slot of its own
    auto square = [&](auto unit, auto &acc, auto *s_part, uint32_t b, const float4 q) {
        if constexpr (kByBlock) acc = 0;
        add_squares<decltype(unit)::value>(acc, q);
        if constexpr (kByBlock) put_sum(acc, s_part, b);
    };
    const std::bool_constant<kUnitPost> post{};
    const std::bool_constant<kUnit> pre{};
    typename NormSum<kUnit>::type acc = 0;
    if constexpr (kAdd) {
        typename NormSum<kUnitPost>::type pacc = 0;
        if constexpr (kPer > 0) {
#pragma unroll
            for (int i = 0; i < kPer; i++) square(post, pacc, s_post, wave + i * waves, v[i]);
        } else {
            for (uint32_t b = wave; b < nb; b += waves) square(post, pacc, s_post, b, x[static_cast<size_t>(b) * 64]);
        }
        if constexpr (!kByBlock) put_sum(pacc, s_post, wave);
        const float post_rms = rms_of<kUnitPost>(nb, post_eps, s_post);
        auto add = [&](float4 q, const float4 a, const float4 raw) {
            const float4 s = unit_scale<kUnitPost>(raw);
            q.x += (a.x / post_rms) * s.x;
            q.y += (a.y / post_rms) * s.y;
            q.z += (a.z / post_rms) * s.z;
            q.w += (a.w / post_rms) * s.w;
            return q;
        };
        if constexpr (kPer > 0) {
#pragma unroll
            for (int i = 0; i < kPer; i++) {
                const uint32_t b = wave + i * waves;
                v[i] = add(r[i], v[i], p[i]);
                if (b < nb) {
                    res[static_cast<size_t>(b) * 64] = v[i];
                    square(pre, acc, s_sum, b, v[i]);
                }
            }
        } else {
            for (uint32_t b = wave; b < nb; b += waves) {
                const size_t at = static_cast<size_t>(b) * 64;
                const float4 q = add(res[at], x[at], pw[at]);
                res[at] = q;  // read again below by the same thread
                square(pre, acc, s_sum, b, q);
            }
            x = res;
        }
    } else {
        if constexpr (kPer > 0) {
#pragma unroll
            for (int i = 0; i < kPer; i++) square(pre, acc, s_sum, wave + i * waves, v[i]);
        } else {
            for (uint32_t b = wave; b < nb; b += waves) square(pre, acc, s_sum, b, x[static_cast<size_t>(b) * 64]);
        }
    }
    if constexpr (!kByBlock) put_sum(acc, s_sum, wave);
    const float rms = rms_of<kUnit>(nb, eps, s_sum);
    auto finish = [&](uint32_t b, const float4 a, const float4 raw) {
        const float4 s = unit_scale<kUnit>(raw);
        const float4 o = make_float4((a.x / rms) * s.x, (a.y / rms) * s.y, (a.z / rms) * s.z, (a.w / rms) * s.w);
        if (out_f32 != nullptr) reinterpret_cast<float4 *>(out_f32 + row * hidden + static_cast<size_t>(b) * 256)[lane] = o;
        if (qs != nullptr) {
            const size_t blk = row * nb + b;
            q8k_quantize_vals(o, lane, qs + blk * 256, d_out + blk, bsums + blk * 16, digits != nullptr ? digits + blk * 16 : nullptr);
        }
    };
    if constexpr (kPer > 0) {
#pragma unroll
        for (int i = 0; i < kPer; i++) {
            const uint32_t b = wave + i * waves;
            if (b < nb) finish(b, v[i], w[i]);
        }
    } else {
        for (uint32_t b = wave; b < nb; b += waves) finish(b, x[static_cast<size_t>(b) * 64], nw[static_cast<size_t>(b) * 64]);
    }
}

// One wave per token: every lane holds the logits e = lane, lane + 64, ... (at most kRouteMaxPerLane of them); `k`
// rounds of a wave-wide arg-max (larger value first, then the lower expert id) pick the experts in rank order, lane 0
// then forms the softmax over the selected logits in that order.
constexpr int kRouteMaxPerLane = 8;  // up to 512 experts
constexpr int kRouteMaxK = 32;

__global__ void __launch_bounds__(kWave)
    route_topk_kernel(const float *__restrict__ logits, uint32_t n_expert, uint32_t k, uint32_t *__restrict__ idx_out,
                      float *__restrict__ w_out) {
    const int lane = threadIdx.x;
    const size_t tok = blockIdx.x;
    const float *lg = logits + tok * n_expert;
    float v[kRouteMaxPerLane];
#pragma unroll
    for (int i = 0; i < kRouteMaxPerLane; i++) {
        const uint32_t e = lane + 64u * i;
        v[i] = e < n_expert ? lg[e] : -INFINITY;
    }
    uint32_t taken = 0;  // bit i: this lane's i-th logit has been selected
    const uint32_t sel = k < n_expert ? k : n_expert;
    float best_v[kRouteMaxK];
    uint32_t best_e[kRouteMaxK];
    for (uint32_t r = 0; r < sel; r++) {
        // this lane's best remaining candidate: larger value, then lower id (its ids grow with i)
        float cv = -INFINITY;
        uint32_t ce = 0xffffffffu;
#pragma unroll
        for (int i = 0; i < kRouteMaxPerLane; i++) {
            const uint32_t e = lane + 64u * i;
            const bool candidate = e < n_expert && !((taken >> i) & 1u) && !(v[i] != v[i]);  // a NaN is never selected
            if (candidate && (ce == 0xffffffffu || v[i] > cv)) {
                cv = v[i];
                ce = e;
            }
        }
        // wave-wide winner
        float wv = cv;
        uint32_t we = ce;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const float ov = __shfl_xor(wv, off, kWave);
            const uint32_t oe = __shfl_xor(we, off, kWave);
            const bool take = oe != 0xffffffffu && (we == 0xffffffffu || ov > wv || (ov == wv && oe < we));
            wv = take ? ov : wv;
            we = take ? oe : we;
        }
        best_v[r] = wv;
        best_e[r] = we;
        if (we != 0xffffffffu && (we & 63u) == static_cast<uint32_t>(lane)) taken |= 1u << (we >> 6);
    }
    if (lane == 0) {
        const float mx = best_v[0];
        float sum = 0.0f;
        float wts[kRouteMaxK];
        for (uint32_t r = 0; r < sel; r++) {
            wts[r] = expf(best_v[r] - mx);
            sum += wts[r];
        }
        for (uint32_t r = 0; r < sel; r++) {
            idx_out[tok * sel + r] = best_e[r];
            w_out[tok * sel + r] = sum != 0.0f ? wts[r] / sum : wts[r];
        }
    }
}

}  // namespace

void launch_rms_norm(const float *input, const float *post_weight, float post_eps, bool post_unit, float *residual,
                     const float *weight, float eps, bool unit, uint32_t seq, uint32_t nb, float *out_f32, int8_t *qs,
                     float *d, int16_t *bsums, uint8_t *digits, hipStream_t stream) {
    if (seq == 0 || nb == 0) return;
    // rows of up to 16 blocks: a wave per block, or four waves per row for many rows; up to 64 blocks: sixteen waves with
    // their two or four blocks in registers
    const bool many = seq >= kNormManyRows && nb >= 4 && nb <= kNormMaxWaves;
    const uint32_t most = many ? 4 : kNormMaxWaves;
    const uint32_t waves = nb < most ? nb : most, per = (nb + waves - 1) / waves;
    const dim3 grid(seq), block(kWave * waves);
#define RNB_NORM_PER(ADD, UP, U, PER, BY_BLOCK)                                                                         \
    hipLaunchKernelGGL((rms_norm_kernel<ADD, UP, U, PER, BY_BLOCK>), grid, block, 0, stream, input, post_weight, post_eps, \
                       residual, weight, eps, nb, out_f32, qs, d, bsums, digits)
#define RNB_NORM(ADD, UP, U)                    \
    do {                                        \
        if (many)                               \
            RNB_NORM_PER(ADD, UP, U, 0, true);  \
        else if (per == 1)                      \
            RNB_NORM_PER(ADD, UP, U, 1, false); \
        else if (per == 2)                      \
            RNB_NORM_PER(ADD, UP, U, 2, false); \
        else if (per <= 4)                      \
            RNB_NORM_PER(ADD, UP, U, 4, false); \
        else                                    \
            RNB_NORM_PER(ADD, UP, U, 0, false); \
    } while (0)
    if (residual == nullptr) {
        if (unit)
            RNB_NORM(false, false, true);
        else
            RNB_NORM(false, false, false);
    } else if (post_unit) {
        if (unit)
            RNB_NORM(true, true, true);
        else
            RNB_NORM(true, true, false);
    } else {
        if (unit)
            RNB_NORM(true, false, true);
        else
            RNB_NORM(true, false, false);
    }
#undef RNB_NORM_PER
#undef RNB_NORM
}

bool route_topk_supported(uint32_t n_expert, uint32_t k) {
    return n_expert >= 1 && n_expert <= 64u * kRouteMaxPerLane && k >= 1 && k <= kRouteMaxK;
}

void launch_route_topk(const float *logits, uint32_t tokens, uint32_t n_expert, uint32_t k, uint32_t *idx_out, float *w_out,
                       hipStream_t stream) {
    if (tokens == 0) return;
    hipLaunchKernelGGL(route_topk_kernel, dim3(tokens), dim3(kWave), 0, stream, logits, n_expert, k, idx_out, w_out);
}

}  // namespace rnb
