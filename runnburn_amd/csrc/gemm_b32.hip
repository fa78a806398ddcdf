// Prefill GEMM of the 32-element formats (Q8_0, Q8_1, Q4_0, Q4_1, Q5_0, Q5_1) for batches of more than 32 tokens on rows of whole
// 256-element steps: out[seq][rows], same contract as the GEMVs.  Per block of 32 elements
//   out += (d * d_x) * I,  I = sum code * a (exact, one v_mfma_i32_32x32x32_i8)
//   out += (m + c d) * (d_x * sum a), with code - c for the code                 (Q4_1, Q5_1)
// (crates/rnb-cpu/src/gemm/neon_dot.rs:376-436, neon_quant.rs:236-253)
//
// What bounds it is the vector port: a result takes a conversion and a multiply-add per block, 32 instructions of 4 cycles
// beside 96 cycles of matrix pipe.  gemm_blocks.hip's form of the same arithmetic had the port busy 31 % of the time, each pair of
// blocks a chain of products, conversions and updates.  Hence gemm_digits.h's arrangement (256 rows x up to 128 tokens a
// workgroup, codes made once for all its tokens, packed rows and activations by LDS-direct loads, one barrier per 256 elements),
// and the updates of one block beside the products of the next:
//   part 1 of a pair   both blocks' d * d_x (one K = 1 f32 product over two blocks) and the first block's I, beside the update
//                      with the previous pair's second block;
//   part 2             the second block's I, beside the update with the first.
// Two sets of d * d_x, 212 registers with four token tiles.  A pair takes 284 cycles of a wave, 256 of them the update's.
// The mins are a product over the blocks by themselves, m[row][block] against d_x * sum a[block][token]: a K = 2 f32 product per
// pair and one addition per result and step (before: a product with ones, conversion and update per block).  That adds eight blocks'
// codes before their mins, so neither may be large where their sum is small, as d * code and m are with tokens of any mean: codes are
// counted from c, the one nearest to the value 0 of its block, which leaves m + c d of at most d / 2 where a block's values have both
// signs (rms error against f64, gemm_blocks.hip : c = 0 : this, geometric mean of 23 shapes: Q4_1 1.9e-7 : 2.2e-7 : 1.1e-7 with tokens of
// mean 0, 2.4e-7 : 5.5e-7 : 1.0e-7 with mean 1, Q5_1 1.8 : 1.9 : 1.2 and 2.5 : 6.3 : 1.2.  An origin of 8 or 16 would do as well but for blocks
// whose codes are mostly 0.)  It costs 27 vector instructions per pair of blocks and step, 5 % of a call.
// Measured per call (quantiser and slice sum included), gemm_blocks.hip -> this, us: Q8_0 4096 x 4096 x 333 tokens 54.6 -> 34.4, x 2048
// 166 -> 107, 4096 x 14336 x 300 107 -> 80, Q4_0 20 % less on average, Q5_1 4096 x 4096 x 2048 223 -> 178, Q4_1 225 -> 165; over 101 random
// shapes 0.79, the two with mins over 46 0.80.
#include "gemm_digits.h"

namespace rnb {

namespace {

typedef float v32f __attribute__((ext_vector_type(32)));

template <uint32_t kFmt>
struct B32 {
    static constexpr bool kNibbles = kFmt == kQ4_0 || kFmt == kQ4_1 || kFmt == kQ5_0 || kFmt == kQ5_1;
    static constexpr bool kFifth = kFmt == kQ5_0 || kFmt == kQ5_1;
    static constexpr bool kMin = kFmt == kQ4_1 || kFmt == kQ5_1;  // value = d * code + m
    static constexpr float kTop = kFifth ? 31.0f : 15.0f;
    static constexpr int kBytes = kFmt == kQ8_0 ? 34 : kFmt == kQ8_1 ? 36 : kFmt == kQ4_0 ? 18 : kFmt == kQ4_1 ? 20 : kFmt == kQ5_0 ? 22 : 24;
    static constexpr int kQhOff = kMin ? 4 : 2;
    static constexpr int kQsOff = kFmt == kQ8_0 ? 2 : kFmt == kQ8_1 ? 4 : kBytes - 16;
    static constexpr int kStride = 8 * kBytes;      // a row's step, also in the strip
    static constexpr int kPieces = kStride / 16;
    static constexpr int kInv = (65536 + kPieces - 1) / kPieces;  // p * kInv >> 16 = p / kPieces for the 576 pieces of a strip
    static constexpr int kFills = (32 * kPieces + kWave - 1) / kWave;
};

// kWords dwords from byte kOff of a row in the strip (rows are 16-byte aligned, blocks of 18, 22 and 34 bytes are not)
template <int kOff, int kWords>
__device__ __forceinline__ void strip_words(const uint8_t *row, uint32_t (&out)[kWords]) {
    const uint32_t *p = reinterpret_cast<const uint32_t *>(row + (kOff & ~3));
    if constexpr (kOff % 4 == 0) {
#pragma unroll
        for (int i = 0; i < kWords; i++) out[i] = p[i];
    } else {
        uint32_t v[kWords + 1];
#pragma unroll
        for (int i = 0; i <= kWords; i++) v[i] = p[i];
#pragma unroll
        for (int i = 0; i < kWords; i++) out[i] = __builtin_amdgcn_alignbit(v[i + 1], v[i], 16);
    }
}
template <int kOff>
__device__ __forceinline__ uint32_t strip_half(const uint8_t *row) {
    return *reinterpret_cast<const uint16_t *>(row + kOff);
}

// a lane's share of block kK of a step: its 16 codes as signed bytes, d and m
template <uint32_t kFmt>
struct B32Block {
    uint32_t q[4], qh;
    uint32_t dh;
    template <int kK>
    __device__ __forceinline__ void fetch(const uint8_t *row, int khalf) {
        typedef B32<kFmt> F;
        constexpr int at = kK * F::kBytes;
        strip_words<at + F::kQsOff, 4>(row + (F::kNibbles ? 0 : 16 * khalf), q);
        if constexpr (F::kFifth) {
            uint32_t h[1];
            strip_words<at + F::kQhOff, 1>(row, h);
            qh = h[0];
        }
        if constexpr (F::kMin) {  // d | m << 16
            uint32_t h[1];
            strip_words<at, 1>(row, h);
            dh = h[0];
        } else {
            dh = strip_half<at>(row);
        }
    }
    // nibbles by K-half, fifth bits spread with one multiply per four (bit j of a 4-bit group to bit 8 j), the symmetric formats'
    // offset (8, 16) and the others' origin (zero_bytes: 128 - origin in each byte) taken in packed bytes
    __device__ __forceinline__ v4i codes(int khalf, [[maybe_unused]] uint32_t zero_bytes) const {
        typedef B32<kFmt> F;
        v4i o;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t v = q[i];
            if constexpr (F::kNibbles) {
                v = (v >> (4 * khalf)) & 0x0f0f0f0fu;
                if constexpr (F::kFifth) v |= ((((qh >> (16 * khalf + 4 * i)) & 0xfu) * 0x00204081u) & 0x01010101u) << 4;
                if constexpr (kFmt == kQ4_0) v = (v + 0x78787878u) ^ 0x80808080u;  // n - 8 per byte, no carries
                if constexpr (kFmt == kQ5_0) v = (v + 0x70707070u) ^ 0x80808080u;  // n - 16
                if constexpr (F::kMin) v = (v + zero_bytes) ^ 0x80808080u;         // n - origin
            }
            o[i] = static_cast<int>(v);
        }
        return o;
    }
};

template <uint32_t kFmt, int kT>
struct B32Lds {
    static constexpr int kToks = 32 * kT;
    static constexpr int kStrip = B32<kFmt>::kFills * 1024;
    static constexpr int kABuf = kToks / 4 * kDgActGroup;
    static constexpr int kA = kDgWaves * kStrip;
    static constexpr int kDxBuf = kToks * 32;  // eight scales per token
    static constexpr int kDx = kA + 2 * kABuf;
    static constexpr int kBytes = kDx + 2 * kDxBuf;
    static_assert(kBytes <= 160 * 1024, "LDS of a compute unit");
};

template <uint32_t kFmt, int kT>
__global__ void __launch_bounds__(kDgThreads, 2)
    gemm_b32_kernel(const uint8_t *__restrict__ w, const int8_t *__restrict__ aq, const float *__restrict__ ad,
                    float *__restrict__ out, uint32_t rows, uint32_t nb, uint32_t seq, uint32_t nb_slice) {
    typedef B32Lds<kFmt, kT> L;
    typedef B32<kFmt> F;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 31, khalf = lane >> 5;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lptr_t)lds));
    const uint32_t row0 = blockIdx.x * kDgRows + wave * 32;
    const uint32_t first = min(row0, rows - 1), last_row = min(rows - 1 - first, 31u);  // clamped loads, masked stores
    const uint32_t tok0 = blockIdx.y * L::kToks, last_tok = seq - 1 - tok0;
    const uint32_t row_bytes = nb * static_cast<uint32_t>(F::kStride);

    // K slice of this workgroup (blockIdx.z): steps slice0 .. slice0 + nbs, its sums go to the slice's own copy of the output
    const uint32_t slice0 = blockIdx.z * nb_slice, nbs = min(nb - slice0, nb_slice);
    out += static_cast<size_t>(blockIdx.z) * seq * rows;
    const uint8_t *w_base = w + static_cast<size_t>(first) * row_bytes + static_cast<size_t>(slice0) * F::kStride;
    const uint8_t *a_base = reinterpret_cast<const uint8_t *>(aq) + (static_cast<size_t>(tok0) * nb + slice0) * 256;
    const uint8_t *dx_base = reinterpret_cast<const uint8_t *>(ad) + (static_cast<size_t>(tok0) * nb + slice0) * 32;
    const uint8_t *strip_row = lds + wave * L::kStrip + lrow * F::kStride;

    // the lanes' offsets are made anew for each request: kept for the whole loop they would cost registers it has not got
    auto fresh = [&](uint32_t v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    auto issue_w = [&](uint32_t b) {
        const uint8_t *src = w_base + b * static_cast<uint32_t>(F::kStride);
        const uint32_t l = fresh(lane);
#pragma unroll
        for (int k = 0; k < F::kFills; k++) {
            const uint32_t p = min(l + k * kWave, 32u * F::kPieces - 1), r = __umul24(p, F::kInv) >> 16;
            lds_fill16(src, __umul24(min(r, last_row), row_bytes) + 16 * (p - r * F::kPieces), lds0 + wave * L::kStrip + k * 1024);
        }
    };
    auto issue_a = [&](uint32_t b) {
        const uint32_t dst = lds0 + L::kA + (b & 1) * L::kABuf;
        const uint8_t *src = a_base + b * 256u;
        const uint32_t l = fresh(lane), col = 16 * ((l & 15) ^ (l >> 4));
#pragma unroll
        for (int k = 0; k < kT; k++) {
            const uint32_t g = k * kDgWaves + wave;  // four tokens
            if (last_tok >= L::kToks - 1)
                lds_fill16(src + static_cast<size_t>(4 * g) * nb * 256u, (l >> 4) * (nb * 256u) + col, dst + g * kDgActGroup);
            else
                lds_fill16(src, min(4 * g + (l >> 4), last_tok) * (nb * 256u) + col, dst + g * kDgActGroup);
        }
        if (wave < kT)  // 32 tokens' scales
            lds_fill16(dx_base + b * 32u, min(wave * 32 + (l >> 1), last_tok) * (nb * 32u) + 16 * (l & 1),
                       lds0 + L::kDx + (b & 1) * L::kDxBuf + wave * 1024);
    };

    float accf[kT][16];
#pragma unroll
    for (int t = 0; t < kT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) accf[t][r] = 0.0f;
    const v16i zero16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const v32f zero32 = {};
    v4i bop[8];      // the present step's codes
    float dk[4];     // d of block 2 p + khalf
    [[maybe_unused]] float mk[4];  // m likewise
    v16i ia, ib = zero16;  // sums of a pair's first and second block
    v32f dd[2];            // d * d_x of a pair's results: [0] of even pairs, [1] of odd ones
    dd[1] = zero32;
    [[maybe_unused]] v16f cm = {};  // the mins' part of a tile and step

    B32Block<kFmt> n0, n1;
    auto of_half = [&](float lower, float upper) {
        asm volatile("" : "+v"(lower), "+v"(upper));
        return khalf ? upper : lower;
    };
    auto take = [&](int p) {  // the next step's pair p in place of the present one
        const float d = of_half(f16_bits_to_f32(n0.dh), f16_bits_to_f32(n1.dh));
        uint32_t zero0 = 0, zero1 = 0;
        dk[p] = d;
        if constexpr (F::kMin) {
            // d n + m = d (n - c) + (m + c d), c the code nearest to the value 0.  (No d, infinities, NaN: c = 0, m as it is.)
            const float m = of_half(f16_bits_to_f32(n0.dh >> 16), f16_bits_to_f32(n1.dh >> 16));
            const float c = __builtin_rintf(fminf(fmaxf(-m * __builtin_amdgcn_rcpf(d), 0.0f), F::kTop));
            mk[p] = c > 0.0f ? __builtin_fmaf(c, d, m) : m;
            const uint32_t z = __builtin_amdgcn_perm(0u, 128u - static_cast<uint32_t>(c), 0u);  // its low byte in all four
            const auto both = __builtin_amdgcn_permlane32_swap(z, z, false, false);
            zero0 = both[0];
            zero1 = both[1];
        }
        bop[2 * p] = n0.codes(khalf, zero0);
        bop[2 * p + 1] = n1.codes(khalf, zero1);
    };
#define RNB_B32_FETCH(P)                            \
    {                                               \
        n0.template fetch<2 * (P)>(strip_row, khalf);     \
        n1.template fetch<2 * (P) + 1>(strip_row, khalf); \
    }
    auto fetch = [&](int p) {
        switch (p) {
        case 0: RNB_B32_FETCH(0) break;
        case 1: RNB_B32_FETCH(1) break;
        case 2: RNB_B32_FETCH(2) break;
        default: RNB_B32_FETCH(3) break;
        }
    };
#undef RNB_B32_FETCH
    // d_x times the sum of the token's activations, of block 2 p in the lower half of the wave and 2 p + 1 in the upper one
    auto pair_sum = [&](const v4i &x0, const v4i &x1, float scale) {
        int h0 = 0, h1 = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            h0 = dot4(static_cast<uint32_t>(x0[i]), 0x01010101u, h0);
            h1 = dot4(static_cast<uint32_t>(x1[i]), 0x01010101u, h1);
        }
        // {h0 lower | h0 upper}, {h1 lower | h1 upper} -> {h0 lower | h1 lower}, {h0 upper | h1 upper}
        const auto s = __builtin_amdgcn_permlane32_swap(h0, h1, false, false);
        return static_cast<float>(static_cast<int>(s[0]) + static_cast<int>(s[1])) * scale;
    };
    auto update = [&](int t, const v16i &sum, const v32f &s, int half, int from, int to) {
#pragma unroll
        for (int r = from; r < to; r++) {
            accf[t][r] = __builtin_fmaf(s[16 * half + r], static_cast<float>(sum[r]), accf[t][r]);
            asm volatile("" : "+v"(accf[t][r]));
        }
    };

    issue_w(0);
    issue_a(0);
    wait_fills();
#pragma unroll
    for (int p = 0; p < 4; p++) {
        fetch(p);
        take(p);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (nbs > 1) issue_w(1);

    for (uint32_t b = 0; b < nbs; b++) {
        // this wave's pieces of step b have landed (waited for below); behind the barrier everyone's have, and nobody reads
        // step b - 1 any more
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (b + 1 < nbs) issue_a(b + 1);
        // token lrow of tile t, block k: column 2 k + khalf at place (2 k + khalf) ^ (lrow & 3)
        const uint8_t *abase = lds + L::kA + (b & 1) * L::kABuf + (lrow >> 2) * kDgActGroup + (lrow & 3) * 256 + 16 * (khalf ^ (lrow & 1));
        const uint8_t *apos[2] = {abase + 16 * (lrow & 2), abase - 16 * (lrow & 2)};  // even and odd k
        const float *dxp = reinterpret_cast<const float *>(lds + L::kDx + (b & 1) * L::kDxBuf) + lrow * 8 + khalf;
        auto act_operand = [&](int t, int k) { return *reinterpret_cast<const v4i *>(apos[k & 1] + 8 * t * kDgActGroup + 32 * k); };
        v4i a0 = act_operand(0, 0), a1 = act_operand(0, 1);
        float dx = dxp[0];
#pragma unroll
        for (int t = 0; t < kT; t++) {
            const int tp = t == 0 ? kT - 1 : t - 1;
            if (t == kT - 1) wait_fills();  // the next step's activations and packed rows
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const int q = 4 * t + p, now = p & 1;
                const v4i x0 = a0, x1 = a1;
                const float xs = dx;
                // first block: its products and both blocks' scales, beside the update with the previous pair's second block
                dd[now] = __builtin_amdgcn_mfma_f32_32x32x1f32(xs, dk[p], zero32, 0, 0, 0);
                asm volatile("" : "+v"(dd[now]));  // pins the instruction inside its group
                update(p == 0 ? tp : t, ib, dd[now ^ 1], 1, 0, 8);
                ia = __builtin_amdgcn_mfma_i32_32x32x32_i8(x0, bop[2 * p], zero16, 0, 0, 0);
                asm volatile("" : "+v"(ia));
                if (q + 1 < 4 * kT) {
                    a0 = act_operand((q + 1) >> 2, 2 * ((q + 1) & 3));
                    a1 = act_operand((q + 1) >> 2, 2 * ((q + 1) & 3) + 1);
                    dx = dxp[256 * ((q + 1) >> 2) + 2 * ((q + 1) & 3)];
                }
                update(p == 0 ? tp : t, ib, dd[now ^ 1], 1, 8, 16);
                [[maybe_unused]] float ps = 0.0f;
                if constexpr (F::kMin) ps = pair_sum(x0, x1, xs);
                __builtin_amdgcn_sched_barrier(0);
                // second block: its products, beside the update with the first
                ib = __builtin_amdgcn_mfma_i32_32x32x32_i8(x1, bop[2 * p + 1], zero16, 0, 0, 0);
                asm volatile("" : "+v"(ib));
                if (t == kT - 1) fetch(p);
                update(t, ia, dd[now], 0, 0, 16);
                if constexpr (F::kMin) {  // the mins of a tile's eight blocks are a product over the blocks: no update of their own
                    if (p == 0)
#pragma unroll
                        for (int r = 0; r < 16; r++) accf[tp][r] += cm[r];
                    cm = __builtin_amdgcn_mfma_f32_32x32x2f32(ps, mk[p], p == 0 ? v16f{} : cm, 0, 0, 0);
                    asm volatile("" : "+v"(cm));
                }
                if (t == kT - 1) {
                    take(p);
                    asm volatile("" : "+v"(bop[2 * p]), "+v"(bop[2 * p + 1]), "+v"(dk[p]));
                    if constexpr (F::kMin) asm volatile("" : "+v"(mk[p]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the strip has been read
        if (b + 2 < nbs) issue_w(b + 2);
    }
    update(kT - 1, ib, dd[1], 1, 0, 16);
    if constexpr (F::kMin)
#pragma unroll
        for (int r = 0; r < 16; r++) accf[kT - 1][r] += cm[r];

    if (row0 + lrow < rows) {
#pragma unroll
        for (int t = 0; t < kT; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const uint32_t tok = tok0 + 32 * t + 8 * (r >> 2) + 4 * khalf + (r & 3);
                if (tok < seq) out[static_cast<size_t>(tok) * rows + row0 + lrow] = accf[t][r];
            }
    }
}

template <uint32_t kFmt, int kT>
void launch_b32(const DgPlan &p, const uint8_t *w, const ActView &act, float *out, float *slice_out, uint32_t rows, uint32_t nb,
                uint32_t seq, hipStream_t stream) {
    static bool configured = false;  // above the default 64 KB of dynamic LDS
    constexpr size_t lds = B32Lds<kFmt, kT>::kBytes;
    if (!allow_dynamic_lds(reinterpret_cast<const void *>(gemm_b32_kernel<kFmt, kT>), lds, &configured, "gemm_b32_kernel")) return;
    const uint32_t slices = slice_out ? p.slices : 1;
    const uint32_t nb_slice = (nb + slices - 1) / slices, nz = (nb + nb_slice - 1) / nb_slice;
    hipLaunchKernelGGL((gemm_b32_kernel<kFmt, kT>), dim3(p.row_tiles, p.groups, nz), dim3(kDgThreads), lds, stream, w, act.qs, act.d,
                       nz > 1 ? slice_out : out, rows, nb, seq, nb_slice);
    if (nz > 1) launch_sum_slices(slice_out, out, static_cast<size_t>(seq) * rows, nz, stream);
}

// One workgroup fits a compute unit, so 256 run at once.  A step costs it about 0.8 tile's time beside its tiles (operands,
// requests, the barrier; Q8_0 0.9 us and 1.08 us a tile, 284 cycles a pair of blocks and wave), its two ends about two; the sum
// of the slices about three and what its reads take (5.5 MB in a tile's time).  The least over two to four tiles a workgroup (two
// or three where there are mins: four would spill 55 registers) and up to 16 slices, whose partial sums stay within
// kSliceScratchBytes.  4096 x 4096 x 333 tokens: three tiles, four slices 34.4 us (four and four 39.0, two and two 38.1, two and
// three, 288 workgroups, 42.1); 4096 x 14336 x 300 two and three 79.8 (three and four 81.8, two and two 106.5); 1000 x 2816 x 130
// two and eight 16.3 (four 18.7, one 39.3).
DgPlan b32_plan(uint32_t quant, uint32_t rows, uint32_t nb, uint32_t seq) {
    const uint32_t tiles = (seq + 31) / 32;
    DgPlan best{};
    double best_cost = 1e30;
    for (uint32_t per = quant == kQ4_1 || quant == kQ5_1 ? 3 : 4; per >= 2; per--) {
        DgPlan p;
        p.tiles_per_wg = per;
        p.groups = (tiles + per - 1) / per;
        p.row_tiles = (rows + kDgRows - 1) / kDgRows;
        const uint64_t wgs = static_cast<uint64_t>(p.row_tiles) * p.groups;
        for (p.slices = 1; p.slices <= 16 && p.slices <= nb; p.slices++) {
            const uint64_t floats = static_cast<uint64_t>(p.slices) * rows * seq;
            if (p.slices > 1 && floats * sizeof(float) > kSliceScratchBytes) break;
            const uint32_t steps = (nb + p.slices - 1) / p.slices, nz = (nb + steps - 1) / steps;
            const double cost = static_cast<double>((wgs * nz + 255) / 256) * (steps * (per + 0.8) + 2.0) +
                                (nz > 1 ? 3.0 + nz * static_cast<double>(rows) * seq * 4.0 / 5.5e6 : 0.0);
            if (cost < best_cost) {
                best_cost = cost;
                best = p;
                best.slices = nz;
            }
        }
    }
    return best;
}

template <uint32_t kFmt>
void launch_b32_plan(const uint8_t *w, const ActView &act, float *out, float *slice_out, uint32_t rows, uint32_t nb, uint32_t seq,
                     hipStream_t stream) {
    const DgPlan p = b32_plan(kFmt, rows, nb, seq);
    if (p.tiles_per_wg == 3)
        launch_b32<kFmt, 3>(p, w, act, out, slice_out, rows, nb, seq, stream);
    else if (p.tiles_per_wg == 2)
        launch_b32<kFmt, 2>(p, w, act, out, slice_out, rows, nb, seq, stream);
    else if constexpr (!B32<kFmt>::kMin)
        launch_b32<kFmt, 4>(p, w, act, out, slice_out, rows, nb, seq, stream);
}

}  // namespace

// Ahead of gemm_blocks.hip everywhere but on Q8_1, whose 36-byte blocks that kernel loads at 4-byte boundaries, where rows are
// short or the last tile of 256 rows is most of them (590 x 1024 x 1414 tokens 21.8 us there against 23.8 here, 736 x 5120 x 90 17.4
// against 18.2; 1030 x 1280 x 700 level; Q8_0 512 x 1024 x 33 15.4 against 11.0), and in less than a round of workgroups on rows of a step or
// two of the formats whose codes take longest to make, which nothing stands beside there (Q5_1 355 x 256 x 104 10.4 against 11.6, 3650 x
// 512 x 407 16.5 against 17.6, Q5_0 5901 x 256 x 225 10.6 against 11.1; 17600 x 256 x 1170 52.7 against 43.1; Q5_0 x 512 within 2 %).
bool gemm_b32_pays(uint32_t quant, const uint8_t *w, size_t rows, size_t cols, size_t seq) {
    if (quant == kQ8_1 && (rows <= 768 || cols <= 1024)) return false;
    if (cols <= (quant == kQ5_1 ? 512 : quant == kQ5_0 ? 256 : 0) && rows * seq <= 2000000) return false;
    return seq > 32 && cols % 256 == 0 && reinterpret_cast<uintptr_t>(w) % 4 == 0 && cols < (size_t(1) << 23);
}

size_t gemm_b32_slice_floats(uint32_t quant, uint32_t rows, uint32_t nb, uint32_t seq) {
    if (rows == 0 || nb == 0 || seq == 0) return 0;
    const DgPlan p = b32_plan(quant, rows, nb, seq);
    return p.slices > 1 ? static_cast<size_t>(p.slices) * seq * rows : 0;
}

void launch_gemm_b32(const uint8_t *w, uint32_t quant, ActView act, float *out, float *slice_out, uint32_t rows, uint32_t nb,
                     uint32_t seq, hipStream_t stream) {
    if (rows == 0 || seq == 0 || nb == 0) return;
    switch (quant) {
    case kQ8_0: launch_b32_plan<kQ8_0>(w, act, out, slice_out, rows, nb, seq, stream); break;
    case kQ8_1: launch_b32_plan<kQ8_1>(w, act, out, slice_out, rows, nb, seq, stream); break;
    case kQ4_0: launch_b32_plan<kQ4_0>(w, act, out, slice_out, rows, nb, seq, stream); break;
    case kQ4_1: launch_b32_plan<kQ4_1>(w, act, out, slice_out, rows, nb, seq, stream); break;
    case kQ5_0: launch_b32_plan<kQ5_0>(w, act, out, slice_out, rows, nb, seq, stream); break;
    default: launch_b32_plan<kQ5_1>(w, act, out, slice_out, rows, nb, seq, stream); break;
    }
}

}  // namespace rnb
