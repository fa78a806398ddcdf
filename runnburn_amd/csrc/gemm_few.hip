// GEMM of a few tokens (sequences decoding together, speculative tokens): up to 32 tokens against Q4_K, Q5_K or Q6_K rows,
// out[seq][rows], same contract as the GEMVs.
//
// A matrix is read once and little is computed per byte, so what counts is how evenly and how early its bytes are asked for,
// and how many launches stand around the one that reads them:
//   * a wave owns 16 or 32 rows and every slices-th block of them; the K slices of a row tile are the waves of ONE
//     workgroup, whose partial sums meet in LDS.  No partial sums in memory, no second kernel (4 us), no workspace.
//   * every wave runs by itself: its next block's rows, activations and digits are on their way into its own stage of LDS
//     (LDS-direct loads, no registers, no barrier) while the present block, read into registers first, is multiplied.
//   * slices are interleaved, so the waves of a workgroup read neighbouring blocks, which share cache lines (14336 x 4096
//     Q4_K, 12 tokens, with the quantiser's launch: 14.6 us with contiguous slices, 13.0 interleaved).
//   * v_mfma_i32_16x16x64_i8: tiles of 16 tokens, so a dozen do not pay for 32.  Integer scales ride on the operands (Q4_K two
//     octal digits; Q5_K the same and the fifth bits as a third chain; Q6_K 16-bit products cut base 256), the chains'
//     sums are exact.  I, the mins' S and the float update are gemm_blocks.hip's:
//     out += d_x * (d * I - dmin * S)   (crates/rnb-cpu/src/gemm/neon_dot.rs:884-916, :1742-1800, :2240-2288)
// Measured per call, quantiser included, before (gemm_blocks.hip with K slices in memory, or GEMV passes of four tokens) ->
// after: 12 tokens 14336 x 4096 Q4_K 15.2 -> 11.8 us (33 MB in 9 us), 4096 x 4096 10.0 -> 7.4, 4096 x 14336 Q6_K 23.5 -> 17.3,
// 13824 x 5120 Q5_K at 21 tokens 26.8 -> 23.9; gate and up in one launch, with SiLU and the down projection 50 -> 37.  Two
// empty launches take 5.9 us.  Parts taken out of the 12-token Q4_K case (13.0 us there): products 1.0, activations 1.4,
// tokens' scales and digits 0.6, packed rows 5.  A second stage per wave gained nothing (14.1): waves in flight do.
#include "gemm_few.h"

namespace rnb {

namespace {

template <uint32_t kFmt, int kMT, int kN, int kWaves, int kMats, bool kGelu>
__global__ void __launch_bounds__(kWave *kWaves)
    gemm_few_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ w2, const int8_t *__restrict__ aq,
                    const float *__restrict__ ad, const uint8_t *__restrict__ adig, float *__restrict__ out, uint32_t rows,
                    uint32_t nb, uint32_t seq, uint32_t log_slices) {
    typedef FewLds<kFmt, kMT, kN, kMats> L;
    typedef FewRows<kFmt> R;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, kq = lane >> 4;
    const uint32_t slices = 1u << log_slices, group = wave >> log_slices, sl = wave & (slices - 1);
    const uint32_t row0 = (blockIdx.x * (kWaves >> log_slices) + group) * (16 * kN);
    const uint32_t first = min(row0, (rows - 1) & ~15u), last_row = min(rows - 1 - first, 16u * kN - 1);  // clamped loads, masked stores
    const uint32_t row_bytes = nb * static_cast<uint32_t>(R::kBytes), last_tok = seq - 1;
    // K slice of the wave: blocks sl, sl + slices, ...: the waves of a workgroup read neighbouring blocks at the same time
    uint8_t *stage = lds + wave * L::kStage;
    float *scales = reinterpret_cast<float *>(lds + kWaves * L::kStage);
    const uint32_t stage0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lptr_t)lds)) + wave * L::kStage;
    const uint8_t *w_base[2] = {w + static_cast<size_t>(first) * row_bytes, w2 + static_cast<size_t>(first) * row_bytes};

    const uint32_t rr = __umul24(lane, R::kInv) >> 16, j = lane - rr * R::kPieces;
    uint32_t row_off[L::kFills], act_off[4 * kMT];
#pragma unroll
    for (int k = 0; k < L::kFills; k++) row_off[k] = min(k * R::kPer + rr, last_row) * row_bytes;
#pragma unroll
    for (int g = 0; g < 4 * kMT; g++)
        act_off[g] = min(static_cast<uint32_t>(4 * g + kq), last_tok) * (nb * 256u) + 16 * (l16 ^ (4 * (g & 3) + kq));
    uint32_t dig_off[kMT];  // a token's sixteen bytes are four lanes' dwords
#pragma unroll
    for (int t = 0; t < kMT; t++) dig_off[t] = min(static_cast<uint32_t>(16 * t + (lane >> 2)), last_tok) * (nb * 16u) + 4 * (lane & 3);
    auto issue = [&](uint32_t b) {
#pragma unroll
        for (int m = 0; m < kMats; m++) {
            const uint8_t *src = w_base[m] + R::block_off(b);
#pragma unroll
            for (int k = 0; k < L::kFills; k++) lds_fill16(src, R::piece(row_off[k], j, b), stage0 + m * L::kStrip + k * 1024);
        }
        const uint8_t *act = reinterpret_cast<const uint8_t *>(aq) + b * 256u;
#pragma unroll
        for (int g = 0; g < 4 * kMT; g++)
            if (4u * g < seq) lds_fill16(act, act_off[g], stage0 + L::kAct + g * 1024);  // places of no token keep what they hold
        if constexpr (R::kMins)
#pragma unroll
            for (int t = 0; t < kMT; t++) lds_fill4(adig + b * 16u, dig_off[t], stage0 + L::kDig + t * 256);
    };
    float acc[kMats][kN][kMT][4];
#pragma unroll
    for (int m = 0; m < kMats; m++)
#pragma unroll
        for (int n = 0; n < kN; n++)
#pragma unroll
            for (int t = 0; t < kMT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[m][n][t][r] = 0.0f;
    if (sl < nb) issue(sl);
    // the tokens' scales of every block: [block][token]
    for (uint32_t i = threadIdx.x; i < 16 * kMT * nb; i += kWave * kWaves) {
        const uint32_t t = i / nb, b = i - t * nb;
        scales[b * (16 * kMT) + t] = ad[min(t, last_tok) * nb + b];
    }
    __syncthreads();
    for (uint32_t b = sl; b < nb; b += slices) {
        wait_fills();
        FewBlock<kFmt, kMT, kN, kMats> blk;
        blk.read(stage, L::kAct, L::kDig, scales + b * (16 * kMT), l16, kq, last_row, nb, b);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage has been read
        if (b + slices < nb) issue(b + slices);
        blk.template multiply<false>(acc, kq);
    }

    // partial sums of the K slices: each wave's into its own stage, whose last loads have been read
#pragma unroll
    for (int m = 0; m < kMats; m++)
#pragma unroll
        for (int n = 0; n < kN; n++)
#pragma unroll
            for (int t = 0; t < kMT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    reinterpret_cast<float *>(stage)[(((m * kN + n) * kMT + t) * 4 + r) * kWave + lane] = acc[m][n][t][r];
    __syncthreads();
    const uint8_t *parts = lds + group * slices * L::kStage;
    for (uint32_t e = sl; e < kN * kMT * 4; e += slices) {  // (row tile, token tile, result)
        float v[2] = {0.0f, 0.0f};
#pragma unroll
        for (int m = 0; m < kMats; m++) {
            const uint8_t *p = parts + ((m * kN * kMT * 4 + e) * kWave + lane) * 4;
            float sum = *reinterpret_cast<const float *>(p);
            for (uint32_t s = 1; s < slices; s++) sum += *reinterpret_cast<const float *>(p + s * L::kStage);
            v[m] = sum;
        }
        const uint32_t r = e & 3, t = (e >> 2) % kMT, n = (e >> 2) / kMT;
        const uint32_t tok = 16 * t + 4 * kq + r, row = row0 + 16 * n + l16;
        if (tok < seq && row < rows) out[static_cast<size_t>(tok) * rows + row] = kMats == 2 ? act_mul<kGelu>(v[0], v[1]) : v[0];
    }
}

template <uint32_t kFmt, int kMT, int kN, int kWaves, int kMats, bool kGelu>
void launch_few(const uint8_t *w, const uint8_t *w2, const ActView &act, float *out, uint32_t rows, uint32_t nb, uint32_t seq,
                uint32_t slices, hipStream_t stream) {  // slices: a power of two, at most kWaves
    static bool configured = false;
    constexpr size_t most = kWaves * FewLds<kFmt, kMT, kN, kMats>::kStage + kFewMaxBlocks * 16 * kMT * sizeof(float);
    static_assert(most <= 160 * 1024, "LDS of a compute unit");
    const size_t lds = kWaves * FewLds<kFmt, kMT, kN, kMats>::kStage + static_cast<size_t>(nb) * 16 * kMT * sizeof(float);
    if (!allow_dynamic_lds(reinterpret_cast<const void *>(gemm_few_kernel<kFmt, kMT, kN, kWaves, kMats, kGelu>), most, &configured,
                           "gemm_few_kernel"))
        return;
    const uint32_t per_wg = kWaves / slices * 16 * kN;
    hipLaunchKernelGGL((gemm_few_kernel<kFmt, kMT, kN, kWaves, kMats, kGelu>), dim3((rows + per_wg - 1) / per_wg), dim3(kWave * kWaves),
                       lds, stream, w, w2, act.qs, act.d, act.digits, out, rows, nb, seq, __builtin_ctz(slices));
}

struct FewPlan {
    int row_tiles, waves;  // 16-row tiles per wave, waves per workgroup
    uint32_t slices;
};
// Sixteen rows a wave and eight slices as long as there is a compute unit for each workgroup (4096 x 14336 Q6_K, 12 tokens: 17.3
// us against 19.7 with four slices and 27.7 with 32 rows); then four slices, three to five workgroups a unit; 32 rows a wave,
// which read the activations half as often, on large matrices (28672 x 8192 Q4_K: 30.6 against 32.8) and where the workgroups
// of 17 to 32 tokens on Q4_K and Q5_K would leave the second round nearly empty (14336 x 4096 Q4_K, 24 tokens: 15.6 against
// 16.8; 10240 rows 15.2 against 13.5).  Two slices where rows are short or many enough to fill the chip with those (28672 x
// 1024 Q4_K, 24 tokens 13.6 -> 12.7, 65536 x 4096 Q6_K, 24 tokens 71.9 -> 66.7).
FewPlan few_plan(uint32_t quant, uint32_t rows, uint32_t nb, uint32_t seq) {
    const uint32_t tiles = (rows + 15) / 16;
    FewPlan p{1, 4, 4};
    if (tiles <= 256) {
        p = {1, 8, 8};
    } else if (static_cast<uint64_t>(rows) * nb > 400000 || (seq > 16 && quant != kQ6K && tiles > 768)) {
        p = {2, 4, tiles > (seq > 16 ? 1600u : 4000u) ? 2u : 4u};
    } else if (tiles > 1280 && nb <= 8) {
        p.slices = 2;
    }
    while (p.slices > nb) p.slices /= 2;
    return p;
}

template <uint32_t kFmt, int kMT, int kMats, bool kGelu>
void launch_few_tokens(const uint8_t *w, const uint8_t *w2, const ActView &act, float *out, uint32_t rows, uint32_t nb,
                       uint32_t seq, hipStream_t stream) {
    const FewPlan p = few_plan(kFmt, rows, nb, seq);
    if (p.waves == 8)
        launch_few<kFmt, kMT, 1, 8, kMats, kGelu>(w, w2, act, out, rows, nb, seq, p.slices, stream);
    else if (p.row_tiles == 1)
        launch_few<kFmt, kMT, 1, 4, kMats, kGelu>(w, w2, act, out, rows, nb, seq, p.slices, stream);
    else
        launch_few<kFmt, kMT, 2, 4, kMats, kGelu>(w, w2, act, out, rows, nb, seq, p.slices, stream);
}

}  // namespace

// The loads want rows at 4-byte addresses, and the last piece of a Q6_K block ends two bytes behind every other block
// (FewRows<kQ6K>): behind the last one of the matrix where the number of blocks is odd.
bool gemm_few_supported(uint32_t quant, const uint8_t *w, size_t rows, size_t nb, size_t seq) {
    if (quant != kQ4K && quant != kQ5K && quant != kQ6K) return false;
    if (seq > 32 || nb > kFewMaxBlocks || reinterpret_cast<uintptr_t>(w) % 4 != 0) return false;
    return quant != kQ6K || rows * nb % 2 == 0;
}

namespace {

// Where the kernel fits a matrix of this shape.  Ahead of the GEMV passes over up to four tokens (us, GEMV : this kernel): rows of more
// than 16 blocks from three tokens on (4096 x 14336 Q4_K 13.2 : 10.9); shorter ones from four (14336 x 4096 Q4_K 13.5 : 11.6, three 11.2 :
// 11.5), Q6_K five (14336 x 4096 22.6 : 16.4, four 17.6 : 16.6).  The GEMV's rows have the bits of the one-token call, this kernel's sums
// are in an order that depends on the matrix (slices); the same holds either side of the next line.
// Matrices of less than 4 MB keep the GEMV up to eight tokens (Q6_K 1024 x 4096 7.4 : 8.0 at eight, Q4_K 7.5 : 6.8) and its bits.
// Ahead of gemm_blocks.hip everywhere up to 16 tokens, and with Q6_K; 17 to 32 tokens of Q4_K and Q5_K read twice the
// activations per row, which costs more than the slices in memory where a wave has many blocks (24 tokens, Q4_K, gemm_blocks :
// this: 1024 x 14336 12.3 : 14.3, 1024 x 8192 9.9 : 10.6; 2048 x 8192 11.6 : 10.9) or the matrix is large (65536 x 4096 47 : 50, Q5_K
// 28672 x 8192 55 : 57, 28672 x 1024 11.8 : 13.6; 28672 x 4096 Q4_K 30.1 : 28.4, Q5_K 34.0 : 33.4).
bool few_shape(uint32_t quant, size_t rows, size_t nb, size_t seq, size_t bytes) {
    if (seq < 3 || seq > 32) return false;
    if (bytes < (size_t(4) << 20)) {
        if (seq <= 8) return false;
    } else if (nb <= 16 && seq < (quant == kQ6K ? 5 : 4)) {
        return false;
    }
    if (seq <= 16 || quant == kQ6K) return true;
    if (rows <= 1024) return nb <= 16;
    if (rows <= 2048) return nb <= 32;
    if (rows > 24576 && nb < 8) return false;
    return quant == kQ4K ? rows <= 32768 : rows * nb <= 480000;
}

// workgroups of a call over those that its rounds of `at_once` have places for
double rounds_fill(const FewPlan &p, uint32_t rows, uint32_t at_once) {
    const uint32_t per_wg = p.waves / p.slices * 16 * p.row_tiles, wgs = (rows + per_wg - 1) / per_wg;
    return static_cast<double>(wgs) / ((wgs + at_once - 1) / at_once * at_once);
}

}  // namespace

// One matrix (us, the other kernel : this one).  Left to kernels that cut K further: a few row tiles with a long chain of blocks each, up
// to 512 rows (160 x 10752 Q4_K, 11 tokens 6.7 : 8.6, 337 x 15360 Q5_K, 12 10.3 : 12.1; 394 x 9728 Q4_K, 11 9.3 : 8.5), 1024 with three
// tokens (the down projection of an FFN 7680 x 1024 Q4_K 13.1 : 14.4 for the whole layer), three tokens of Q5_K up to 2048 rows of more than
// 32 blocks (eight matrices 0.73 - 1.0), of Q6_K any (41 matrices 0.68 - 1.11), four up to 2400 rows (0.71 - 1.06).
// Left to gemm_blocks.hip where the last round of workgroups is nearly empty and each has much to read: two row tiles a wave over one
// workgroup a unit (Q6_K 8268 x 12544, 13 tokens, 259 workgroups 28.5 : 36.3, Q4_K 8595 x 14592, three, 0.87) and, with 17 to 32 tokens from
// 24 MB on, over the places of all (Q4_K 18981 x 15872 47.4 : 53.4, 17249 x 4352 21.4 : 23.5; Q5_K 9170 x 9216 23.2 : 27.8; 13824 x 5120, 84 %
// full, 23.3 : 20.0); many short rows (19963 x 1536 11.4 : 13.4; 15330 x 1280 10.4 : 9.7).
// Of 927 random matrices that take longer than a launch 34 are more than 3 % behind the kernels before this one (99 by few_shape alone),
// 0.841 of their time on average.
bool gemm_few_pays(uint32_t quant, size_t rows, size_t nb, size_t seq) {
    const size_t bytes = rows * nb * (quant == kQ4K ? kQ4KBytes : quant == kQ5K ? kQ5KBytes : kQ6KBytes);
    if (!few_shape(quant, rows, nb, seq, bytes)) return false;
    if (seq <= 16 && rows <= (seq == 3 ? 1024 : 512)) return false;
    if (seq == 3 && (quant == kQ6K || (quant == kQ5K && rows <= 2048 && nb > 32))) return false;
    if (seq == 4 && quant == kQ6K && rows <= 2400) return false;
    const uint32_t r = static_cast<uint32_t>(rows), b = static_cast<uint32_t>(nb);
    const FewPlan p = few_plan(quant, r, b, static_cast<uint32_t>(seq));
    if (p.row_tiles == 2 && bytes >= (size_t(24) << 20) && rounds_fill(p, r, 256) < 0.65) return false;
    if (seq <= 16 || quant == kQ6K) return true;
    if (rows > 16384 && nb < 8) return false;
    if (bytes < (size_t(24) << 20) || (quant == kQ4K && p.row_tiles == 1)) return true;
    const size_t stage = quant == kQ4K         ? FewLds<kQ4K, 2, 2, 1>::kStage
                         : p.row_tiles == 1 ? FewLds<kQ5K, 2, 1, 1>::kStage
                                            : FewLds<kQ5K, 2, 2, 1>::kStage;
    const size_t lds = p.waves * stage + nb * 32 * sizeof(float);
    return lds <= 160 * 1024 && rounds_fill(p, r, 256 * static_cast<uint32_t>(160 * 1024 / lds)) >= 0.75;
}

// both matrices of a gated FFN; three tokens of short rows: in the paired GEMV 34.2 us for the whole layer against 36.4, four 44 : 36.5
// (rows of more than 16 blocks, which the paired GEMV does not take: 22.6 : 18.8)
bool gemm_few_gate_up_pays(size_t rows, size_t nb, size_t seq) { return few_shape(kQ4K, rows, nb, seq, rows * nb * kQ4KBytes) && (seq > 3 || nb > 16); }

void launch_gemm_few(const uint8_t *w, uint32_t quant, ActView act, float *out, uint32_t rows, uint32_t nb, uint32_t seq,
                     hipStream_t stream) {
    if (rows == 0 || seq == 0 || nb == 0) return;
#define RNB_FEW(FMT)                                                                          \
    if (seq <= 16)                                                                            \
        launch_few_tokens<FMT, 1, 1, false>(w, w, act, out, rows, nb, seq, stream);           \
    else                                                                                      \
        launch_few_tokens<FMT, 2, 1, false>(w, w, act, out, rows, nb, seq, stream)
    if (quant == kQ4K) {
        RNB_FEW(kQ4K);
    } else if (quant == kQ5K) {
        RNB_FEW(kQ5K);
    } else {
        RNB_FEW(kQ6K);
    }
#undef RNB_FEW
}

void launch_gemm_few_gate_up(const uint8_t *wg, const uint8_t *wu, ActView act, float *mid, uint32_t rows, uint32_t nb,
                             uint32_t seq, bool gelu, hipStream_t stream) {
    if (rows == 0 || seq == 0 || nb == 0) return;
    if (seq <= 16) {
        if (gelu)
            launch_few_tokens<kQ4K, 1, 2, true>(wg, wu, act, mid, rows, nb, seq, stream);
        else
            launch_few_tokens<kQ4K, 1, 2, false>(wg, wu, act, mid, rows, nb, seq, stream);
    } else {
        if (gelu)
            launch_few_tokens<kQ4K, 2, 2, true>(wg, wu, act, mid, rows, nb, seq, stream);
        else
            launch_few_tokens<kQ4K, 2, 2, false>(wg, wu, act, mid, rows, nb, seq, stream);
    }
}

}  // namespace rnb
