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
#include "device_utils.h"
#include "kernels.h"
#include <algorithm>

namespace rnb {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ u16x2 as_u16(uint32_t v) { return __builtin_bit_cast(u16x2, v); }
__device__ __forceinline__ uint32_t as_u32(u16x2 v) { return __builtin_bit_cast(uint32_t, v); }

// One format's share of a 16-row tile and super-block: lane (row lane % 16, quarter kq = lane / 16) owns 64 elements of its
// row, four matrix instructions of K = 64 cover them.  What sits in a lane's K slots is the format's own choice (act_piece:
// the 16-element piece of instruction 0, instruction i takes piece ^ xor_i), the tokens' operands follow it.
//   kBytes, kPieces, kPer   bytes of a block; 16-byte pieces a block is fetched as; rows to one LDS-direct load of 64 pieces
//   fetch, prepare          the packed bytes from the wave's strip; the scales
//   operand(i)              instruction i's weight operands, one per chain of products
//   total                   the chains' sums of one result put together
template <uint32_t kFmt>
struct FewRows;

template <>
struct FewRows<kQ4K> {
    static constexpr int kBytes = kQ4KBytes, kPieces = 9, kInv = 7282, kPer = 7, kChains = 2;
    static constexpr bool kMins = true;
    uint4 hdr, q[2];
    float d, dmin;
    long mnop;
    u16x2 slo[2], shi[2];
    __device__ __forceinline__ static uint32_t act_piece(int kq) { return 4 * kq; }
    __device__ __forceinline__ static constexpr int act_xor(int i) { return i; }
    __device__ __forceinline__ static uint32_t block_off(uint32_t b) { return b * kBytes; }
    __device__ __forceinline__ static uint32_t piece(uint32_t row_off, uint32_t j, uint32_t) { return row_off + 16 * j; }
    __device__ __forceinline__ void fetch(const uint8_t *row, int kq, uint32_t) {
        hdr = *reinterpret_cast<const uint4 *>(row);
        q[0] = *reinterpret_cast<const uint4 *>(row + 16 + 32 * kq);
        q[1] = *reinterpret_cast<const uint4 *>(row + 32 + 32 * kq);
    }
    __device__ __forceinline__ void prepare(int kq) {
        d = f16_bits_to_f32(hdr.x);
        dmin = f16_bits_to_f32(hdr.x >> 16);
        const Q4KScales s = unpack_q4k_scales(hdr.y, hdr.z, hdr.w);
        mnop = kq == 0 ? static_cast<long>(static_cast<unsigned long>(s.mn_lo) | (static_cast<unsigned long>(s.mn_hi) << 32)) : 0L;
        const uint32_t pair = (kq & 2 ? s.sc_hi : s.sc_lo) >> (16 * (kq & 1));  // scales of sub-blocks 2 kq, 2 kq + 1
        const uint32_t lo = pair & 0x0707u, hi = (pair >> 3) & 0x0707u;
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const uint32_t sel = 0x0c000c00u | (g << 16) | g;
            slo[g] = as_u16(__builtin_amdgcn_perm(0u, lo, sel));
            shi[g] = as_u16(__builtin_amdgcn_perm(0u, hi, sel));
        }
    }
    __device__ __forceinline__ void operand(int i, v4i (&op)[kChains]) const {
        const uint32_t v[4] = {q[i & 1].x, q[i & 1].y, q[i & 1].z, q[i & 1].w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const u16x2 nib = as_u16((i < 2 ? v[k] : v[k] >> 4) & 0x0f0f0f0fu);  // products stay inside their bytes
            op[0][k] = static_cast<int>(as_u32(nib * slo[i >> 1]));
            op[1][k] = static_cast<int>(as_u32(nib * shi[i >> 1]));
        }
    }
    __device__ __forceinline__ static int total(const v4i (&c)[kChains], int r) { return c[0][r] + 8 * c[1][r]; }
};

// Q5_K: the fifth bits as a chain of their own, scale times bit
template <>
struct FewRows<kQ5K> {
    static constexpr int kBytes = kQ5KBytes, kPieces = 11, kInv = 5958, kPer = 5, kChains = 3;
    static constexpr bool kMins = true;
    uint4 hdr, q[2], f[2];
    float d, dmin;
    long mnop;
    u16x2 slo[2], shi[2], s16[2];
    __device__ __forceinline__ static uint32_t act_piece(int kq) { return 4 * kq; }
    __device__ __forceinline__ static constexpr int act_xor(int i) { return i; }
    __device__ __forceinline__ static uint32_t block_off(uint32_t b) { return b * kBytes; }
    __device__ __forceinline__ static uint32_t piece(uint32_t row_off, uint32_t j, uint32_t) { return row_off + 16 * j; }
    __device__ __forceinline__ void fetch(const uint8_t *row, int kq, uint32_t) {
        hdr = *reinterpret_cast<const uint4 *>(row);
        f[0] = *reinterpret_cast<const uint4 *>(row + 16);
        f[1] = *reinterpret_cast<const uint4 *>(row + 32);
        q[0] = *reinterpret_cast<const uint4 *>(row + 48 + 32 * kq);
        q[1] = *reinterpret_cast<const uint4 *>(row + 64 + 32 * kq);
    }
    __device__ __forceinline__ void prepare(int kq) {
        d = f16_bits_to_f32(hdr.x);
        dmin = f16_bits_to_f32(hdr.x >> 16);
        const Q4KScales s = unpack_q4k_scales(hdr.y, hdr.z, hdr.w);
        mnop = kq == 0 ? static_cast<long>(static_cast<unsigned long>(s.mn_lo) | (static_cast<unsigned long>(s.mn_hi) << 32)) : 0L;
        const uint32_t pair = (kq & 2 ? s.sc_hi : s.sc_lo) >> (16 * (kq & 1));
        const uint32_t lo = pair & 0x0707u, hi = (pair >> 3) & 0x0707u;
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const uint32_t sel = 0x0c000c00u | (g << 16) | g;
            slo[g] = as_u16(__builtin_amdgcn_perm(0u, lo, sel));
            shi[g] = as_u16(__builtin_amdgcn_perm(0u, hi, sel));
            s16[g] = as_u16(__builtin_amdgcn_perm(0u, pair, sel));
            // bits 2 kq (low nibbles) and 2 kq + 1 (high ones) of each byte
            f[g] = make_uint4(f[g].x >> (2 * kq), f[g].y >> (2 * kq), f[g].z >> (2 * kq), f[g].w >> (2 * kq));
        }
    }
    __device__ __forceinline__ void operand(int i, v4i (&op)[kChains]) const {
        const uint32_t v[4] = {q[i & 1].x, q[i & 1].y, q[i & 1].z, q[i & 1].w};
        const uint32_t h[4] = {f[i & 1].x, f[i & 1].y, f[i & 1].z, f[i & 1].w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const u16x2 nib = as_u16((i < 2 ? v[k] : v[k] >> 4) & 0x0f0f0f0fu);
            const u16x2 bit = as_u16((i < 2 ? h[k] : h[k] >> 1) & 0x01010101u);
            op[0][k] = static_cast<int>(as_u32(nib * slo[i >> 1]));
            op[1][k] = static_cast<int>(as_u32(nib * shi[i >> 1]));
            op[2][k] = static_cast<int>(as_u32(bit * s16[i >> 1]));
        }
    }
    __device__ __forceinline__ static int total(const v4i (&c)[kChains], int r) { return c[0][r] + 8 * c[1][r] + 16 * c[2][r]; }
};

// Q6_K: scale times (code - 32) as a 16-bit product in two digits base 256.  Blocks are 210 bytes, every other one starts two
// bytes off a 4-byte boundary: pieces are fetched from the boundary below (m = 0 or 2 bytes early) and shifted when read;
// piece 13 holds d, fourteen (m = 2) or twelve bytes in: there it ends two bytes behind the block, which is inside the
// matrix unless its number of blocks is odd (gemm_few_supported).
template <>
struct FewRows<kQ6K> {
    static constexpr int kBytes = kQ6KBytes, kPieces = 14, kInv = 4682, kPer = 4, kChains = 2;
    static constexpr bool kMins = false;
    uint32_t ql[2][4], qh[2][4], sc[2], dh;
    float d, dmin;
    long mnop;
    u16x2 s[4];
    __device__ __forceinline__ static uint32_t act_piece(int kq) { return 8 * (kq >> 1) + 2 * (kq & 1); }
    __device__ __forceinline__ static constexpr int act_xor(int i) { return i < 2 ? i : i + 2; }
    __device__ __forceinline__ static uint32_t block_off(uint32_t b) { return b * kBytes - 2 * (b & 1); }
    // row_off = row * nb * 210: bit 1 is the parity of the row's first block
    __device__ __forceinline__ static uint32_t piece(uint32_t row_off, uint32_t j, uint32_t b) {
        const uint32_t m = (row_off ^ (2 * b)) & 2;
        return row_off + 2 * (b & 1) - m + (j < 13 ? 16 * j : 196);
    }
    __device__ __forceinline__ static void words(const uint8_t *p, uint32_t sh, uint32_t (&out)[4]) {
        const uint4 v = *reinterpret_cast<const uint4 *>(p);
        const uint32_t nx = *reinterpret_cast<const uint32_t *>(p + 16);
        out[0] = __builtin_amdgcn_alignbit(v.y, v.x, sh);
        out[1] = __builtin_amdgcn_alignbit(v.z, v.y, sh);
        out[2] = __builtin_amdgcn_alignbit(v.w, v.z, sh);
        out[3] = __builtin_amdgcn_alignbit(nx, v.w, sh);
    }
    __device__ __forceinline__ void fetch(const uint8_t *row, int kq, uint32_t odd) {
        const int h = kq >> 1, a = kq & 1;
        const uint32_t sh = 16 * odd;
#pragma unroll
        for (int g = 0; g < 2; g++) {
            words(row + 64 * h + 32 * a + 16 * g, sh, ql[g]);
            words(row + 128 + 32 * h + 16 * g, sh, qh[g]);
        }
        const uint32_t at = 192 + 2 * odd + 8 * h + 2 * a;
        sc[0] = *reinterpret_cast<const uint16_t *>(row + at);
        sc[1] = *reinterpret_cast<const uint16_t *>(row + (at + 4 == 208 ? 220 : at + 4));
        dh = *reinterpret_cast<const uint16_t *>(row + 220 + 2 * odd);
    }
    __device__ __forceinline__ void prepare(int kq) {
        d = f16_bits_to_f32(dh);
        dmin = 0.0f;
        mnop = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const unsigned short v = static_cast<unsigned short>(static_cast<short>(static_cast<int8_t>(sc[i >> 1] >> (8 * (i & 1)))));
            s[i] = u16x2{v, v};
        }
#pragma unroll
        for (int g = 0; g < 2; g++)
#pragma unroll
            for (int k = 0; k < 4; k++) qh[g][k] >>= 2 * (kq & 1);
    }
    __device__ __forceinline__ void operand(int i, v4i (&op)[kChains]) const {
        const u16x2 m = s[i], off = m * u16x2{static_cast<unsigned short>(-32), static_cast<unsigned short>(-32)} + u16x2{128, 128};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t nib = (i < 2 ? ql[i & 1][k] : ql[i & 1][k] >> 4) & 0x0f0f0f0fu;
            const uint32_t two = (i < 2 ? qh[i & 1][k] << 4 : qh[i & 1][k]) & 0x30303030u;
            const uint32_t codes = nib | two;
            const uint32_t pe = as_u32(as_u16(codes & 0x00ff00ffu) * m + off);  // code * sc - 32 sc + 128
            const uint32_t po = as_u32(as_u16((codes >> 8) & 0x00ff00ffu) * m + off);
            op[0][k] = static_cast<int>(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
            op[1][k] = static_cast<int>(__builtin_amdgcn_perm(po, pe, 0x07030501u));
        }
    }
    __device__ __forceinline__ static int total(const v4i (&c)[kChains], int r) {
        return c[0][r] + static_cast<int>(static_cast<uint32_t>(c[1][r]) << 8);
    }
};

// A wave's share of LDS: the strips of its rows (one per matrix), its tokens' activations, sums and scales of one block
constexpr uint32_t kFewMaxBlocks = 64;  // of a row: the tokens' scales of all of them lie in LDS

template <uint32_t kFmt, int kMT, int kN, int kMats>
struct FewLds {
    typedef FewRows<kFmt> R;
    static constexpr int kFills = (16 * kN + R::kPer - 1) / R::kPer;
    static constexpr int kStrip = kFills * 1024;
    static constexpr int kAct = kMats * kStrip;
    static constexpr int kDig = kAct + kMT * 4096;
    static constexpr int kStage = kDig + (R::kMins ? kMT * 256 : 0);
    static_assert(kMats * kN * kMT * 1024 <= kStage, "the partial sums take the stage's place");
};

template <uint32_t kFmt, int kMT, int kN, int kWaves, int kMats, bool kGelu>
__global__ void __launch_bounds__(kWave *kWaves)
    gemm_few_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ w2, const int8_t *__restrict__ aq,
                    const float *__restrict__ ad, const uint8_t *__restrict__ adig, float *__restrict__ out, uint32_t rows,
                    uint32_t nb, uint32_t seq, uint32_t slices) {
    typedef FewLds<kFmt, kMT, kN, kMats> L;
    typedef FewRows<kFmt> R;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, kq = lane >> 4;
    const uint32_t group = __builtin_amdgcn_readfirstlane(wave / slices), sl = wave - group * slices;  // divided on the vector units
    const uint32_t row0 = __builtin_amdgcn_readfirstlane((blockIdx.x * (kWaves / slices) + group) * (16 * kN));
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
        for (int g = 0; g < 4 * kMT; g++) lds_fill16(act, act_off[g], stage0 + L::kAct + g * 1024);
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
        R rw[kMats][kN];
        v4i a[kMT][4];
        long dig[kMT][2];
        float4 dx[kMT];
#pragma unroll
        for (int m = 0; m < kMats; m++)
#pragma unroll
            for (int n = 0; n < kN; n++) {
                const uint32_t r = 16 * n + l16, odd = (min(r, last_row) * nb + b) & 1;
                rw[m][n].fetch(stage + m * L::kStrip + r / R::kPer * 1024 + r % R::kPer * (16 * R::kPieces), kq, odd);
            }
#pragma unroll
        for (int t = 0; t < kMT; t++) {
            const uint8_t *tok = stage + L::kAct + (16 * t + l16) * 256;
            const uint32_t place = R::act_piece(kq) ^ l16;
#pragma unroll
            for (int i = 0; i < 4; i++) a[t][i] = *reinterpret_cast<const v4i *>(tok + 16 * (place ^ R::act_xor(i)));
            if constexpr (R::kMins) {
                const uint8_t *dg = stage + L::kDig + (16 * t + l16) * 16;
                dig[t][0] = *reinterpret_cast<const long *>(dg);
                dig[t][1] = *reinterpret_cast<const long *>(dg + 8);
            }
            dx[t] = *reinterpret_cast<const float4 *>(scales + b * (16 * kMT) + 16 * t + 4 * kq);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage has been read
        if (b + slices < nb) issue(b + slices);
#pragma unroll
        for (int m = 0; m < kMats; m++)
#pragma unroll
            for (int n = 0; n < kN; n++) {
                R &x = rw[m][n];
                x.prepare(kq);
                v4i c[kMT][R::kChains];
#pragma unroll
                for (int t = 0; t < kMT; t++)
#pragma unroll
                    for (int h = 0; h < R::kChains; h++) c[t][h] = v4i{0, 0, 0, 0};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    v4i op[R::kChains];
                    x.operand(i, op);
#pragma unroll
                    for (int t = 0; t < kMT; t++)
#pragma unroll
                        for (int h = 0; h < R::kChains; h++)
                            c[t][h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[t][i], op[h], c[t][h], 0, 0, 0);
                }
#pragma unroll
                for (int t = 0; t < kMT; t++) {
                    const float dxr[4] = {dx[t].x, dx[t].y, dx[t].z, dx[t].w};
                    v4i s0 = {0, 0, 0, 0}, s1 = {0, 0, 0, 0};
                    if constexpr (R::kMins) {
                        s0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(dig[t][0], x.mnop, s0, 0, 0, 0);
                        s1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(dig[t][1], x.mnop, s1, 0, 0, 0);
                    }
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        float v = x.d * static_cast<float>(R::total(c[t], r));
                        if constexpr (R::kMins) v = __builtin_fmaf(-x.dmin, static_cast<float>(s0[r] + 64 * s1[r]), v);
                        acc[m][n][t][r] = __builtin_fmaf(dxr[r], v, acc[m][n][t][r]);
                    }
                }
            }
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
                uint32_t slices, hipStream_t stream) {
    static bool configured = false;
    constexpr size_t most = kWaves * FewLds<kFmt, kMT, kN, kMats>::kStage + kFewMaxBlocks * 16 * kMT * sizeof(float);
    static_assert(most <= 160 * 1024, "LDS of a compute unit");
    const size_t lds = kWaves * FewLds<kFmt, kMT, kN, kMats>::kStage + static_cast<size_t>(nb) * 16 * kMT * sizeof(float);
    if (!allow_dynamic_lds(reinterpret_cast<const void *>(gemm_few_kernel<kFmt, kMT, kN, kWaves, kMats, kGelu>), most, &configured,
                           "gemm_few_kernel"))
        return;
    const uint32_t per_wg = kWaves / slices * 16 * kN;
    hipLaunchKernelGGL((gemm_few_kernel<kFmt, kMT, kN, kWaves, kMats, kGelu>), dim3((rows + per_wg - 1) / per_wg), dim3(kWave * kWaves),
                       lds, stream, w, w2, act.qs, act.d, act.digits, out, rows, nb, seq, slices);
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

// Where it is ahead of the GEMV passes over up to four tokens (us, GEMV : this kernel): rows of more than 16 blocks from three
// tokens on (4096 x 14336 Q4_K 13.2 : 10.9, Q6_K 18.0 : 16.1); shorter ones, whose bits at two to four tokens do not depend on how
// many rows the matrix has, from four (14336 x 4096 Q4_K 13.5 : 11.6, three 11.2 : 11.5), Q6_K five (14336 x 4096 22.6 : 16.4, four 17.6
// : 16.6).
// Matrices of less than 4 MB keep the GEMV up to eight tokens (Q6_K 1024 x 4096 7.4 : 8.0 at eight, Q4_K 7.5 : 6.8) and its bits.
// Ahead of gemm_blocks.hip everywhere up to 16 tokens, and with Q6_K; 17 to 32 tokens of Q4_K and Q5_K read twice the
// activations per row, which costs more than the slices in memory where a wave has many blocks (24 tokens, Q4_K, gemm_blocks :
// this: 1024 x 14336 12.3 : 14.3, 1024 x 8192 9.9 : 10.6; 2048 x 8192 11.6 : 10.9) or the matrix is large (65536 x 4096 47 : 50, Q5_K
// 28672 x 8192 55 : 57, 28672 x 1024 11.8 : 13.6; 28672 x 4096 Q4_K 30.1 : 28.4, Q5_K 34.0 : 33.4).
bool gemm_few_pays(uint32_t quant, size_t rows, size_t nb, size_t seq) {
    if (seq < 3 || seq > 32) return false;
    const size_t bytes = rows * nb * (quant == kQ4K ? kQ4KBytes : quant == kQ5K ? kQ5KBytes : kQ6KBytes);
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
