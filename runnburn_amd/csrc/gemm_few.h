// Pieces of the few-token GEMMs (gemm_few.hip: one matrix; moe_few.hip: routed experts): how a wave's share of a block lies in its
// stage of LDS, is read into registers and multiplied.
#pragma once

#include "device_utils.h"
#include "kernels.h"
#include <algorithm>
#include <type_traits>

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

// A block's operands in registers: the stage they came from is free again
template <uint32_t kFmt, int kMT, int kN, int kMats>
struct FewBlock {
    typedef FewRows<kFmt> R;
    static constexpr int kStrip = FewLds<kFmt, kMT, kN, kMats>::kStrip;
    R rw[kMats][kN];
    v4i a[kMT][4];
    long dig[kMT][2];
    float4 dx[kMT];

    // act_at, dig_at: where activations and digits lie in the stage; scales: the tokens' of block b
    __device__ __forceinline__ void read(const uint8_t *stage, int act_at, int dig_at, const float *scales, int l16, int kq, uint32_t last_row, uint32_t nb, uint32_t b) {
#pragma unroll
        for (int m = 0; m < kMats; m++)
#pragma unroll
            for (int n = 0; n < kN; n++) {
                const uint32_t r = 16 * n + l16, odd = (min(r, last_row) * nb + b) & 1;
                rw[m][n].fetch(stage + m * kStrip + r / R::kPer * 1024 + r % R::kPer * (16 * R::kPieces), kq, odd);
            }
#pragma unroll
        for (int t = 0; t < kMT; t++) {
            const uint8_t *tok = stage + act_at + (16 * t + l16) * 256;
            const uint32_t place = R::act_piece(kq) ^ l16;
#pragma unroll
            for (int i = 0; i < 4; i++) a[t][i] = *reinterpret_cast<const v4i *>(tok + 16 * (place ^ R::act_xor(i)));
            if constexpr (R::kMins) {
                const uint8_t *dg = stage + dig_at + (16 * t + l16) * 16;
                dig[t][0] = *reinterpret_cast<const long *>(dg);
                dig[t][1] = *reinterpret_cast<const long *>(dg + 8);
            }
            dx[t] = *reinterpret_cast<const float4 *>(scales + 16 * t + 4 * kq);
        }
    }
    // acc += the block's products; kExact: in the roundings of the kernels that have no fused multiply-add
    template <bool kExact>
    __device__ __forceinline__ void multiply(float (&acc)[kMats][kN][kMT][4], int kq) {
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
                        const float mins = static_cast<float>(s0[r] + 64 * s1[r]);
                        if constexpr (R::kMins) v = kExact ? v - x.dmin * mins : __builtin_fmaf(-x.dmin, mins, v);
                        acc[m][n][t][r] = kExact ? acc[m][n][t][r] + dxr[r] * v : __builtin_fmaf(dxr[r], v, acc[m][n][t][r]);
                    }
                }
            }
    }
};

}  // namespace

}  // namespace rnb
