// The GEMM of gemm_digits.h for Q4_K, Q5_K and Q6_K.
#include "gemm_digits.h"

namespace rnb {

namespace {

template <>
struct Rows<kQ4K> {
    static constexpr int kBytes = kQ4KBytes, kPieces = 9, kInv = 7282, kRows = 7, kShift = 3;
    static constexpr bool kMins = true, kDirect = false;
    static constexpr int kTableBytes = 0;
    uint4 raw;
    uint32_t dlo[2], dhi[2];
    __device__ __forceinline__ static uint32_t piece(uint32_t r, uint32_t j, uint32_t row_bytes, uint32_t, uint32_t) {
        return r * row_bytes + 16 * j;
    }
    __device__ __forceinline__ static uint32_t block_off(uint32_t b) { return b * kBytes; }
    __device__ __forceinline__ void head(const uint8_t *row, int, uint32_t) {
        const uint4 hdr = *reinterpret_cast<const uint4 *>(row);
        const Q4KScales sc = unpack_q4k_scales(hdr.y, hdr.z, hdr.w);
        dlo[0] = sc.sc_lo & 0x07070707u;
        dlo[1] = sc.sc_hi & 0x07070707u;
        dhi[0] = (sc.sc_lo >> 3) & 0x07070707u;
        dhi[1] = (sc.sc_hi >> 3) & 0x07070707u;
    }
    __device__ __forceinline__ void fetch(int s, const uint8_t *row, int khalf) {
        if ((s & 1) == 0) raw = *reinterpret_cast<const uint4 *>(row + 16 + 16 * s + 16 * khalf);
    }
    __device__ __forceinline__ void operand(int s, int, const void *, v4i &lo, v4i &hi) {
        const uint32_t q[4] = {raw.x, raw.y, raw.z, raw.w};
        const uint32_t sel = 0x0c000c00u | ((s & 3) << 16) | (s & 3);
        const u16x2 sl = as_u16(__builtin_amdgcn_perm(0u, dlo[s >> 2], sel)), sh = as_u16(__builtin_amdgcn_perm(0u, dhi[s >> 2], sel));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const u16x2 nib = as_u16((q[i] >> (4 * (s & 1))) & 0x0f0f0f0fu);  // products stay inside their bytes
            lo[i] = static_cast<int>(as_u32(nib * sl));
            hi[i] = static_cast<int>(as_u32(nib * sh));
        }
    }
};

template <>
struct Rows<kQ5K> {
    static constexpr int kBytes = kQ5KBytes, kPieces = 11, kInv = 5958, kRows = 5, kShift = 8;
    static constexpr bool kMins = true, kDirect = false;
    static constexpr int kTableBytes = 0;
    uint4 qh, raw;
    uint32_t sc[2];
    __device__ __forceinline__ static uint32_t piece(uint32_t r, uint32_t j, uint32_t row_bytes, uint32_t, uint32_t) {
        return r * row_bytes + 16 * j;
    }
    __device__ __forceinline__ static uint32_t block_off(uint32_t b) { return b * kBytes; }
    __device__ __forceinline__ void head(const uint8_t *row, int khalf, uint32_t) {
        const uint4 hdr = *reinterpret_cast<const uint4 *>(row);
        qh = *reinterpret_cast<const uint4 *>(row + 16 + 16 * khalf);
        const Q4KScales s = unpack_q4k_scales(hdr.y, hdr.z, hdr.w);
        sc[0] = s.sc_lo;
        sc[1] = s.sc_hi;
    }
    __device__ __forceinline__ void fetch(int s, const uint8_t *row, int khalf) {
        if ((s & 1) == 0) raw = *reinterpret_cast<const uint4 *>(row + 48 + 16 * s + 16 * khalf);
    }
    __device__ __forceinline__ void operand(int s, int, const void *, v4i &lo, v4i &hi) {
        const uint32_t q[4] = {raw.x, raw.y, raw.z, raw.w}, f[4] = {qh.x, qh.y, qh.z, qh.w};
        const u16x2 m = as_u16(__builtin_amdgcn_perm(0u, sc[s >> 2], 0x0c000c00u | ((s & 3) << 16) | (s & 3)));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t fifth = (s <= 4 ? f[i] << (4 - s) : f[i] >> (s - 4)) & 0x10101010u;
            int l, h;
            digits256(((q[i] >> (4 * (s & 1))) & 0x0f0f0f0fu) | fifth, m, splat(128), l, h);
            lo[i] = l;
            hi[i] = h;
        }
    }
};

// Q6_K blocks are 210 bytes: every other one starts two bytes off a 4-byte boundary.  Pieces are fetched from the
// boundary below (m = 0 or 2 bytes early) and shifted when read; piece 13 is the sixteen bytes up to the block's end for
// m = 2 (its last dword lies at 220 of the strip's row) and unused for m = 0.  d is read by the row's lanes themselves.
template <>
struct Rows<kQ6K> {
    static constexpr int kBytes = kQ6KBytes, kPieces = 14, kInv = 4682, kRows = 4, kShift = 8;
    static constexpr bool kMins = false, kDirect = false;
    static constexpr int kTableBytes = 0, kDOff = 208;
    static constexpr float kD = 1.0f;
    uint32_t sh;             // 8 m of the lane's row
    uint32_t ql[2][4], qh[4];  // of the present half
    u16x2 sc[4];             // the K-half's scales of sub-block pairs 2i (x) and 2i + 1 (y)
    __device__ __forceinline__ static uint32_t piece(uint32_t r, uint32_t j, uint32_t row_bytes, uint32_t b, uint32_t nb) {
        const uint32_t m = 2 * ((b + r * nb) & 1);
        return r * row_bytes + 2 * (b & 1) - m + (j < 13 ? 16 * j : 192 + 2 * m);
    }
    __device__ __forceinline__ static uint32_t block_off(uint32_t b) { return b * kBytes - 2 * (b & 1); }
    __device__ __forceinline__ void words(const uint8_t *p, uint32_t (&out)[4]) const {
        const uint4 v = *reinterpret_cast<const uint4 *>(p);
        const uint32_t nx = *reinterpret_cast<const uint32_t *>(p + 16);
        out[0] = __builtin_amdgcn_alignbit(v.y, v.x, sh);
        out[1] = __builtin_amdgcn_alignbit(v.z, v.y, sh);
        out[2] = __builtin_amdgcn_alignbit(v.w, v.z, sh);
        out[3] = __builtin_amdgcn_alignbit(nx, v.w, sh);
    }
    __device__ __forceinline__ void head(const uint8_t *row, int khalf, uint32_t odd) {
        sh = 16 * odd;
        const uint4 v = *reinterpret_cast<const uint4 *>(row + 192);
        const uint32_t nx = *reinterpret_cast<const uint32_t *>(row + 220);
        const uint32_t w[5] = {v.x, v.y, v.z, v.w, nx};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t t = __builtin_amdgcn_alignbit(w[i + 1], w[i], sh) << (khalf ? 0 : 8);  // the K-half's scales in bytes 1, 3
            typedef short s16x2 __attribute__((ext_vector_type(2)));
            sc[i] = __builtin_bit_cast(u16x2, static_cast<s16x2>(__builtin_bit_cast(s16x2, t) >> 8));
        }
    }
    __device__ __forceinline__ void fetch(int s, const uint8_t *row, int khalf) {
        const int h = s >> 2, p = s & 3;
        if (p < 2) words(row + 64 * h + 32 * p + 16 * khalf, ql[p]);
        if (p == 0) words(row + 128 + 32 * h + 16 * khalf, qh);
    }
    __device__ __forceinline__ void operand(int s, int, const void *, v4i &lo, v4i &hi) {
        const int p = s & 3;
        const unsigned short c = (s & 1) ? sc[s >> 1].y : sc[s >> 1].x;
        const u16x2 m = splat(c), off = m * splat(static_cast<unsigned short>(-32)) + splat(128);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t nib = (ql[p & 1][i] >> (4 * (p >> 1))) & 0x0f0f0f0fu;
            const uint32_t two = (p < 2 ? qh[i] << (4 - 2 * p) : qh[i] >> (2 * p - 4)) & 0x30303030u;
            int l, hh;
            digits256(nib | two, m, off, l, hh);
            lo[i] = l;
            hi[i] = hh;
        }
    }
};

}  // namespace

// Where it is ahead of the kernels that make operands per 32 or 64 tokens (gemm_q4k.hip, gemm_blocks.hip), measured over
// rows 1024 - 28672, columns 1024 - 16384, 33 - 2048 tokens, us per step: a workgroup starts slowly (LDS of 110 - 137 KB, a
// block's operands before the first product), so it needs work.  Q6_K from 2.2e9 multiply-adds (14336 x 4096 x 40 tokens
// 36 -> 31, 4096 x 4096 x 192 40 -> 33; below: 4096 x 4096 x 128 27 against 32), Q5_K from 5e9 (14336 x 4096 x 96 41 ->
// 37; 4096 x 4096 x 256 32 against 37), Q4_K, whose ping-pong kernel already folds the scales, from 18e9 (14336 x 4096 x 333
// 79 -> 72, 26742 x 11264 x 117 111 -> 108; 14336 x 4096 x 256 47 against 55).  The last two lose where the last round of
// workgroups is nearly empty (Q4_K 9289 x 6400 x 779, 259 workgroups: 143 against 152), see digits_fill_the_chip.  Q4_K
// gains nothing either where a workgroup is dealt two token tiles, the 64 tokens its ping-pong kernel makes operands for
// (20284 x 7936 x 134 80.3 us against 82.7, 17567 x 11776 x 157 109 against 115); Q5_K does (20430 x 4352 x 191 74 -> 63),
// but not on rows of fewer than 16 blocks: there the start of a workgroup wants four tiles behind it (10000 x 1280 x 1500
// 85 -> 67) or one round of whole rows (threes of 8192 x 2048 x 700 53 -> 46), else it is behind (15360 x 1024 x 639 dealt in
// threes 43.6 against 47.7, 13959 x 3328 x 513 in twos 97 against 101, 10850 x 3072 x 287 in one round of twos 46.6 against
// 48.2, 4255 x 3328 x 658 in two slices 45 against 50).
bool gemm_digits_pays(uint32_t quant, const uint8_t *w, size_t rows, size_t cols, size_t seq) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(w);
    const double macs = static_cast<double>(rows) * static_cast<double>(cols) * static_cast<double>(seq);
    if (seq <= 32) return false;
    if (quant == kQ6K) return a % 4 == 0 && macs >= 2.2e9;
    if (quant != kQ4K && quant != kQ5K) return false;
    if (a % 16 != 0 || macs < (quant == kQ4K ? 18e9 : 5e9)) return false;
    const uint32_t r = static_cast<uint32_t>(rows), nb = static_cast<uint32_t>(cols / 256), q = static_cast<uint32_t>(seq);
    const DgPlan p = digits_plan(r, nb, q);
    const bool one_round = p.slices == 1 && static_cast<uint64_t>(p.row_tiles) * p.groups <= 256;
    const uint32_t min_tiles = quant == kQ4K ? 3 : nb >= 16 ? 2 : one_round ? 3 : 4;
    return p.tiles_per_wg >= min_tiles && digits_fill_the_chip(r, nb, q);
}

bool gemm_digits_pair_pays(size_t rows, size_t nb, size_t seq) {
    const uint32_t r = static_cast<uint32_t>(rows), b = static_cast<uint32_t>(nb), q = static_cast<uint32_t>(seq);
    const DgPlan one = digits_plan(r, b, q);
    return one.slices > 1 || digits_plan(2 * r, b, q).cost < 2 * one.cost;
}

size_t gemm_digits_slice_floats(uint32_t rows, uint32_t nb, uint32_t seq) {
    if (rows == 0 || nb == 0 || seq == 0) return 0;
    const DgPlan p = digits_plan(rows, nb, seq);
    return p.slices > 1 ? static_cast<size_t>(p.slices) * seq * rows : 0;
}

void launch_gemm_digits(const uint8_t *w, uint32_t quant, ActView act, float *out, float *slice_out, uint32_t rows, uint32_t nb,
                        uint32_t seq, hipStream_t stream, const uint8_t *w2, uint32_t *left) {
    if (rows == 0 || seq == 0 || nb == 0) return;
    if (quant == kQ4K && w2 != nullptr)
        launch_digits_plan<kQ4K, true>(w, act, out, slice_out, rows, nb, seq, stream, w2, left);
    else if (quant == kQ4K)
        launch_digits_plan<kQ4K>(w, act, out, slice_out, rows, nb, seq, stream);
    else if (quant == kQ5K)
        launch_digits_plan<kQ5K>(w, act, out, slice_out, rows, nb, seq, stream);
    else
        launch_digits_plan<kQ6K>(w, act, out, slice_out, rows, nb, seq, stream);
}

}  // namespace rnb
