// Prefill GEMM of the formats with an integer sub-block scale (here Q4_K, Q5_K and Q6_K; gemv_iq.hip brings the importance
// quants) for batches of more than 32 tokens: out[seq][rows], same contract as the GEMVs.  Scale times code goes onto the int8 matrix cores as two digits, the float
// scales onto the results once per super-block:
//   I = sum_sb sc * sum_k code * a  =  I_lo + 2^kShift * I_hi        (exact int32, two v_mfma_i32_32x32x32_i8 chains)
//     Q4_K  sc = lo + 8 hi, digits lo * nibble and hi * nibble (<= 105)
//     Q5_K  sc * code <= 1953 and Q6_K sc * (code - 32), |.| <= 4096: made as 16-bit products, digits base 256
//   S = sum_sb mn * bsum32 (Q4_K, Q5_K): one v_mfma_f32_32x32x16_f16 over the quantiser's digits b0 + 64 b1 (exact: every
//     operand has at most 7 significant bits, sums stay below 2^24)
//   out += d_x * (d * I - dmin * S)
// (crates/rnb-cpu/src/gemm/neon_dot.rs:884-916, :1742-1800, :2240-2288)
//
// What bounds it is the vector port: a SIMD issues one vector instruction in 4 cycles, a matrix instruction occupies
// its pipe for 32, and a tile of 32 x 32 results takes 16 (17) of these per super-block beside 4 (5) vector
// instructions a result and the making of the operands.  Hence
//   * operands are made once for kT * 32 (up to 128) tokens: a wave owns 32 rows, holds both digits of a whole
//     super-block in registers (64) and walks the token tiles with them, one tile's sums at a time;
//   * the float update of a tile is dealt out between the matrix instructions of the next one, the next super-block's
//     operands replace the present ones behind their last use, so each wave feeds both the pipe and the port all the
//     time and the workgroup meets at one barrier per super-block.
// Measured per step (quantiser and slice sums included), before, with operands made per 64 tokens and the scales of Q5_K and
// Q6_K put on every result of a sub-block -> after: Q4_K 14336 x 4096 x 512 80 -> 71 us (0.84 PFLOP/s), Q5_K 14336 x 4096 x
// 1024 205 -> 176, Q6_K 4096 x 14336 x 2048 516 -> 322, 4096 x 14336 x 300 176 -> 89.  Counters at 14336 x 4096 x 2048 Q4_K:
// 2.0 GHz, matrix pipe 48 % and vector port 49 % of a busy unit's time; without the fills it would be 10 % faster, without
// the float update 11 %, without making operands 6 %.  Tried without gain: wave priorities, the waves of a SIMD making
// their operands in different tiles.
// A workgroup is eight waves = 256 rows; the tokens' activations and the waves' packed rows come into
// LDS by LDS-direct loads, the packed rows into a strip of the wave's own (no barrier), requested as soon as the strip
// has been read.  MFMA "M" is the token and "N" the weight row: a lane's 16 results belong to row lane % 32.
#pragma once

#include "device_utils.h"
#include "kernels.h"
#include <algorithm>

namespace rnb {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr int kDgWaves = 8;
constexpr int kDgThreads = kWave * kDgWaves;
constexpr int kDgRows = 32 * kDgWaves;
// Four tokens' activations of a block (one LDS-direct load) are 1024 bytes, 64 more to the next four; token 4g + i keeps
// its 16-byte column c at place c ^ i, so that sixteen consecutive tokens' reads fall on different banks.
constexpr int kDgActGroup = 1088;

__device__ __forceinline__ u16x2 as_u16(uint32_t v) { return __builtin_bit_cast(u16x2, v); }
__device__ __forceinline__ uint32_t as_u32(u16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ u16x2 splat(unsigned short v) { return u16x2{v, v}; }

// four codes (bytes) -> code * sc + off in 16 bits each, as a digit base 256 between -128 and 127 and the rest above
// it; `off` carries 128 so that the low byte is the digit + 128
__device__ __forceinline__ void digits256(uint32_t codes, u16x2 sc, u16x2 off, int &lo, int &hi) {
    const uint32_t pe = as_u32(as_u16(codes & 0x00ff00ffu) * sc + off);
    const uint32_t po = as_u32(as_u16((codes >> 8) & 0x00ff00ffu) * sc + off);
    lo = static_cast<int>(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
    hi = static_cast<int>(__builtin_amdgcn_perm(po, pe, 0x07030501u));
}

// How a format's packed rows come into a wave's strip and leave it as operands.  kPieces 16-byte pieces per row and
// block, kRows rows to a load (kInv = 65536 / kPieces, rounded up, divides a lane's number); a lane's share of sub-block pair s (32 elements) is the 16 elements of its K-half.
//   kBytes, kShift, kMins   bytes of a block, power of the high digit, whether there are mins
//   fetch(s), operand(s)    read a pair's packed bytes, make its two operands
//   without mins: kDOff, kD  where the block's f16 d lies, and its factor
// kDirect formats have no strip: load() takes the lane's own bytes into registers a block ahead.
template <uint32_t kFmt>
struct Rows;

// eight bytes -> f16: 0x64 above a byte is the f16 number 1024 + byte
__device__ __forceinline__ v8h bytes_f16(uint32_t lo, uint32_t hi, _Float16 minus) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    v8h o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t pair = __builtin_amdgcn_perm(0x64646464u, i < 2 ? lo : hi, (i & 1) ? 0x04030402u : 0x04010400u);
        const h2 v = __builtin_bit_cast(h2, pair) - h2{minus, minus};
        o[2 * i] = v.x;
        o[2 * i + 1] = v.y;
    }
    return o;
}

template <uint32_t kFmt, int kT>
struct DgLds {
    static constexpr int kToks = 32 * kT;
    static constexpr int kFills = Rows<kFmt>::kDirect ? 0 : (32 + Rows<kFmt>::kRows - 1) / Rows<kFmt>::kRows;  // per wave and block
    static constexpr int kStrip = kFills * 1024;
    static constexpr int kABuf = kToks / 4 * kDgActGroup;
    static constexpr int kA = kDgWaves * kStrip;
    static constexpr int kDx = kA + 2 * kABuf;        // ring of four: 128 activation scales each
    static constexpr int kDig = kDx + 4 * 512;        // two: 32 bytes of f16 digits per token
    static constexpr int kTable = kDig + (Rows<kFmt>::kMins ? 2 * kToks * 32 : 0);
    static constexpr int kBytes = kTable + Rows<kFmt>::kTableBytes;
    static_assert(kBytes <= 160 * 1024, "LDS of a compute unit");
};

template <uint32_t kFmt, int kT, bool kPair>
__global__ void __launch_bounds__(kDgThreads, 2)
    gemm_digits_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ w2, const int8_t *__restrict__ aq,
                       const float *__restrict__ ad, const uint8_t *__restrict__ adig, float *__restrict__ out, uint32_t rows,
                       uint32_t nb, uint32_t seq, uint32_t nb_slice) {
    typedef DgLds<kFmt, kT> L;
    typedef Rows<kFmt> R;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: what derives from it stays in SGPRs
    const int lrow = lane & 31, khalf = lane >> 5;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lptr_t)lds));
    const uint32_t row_tile = gemm_matrix<kPair>(w, w2, out, rows, seq, kDgRows);
    const uint32_t row0 = row_tile * kDgRows + wave * 32;
    // clamped loads, masked stores; a multiple of 32, so that Q6_K rows sit as far off a 4-byte boundary as their index says
    const uint32_t first = min(row0, (rows - 1) & ~31u), last_row = min(rows - 1 - first, 31u);
    const uint32_t tok0 = blockIdx.y * L::kToks, last_tok = seq - 1 - tok0;
    const uint32_t row_bytes = nb * static_cast<uint32_t>(R::kBytes);

    // K slice of this workgroup (blockIdx.z): blocks slice0 .. slice0 + nbs, its sums go to the slice's own copy of the output
    const uint32_t slice0 = blockIdx.z * nb_slice, nbs = min(nb - slice0, nb_slice);
    const uint8_t *w_base = w + static_cast<size_t>(first) * row_bytes;
    const uint8_t *a_base = reinterpret_cast<const uint8_t *>(aq) + (static_cast<size_t>(tok0) * nb + slice0) * 256;
    const uint8_t *dig_base = adig + (static_cast<size_t>(tok0) * nb + slice0) * 16;
    const uint8_t *dx_base = reinterpret_cast<const uint8_t *>(ad) + (static_cast<size_t>(tok0) * nb + slice0) * 4;
    const uint8_t *strip_row = nullptr;
    if constexpr (!R::kDirect) strip_row = lds + wave * L::kStrip + lrow / R::kRows * 1024 + lrow % R::kRows * 16 * R::kPieces;
    const uint32_t my_row = min(static_cast<uint32_t>(lrow), last_row);

    // the lanes' offsets are made anew for each request: kept for the whole loop they would cost registers it has not got
    auto fresh = [&](uint32_t v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    auto issue_w = [&](uint32_t b) {  // b counted from the start of the row
        if constexpr (!R::kDirect) {
            const uint8_t *src = w_base + static_cast<int64_t>(R::block_off(b));
            const uint32_t l = fresh(lane);
            const uint32_t rr = __umul24(l, R::kInv) >> 16, j = l - rr * R::kPieces;
            const uint32_t off = R::piece(rr, j, row_bytes, b, nb);
            constexpr int kEnd = 31 - (L::kFills - 1) * R::kRows;  // the last load's rows end here
#pragma unroll
            for (int k = 0; k < L::kFills; k++) {
                const uint32_t dst = lds0 + wave * L::kStrip + k * 1024;
                if (last_row == 31) {  // the loads but the last differ in a scalar only
                    const uint8_t *at = src + static_cast<size_t>(k * R::kRows) * row_bytes;
                    lds_fill16(at, k + 1 < L::kFills ? off : R::piece(min(rr, static_cast<uint32_t>(kEnd)), j, row_bytes, b, nb), dst);
                } else {
                    lds_fill16(src, R::piece(min(k * R::kRows + rr, last_row), j, row_bytes, b, nb), dst);
                }
            }
        }
    };
    auto issue_a = [&](uint32_t b) {  // b counted from the slice's start, as below
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
        if (wave < (kT > 2 ? 2 : 1))
            lds_fill4(dx_base + b * 4u, min(wave * 64 + l, last_tok) * (nb * 4u), lds0 + L::kDx + (b & 3) * 512 + wave * 256);
    };
    // digits of token tid / 2: b0 (even threads), 64 * b1 (odd threads)
    const bool dig_thread = tid < 2 * L::kToks;
    auto load_dig = [&](uint32_t b) {
        uint2 v = make_uint2(0, 0);
        const uint32_t t = fresh(tid);
        if (R::kMins && dig_thread)
            v = *reinterpret_cast<const uint2 *>(dig_base + b * 16u + min(t >> 1, last_tok) * (nb * 16u) + (t & 1) * 8u);
        return v;
    };
    auto store_dig = [&](uint32_t b, uint2 v) {
        const uint32_t t = fresh(tid);
        if (R::kMins && dig_thread)
            *reinterpret_cast<v8h *>(lds + L::kDig + (b & 1) * (L::kToks * 32) + t * 16) =
                bytes_f16(v.x ^ 0x80808080u, v.y ^ 0x80808080u, static_cast<_Float16>(1152.0f)) * static_cast<_Float16>(t & 1 ? 64.0f : 1.0f);
    };
    const uint8_t *w_row = w_base + static_cast<size_t>(my_row) * row_bytes;
    auto load_d = [&](uint32_t b) {  // formats without mins: the row's own d
        if constexpr (R::kMins) return 0.0f;
        else return ld_f16(w_row + static_cast<size_t>(b) * R::kBytes + R::kDOff) * R::kD;
    };

    float accf[kT][16];
#pragma unroll
    for (int t = 0; t < kT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) accf[t][r] = 0.0f;
    const v16i zero16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const v16f zerof = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    v4i wlo[8], whi[8];  // the present super-block's operands
    v8h mnop = {0, 0, 0, 0, 0, 0, 0, 0};
    float d = 0.0f, ndmin = 0.0f;
    v16i plo = zero16, phi = zero16;  // sums of the previous tile, updated while the present one's are made
    v16f ps = zerof;
    float pd = 0.0f, pndmin = 0.0f;

    R rw;
    auto finish_head = [&](float d6) {
        if constexpr (R::kMins) {
            const uint4 h = *reinterpret_cast<const uint4 *>(strip_row);
            d = f16_bits_to_f32(h.x);
            ndmin = -f16_bits_to_f32(h.x >> 16);
            const Q4KScales sc = unpack_q4k_scales(h.y, h.z, h.w);
            mnop = bytes_f16(sc.mn_lo, sc.mn_hi, static_cast<_Float16>(1024.0f));
        } else {
            d = d6;
        }
    };
    // results 2s, 2s + 1 of tile t of the block whose scales lie in ring slot `slot`
    float4 dx4 = make_float4(0.f, 0.f, 0.f, 0.f);
    auto load_dx = [&](int t, int j, uint32_t slot) {
        dx4 = reinterpret_cast<const float4 *>(lds + L::kDx + slot * 512)[8 * t + 2 * j + khalf];
    };
    // group s of eight: the sums of a tile's last matrix instructions are not there yet in the first group
    auto upd_first = [](int s) { return s == 0 ? 0 : s < 7 ? 2 * s - 2 : 13; };
    auto upd_end = [](int s) { return s == 0 ? 0 : s < 6 ? 2 * s : s == 6 ? 13 : 16; };
    auto update = [&](int t, int s, int half, uint32_t slot) {
        const int mid = (upd_first(s) + upd_end(s)) / 2;
#pragma unroll
        for (int r = half == 0 ? upd_first(s) : mid; r < (half == 0 ? mid : upd_end(s)); r++) {
            const float dx = (r & 3) == 0 ? dx4.x : (r & 3) == 1 ? dx4.y : (r & 3) == 2 ? dx4.z : dx4.w;
            float v = pd * static_cast<float>(plo[r] + static_cast<int>(static_cast<uint32_t>(phi[r]) << R::kShift));
            if constexpr (R::kMins) v = __builtin_fmaf(pndmin, ps[r], v);
            accf[t][r] = __builtin_fmaf(dx, v, accf[t][r]);
            asm volatile("" : "+v"(accf[t][r]));
            if ((r & 3) == 3 && r < 15) load_dx(t, (r + 1) >> 2, slot);
        }
    };

    if constexpr (R::kDirect)
        rw.load(w_row + static_cast<size_t>(slice0) * R::kBytes, khalf);
    else
        issue_w(slice0);
    issue_a(0);
    if constexpr (R::kTableBytes > 0) {
        const uint4 *src = static_cast<const uint4 *>(R::table());
        for (int i = tid; i < R::kTableBytes / 16; i += kDgThreads) reinterpret_cast<uint4 *>(lds + L::kTable)[i] = src[i];
        __syncthreads();
    }
    store_dig(0, load_dig(0));
    if (tid < 128) reinterpret_cast<float *>(lds + L::kDx + 3 * 512)[tid] = 0.0f;  // what the first "previous" tile reads
    const float d_first = load_d(slice0);
    wait_fills();
    if constexpr (!R::kDirect) rw.head(strip_row, khalf, (my_row * nb + slice0) & 1);
#pragma unroll
    for (int s = 0; s < 8; s++) {
        rw.fetch(s, strip_row, khalf);
        rw.operand(s, khalf, lds + L::kTable, wlo[s], whi[s]);
    }
    finish_head(d_first);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (!R::kDirect && nbs > 1) issue_w(slice0 + 1);

    for (uint32_t b = 0; b < nbs; b++) {
        // this wave's pieces of block b have landed (waited for below); behind the barrier everyone's have, and nobody
        // reads block b - 1 any more
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        uint2 dig = make_uint2(0, 0);
        float d_next = 0.0f;
        const uint32_t bn = min(b + 1, nbs - 1);
        if (b + 1 < nbs) issue_a(b + 1);
        dig = load_dig(bn);
        d_next = load_d(slice0 + bn);
        if constexpr (R::kDirect) rw.load(w_row + static_cast<size_t>(slice0 + bn) * R::kBytes, khalf);
        // token lrow of tile t, sub-block s: column 2 s + khalf at place (2 s + khalf) ^ (lrow & 3)
        const uint8_t *abase = lds + L::kA + (b & 1) * L::kABuf + (lrow >> 2) * kDgActGroup + (lrow & 3) * 256 + 16 * (khalf ^ (lrow & 1));
        const uint8_t *apos[2] = {abase + 16 * (lrow & 2), abase - 16 * (lrow & 2)};  // even and odd s
        auto act_operand = [&](int q) {
            return *reinterpret_cast<const v4i *>(apos[q & 1] + 8 * (q >> 3) * kDgActGroup + 32 * (q & 7));
        };
        const uint8_t *digbase = lds + L::kDig + (b & 1) * (L::kToks * 32) + lrow * 32 + 16 * khalf;
        v4i a[3];
        a[0] = act_operand(0);
        a[1] = act_operand(1);
#pragma unroll
        for (int t = 0; t < kT; t++) {
            const int tp = t == 0 ? kT - 1 : t - 1;
            const uint32_t pslot = t == 0 ? (b + 3) & 3 : b & 3;
            v16i clo = zero16, chi = zero16;
            v16f cs = zerof;
            v8h dg;
            if (t == kT - 1) {
                wait_fills();  // the next block's activations and packed rows
                store_dig(b + 1, dig);
                if constexpr (!R::kDirect) rw.head(strip_row, khalf, (my_row * nb + slice0 + b + 1) & 1);
            }
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const int q = t * 8 + s;
                if (q + 2 < 8 * kT) a[(q + 2) % 3] = act_operand(q + 2);
                if (t == kT - 1) rw.fetch(s, strip_row, khalf);
                if constexpr (R::kMins)
                    if (s == 7) dg = *reinterpret_cast<const v8h *>(digbase + 32 * 32 * t);
                clo = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[q % 3], wlo[s], clo, 0, 0, 0);
                asm volatile("" : "+v"(clo));  // pins the instruction inside its group
                update(tp, s, 0, pslot);
                chi = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[q % 3], whi[s], chi, 0, 0, 0);
                asm volatile("" : "+v"(chi));
                update(tp, s, 1, pslot);
                if (s == 7) load_dx(t, 0, b & 3);
                if (t == kT - 1) {
                    rw.operand(s, khalf, lds + L::kTable, wlo[s], whi[s]);
                    asm volatile("" : "+v"(wlo[s]), "+v"(whi[s]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (R::kMins) cs = __builtin_amdgcn_mfma_f32_32x32x16_f16(dg, mnop, cs, 0, 0, 0);
            plo = clo;
            phi = chi;
            ps = cs;
            if (t == 0) {
                pd = d;
                pndmin = ndmin;
            }
        }
        finish_head(d_next);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the strip has been read
        if (!R::kDirect && b + 2 < nbs) issue_w(slice0 + b + 2);
    }
#pragma unroll
    for (int s = 1; s < 8; s++) {
        update(kT - 1, s, 0, (nbs - 1) & 3);
        update(kT - 1, s, 1, (nbs - 1) & 3);
    }

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

struct DgPlan {
    uint32_t tiles_per_wg, groups, row_tiles, slices;
    uint64_t cost;  // rounds * blocks of a slice * half tiles
};
// Token tiles of 32 are dealt into groups of two to four per workgroup, one workgroup fits a compute unit.  A block costs
// a workgroup about a tile and a half beside its tiles (making the operands): the group size with the least of
// rounds * blocks * (tiles + 1.5).  Up to 128 workgroups K is cut so that the slices fill the 256 units once (a slice
// keeps at least 4 blocks); their partial sums are at most 256 workgroups' results.
static_assert(size_t(256) * kDgRows * 4 * 32 * sizeof(float) <= kSliceScratchBytes, "bound of the slices' workspace");
inline DgPlan digits_plan(uint32_t rows, uint32_t nb, uint32_t seq) {
    const uint32_t tiles = (seq + 31) / 32;
    DgPlan best{};
    uint64_t best_cost = ~0ull;
    for (uint32_t per = 4; per >= 2; per--) {
        DgPlan p;
        p.tiles_per_wg = per;
        p.groups = (tiles + per - 1) / per;
        p.row_tiles = (rows + kDgRows - 1) / kDgRows;
        const uint64_t wgs = static_cast<uint64_t>(p.row_tiles) * p.groups;
        p.slices = wgs > 128 ? 1 : static_cast<uint32_t>(std::max<uint64_t>(1, std::min<uint64_t>(256 / wgs, nb / 4)));
        p.cost = (wgs * p.slices + 255) / 256 * ((nb + p.slices - 1) / p.slices) * (2 * per + 3);
        if (p.cost < best_cost) {
            best_cost = p.cost;
            best = p;
        }
    }
    return best;
}

// whether the rounds of one workgroup per unit that a call takes are at least 70 % full (333 workgroups are not: IQ2_S
// 9289 x 6400 x 779 tokens 288 us in the 64-token kernel against 325; 392 are: 14336 x 4096 x 640 226 -> 172)
inline bool digits_fill_the_chip(uint32_t rows, uint32_t nb, uint32_t seq) {
    const DgPlan p = digits_plan(rows, nb, seq);
    const uint64_t wgs = static_cast<uint64_t>(p.row_tiles) * p.groups * p.slices;
    return 10 * wgs >= 7 * ((wgs + 255) / 256 * 256);
}

template <uint32_t kFmt, int kT, bool kPair>
void launch_digits(const DgPlan &p, const uint8_t *w, const uint8_t *w2, const ActView &act, float *out, float *slice_out,
                   uint32_t rows, uint32_t nb, uint32_t seq, uint32_t *left, hipStream_t stream) {
    static bool configured = false;  // above the default 64 KB of dynamic LDS
    constexpr size_t lds = DgLds<kFmt, kT>::kBytes;
    if (!allow_dynamic_lds(reinterpret_cast<const void *>(gemm_digits_kernel<kFmt, kT, kPair>), lds, &configured, "gemm_digits_kernel"))
        return;
    const uint32_t slices = slice_out ? p.slices : 1;
    const uint32_t nb_slice = (nb + slices - 1) / slices, nz = (nb + nb_slice - 1) / nb_slice;
    hipLaunchKernelGGL((gemm_digits_kernel<kFmt, kT, kPair>), dim3(p.row_tiles, p.groups, nz), dim3(kDgThreads), lds, stream, w, w2,
                       act.qs, act.d, act.digits, nz > 1 ? slice_out : out, rows, nb, seq, nb_slice);
    finish_slices(slice_out, out, (kPair ? 2 : 1) * static_cast<size_t>(seq) * rows, nz, left, stream);
}

template <uint32_t kFmt, bool kPair = false>
void launch_digits_plan(const uint8_t *w, const ActView &act, float *out, float *slice_out, uint32_t rows, uint32_t nb,
                        uint32_t seq, hipStream_t stream, const uint8_t *w2 = nullptr, uint32_t *left = nullptr) {
    const DgPlan p = digits_plan(kPair ? 2 * rows : rows, nb, seq);
    if (p.tiles_per_wg == 4)
        launch_digits<kFmt, 4, kPair>(p, w, w2, act, out, slice_out, rows, nb, seq, left, stream);
    else if (p.tiles_per_wg == 3)
        launch_digits<kFmt, 3, kPair>(p, w, w2, act, out, slice_out, rows, nb, seq, left, stream);
    else
        launch_digits<kFmt, 2, kPair>(p, w, w2, act, out, slice_out, rows, nb, seq, left, stream);
}

}  // namespace

}  // namespace rnb
