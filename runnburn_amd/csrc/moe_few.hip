// Routed experts of a batch on the few-token GEMM's tiles (gemm_few.h): every expert's slots in tiles of 16 or 32, a workgroup per
// (tile, 64 rows), a wave per 16 rows.
//   gate/up   mid[slot][n_ff] = silu(Wg[e] . a_tok) * (Wu[e] . a_tok), both Q4_K            fanout.rs:260-327, activation.rs:73-89
//   down      slot_out[slot][n_embd] = route[slot] * (Wd[e] . Q8_K(mid[slot])), Q4_K, Q5_K or Q6_K
// (crates/rnb-llm/src/engine/models/shared_expert_moe/moe_view/fanout.rs, crates/rnb-cpu/src/kernels/activation.rs)
//
// An expert's rows are read once per tile and little is computed with them, so what counts are waves in flight.  The four waves of a
// workgroup share the tile's activations (each fetches a quarter of the next block's while the present one's are used, one barrier a
// block) and have strips of LDS of their own for their rows: 42 KB for gate and up with 32 slots, three workgroups a compute unit.
// moe_mfma.hip's workgroups stage a whole tile of all blocks first, which leaves room for one, and 191 tiles of 128 experts
// x top-8 at 512 tokens kept 191 of 256 units busy.  A wave walks its rows' blocks in order with the same roundings, so the bits are
// those of moe_mfma.hip.  Measured, us a call (moe_mfma.hip : every wave with activations of its own : shared): 128 x top-8 of 768 x
// 2048 at 512 tokens 194 : 203 : 177, at 64 110 : 103 : 99, 64 x top-8 of 512 x 2816 at 446 161 : 138 : 130, 128 x top-8 of 1024 x 4096 at
// 512 466 : 450 : 390; grids that fit at once wait for the barrier instead (8 x top-2 of 2048 x 4096 at 64 93 : 61 : 64).  Two waves a
// workgroup 10 % slower, eight 7 - 15 %, 32 rows a wave 5 - 25 %; two and four K slices a row tile were up to 10 % faster on the smallest
// grids and 5 % slower on large ones.
#include "gemm_few.h"

namespace rnb {

namespace {

constexpr int kMfWaves = 4;

// a workgroup's LDS: the waves' strips (one per matrix), then two buffers with a block's activations, sums and scales of the tile's slots
template <uint32_t kFmt, int kMT, int kMats>
struct MfLds {
    typedef FewLds<kFmt, kMT, 1, kMats> L;
    static constexpr int kStrips = kMats * L::kStrip;  // a wave's
    static constexpr int kDig = kMT * 4096, kDx = kDig + (FewRows<kFmt>::kMins ? kMT * 256 : 0), kBuf = kDx + 256;
    static constexpr int kBytes = kMfWaves * kStrips + 2 * kBuf;
    static_assert(kBytes <= 160 * 1024, "LDS of a compute unit");
};

template <uint32_t kFmt, int kMT, int kMats>
__global__ void __launch_bounds__(kWave *kMfWaves)
    moe_few_kernel(const uint8_t *__restrict__ w_all, const uint8_t *__restrict__ w2_all, const uint8_t *__restrict__ w_shared,
                   const uint8_t *__restrict__ w2_shared, uint32_t n_routed, const int8_t *__restrict__ aq,
                   const float *__restrict__ ad, const uint8_t *__restrict__ adig, const uint32_t *__restrict__ units,
                   const uint32_t *__restrict__ act_rows, const uint32_t *__restrict__ out_rows,
                   const float *__restrict__ out_scale, float *__restrict__ out, uint32_t rows, uint32_t nb, uint32_t unit0) {
    typedef FewLds<kFmt, kMT, 1, kMats> L;
    typedef MfLds<kFmt, kMT, kMats> S;
    typedef FewRows<kFmt> R;
    constexpr int kActs = kMfWaves * S::kStrips;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, kq = lane >> 4;
    const uint32_t *unit = units + 3 * (unit0 + blockIdx.y);
    const uint32_t expert = unit[0], start = unit[1], live = unit[2];
    const uint32_t row0 = (blockIdx.x * kMfWaves + wave) * 16;
    const uint32_t first = min(row0, (rows - 1) & ~15u), last_row = min(rows - 1 - first, 15u);  // clamped loads, masked stores
    const uint32_t row_bytes = nb * static_cast<uint32_t>(R::kBytes), last_tok = live - 1;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lptr_t)lds));
    const uint8_t *strips = lds + wave * S::kStrips;
    const uint32_t strips0 = lds0 + wave * S::kStrips;
    const size_t per_expert = static_cast<size_t>(rows) * row_bytes, at = static_cast<size_t>(first) * row_bytes;
    const uint8_t *w_base[2] = {expert_base(w_all, w_shared, n_routed, expert, per_expert) + at,
                                expert_base(w2_all, w2_shared, n_routed, expert, per_expert) + at};

    // the list before the first fill: loads return in order, and the compiler counts its own only.  The waves share the fetching of the
    // tile's activations, four slots a load
    const uint32_t *list = act_rows + start;
    const uint32_t rr = __umul24(lane, R::kInv) >> 16, j = lane - rr * R::kPieces;
    constexpr int kGroups = (4 * kMT + kMfWaves - 1) / kMfWaves;
    uint32_t row_off[L::kFills], act_off[kGroups];
#pragma unroll
    for (int i = 0; i < kGroups; i++) {
        const uint32_t g = wave + i * kMfWaves;
        act_off[i] = list[min(4 * g + kq, last_tok)] * (nb * 256u) + 16 * (l16 ^ (4 * (g & 3) + kq));
    }
    // a token's sixteen bytes of sums are four lanes' dwords
    const uint32_t dig_off = list[min(16 * (wave % kMT) + (lane >> 2), last_tok)] * (nb * 16u) + 4 * (lane & 3);
    const uint32_t dx_off = list[min(static_cast<uint32_t>(lane), last_tok)] * (nb * 4u);
#pragma unroll
    for (int k = 0; k < L::kFills; k++) row_off[k] = min(k * R::kPer + rr, last_row) * row_bytes;

    auto run = [&](auto tiles_tag) {  // with the token tiles that have live slots
        constexpr int kLive = decltype(tiles_tag)::value;
        auto issue_w = [&](uint32_t b) {
#pragma unroll
            for (int m = 0; m < kMats; m++) {
                const uint8_t *src = w_base[m] + R::block_off(b);
#pragma unroll
                for (int k = 0; k < L::kFills; k++) lds_fill16(src, R::piece(row_off[k], j, b), strips0 + m * L::kStrip + k * 1024);
            }
        };
        auto issue_a = [&](uint32_t b) {
            const uint32_t dst = lds0 + kActs + (b & 1) * S::kBuf;
#pragma unroll
            for (int i = 0; i < kGroups; i++) {
                const uint32_t g = wave + i * kMfWaves;  // places of no slot keep what they hold
                if (g < 4u * kLive && 4 * g < live) lds_fill16(reinterpret_cast<const uint8_t *>(aq) + b * 256u, act_off[i], dst + g * 1024);
            }
            if constexpr (R::kMins)
                if (wave < kLive) lds_fill4(adig + b * 16u, dig_off, dst + S::kDig + wave * 256);
            if (wave == kMfWaves - 1) lds_fill4(reinterpret_cast<const uint8_t *>(ad) + b * 4u, dx_off, dst + S::kDx);
        };
        float acc[kMats][1][kLive][4];
#pragma unroll
        for (int m = 0; m < kMats; m++)
#pragma unroll
            for (int t = 0; t < kLive; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[m][0][t][r] = 0.0f;
        issue_a(0);
        issue_w(0);
        for (uint32_t b = 0; b < nb; b++) {
            wait_fills();
            __syncthreads();  // everybody's part of block b has come, block b - 1 has been read
            if (b + 1 < nb) issue_a(b + 1);
            const int at = static_cast<int>(kActs + (b & 1) * S::kBuf - wave * S::kStrips);  // from the wave's strips
            FewBlock<kFmt, kLive, 1, kMats> blk;
            blk.read(strips, at, at + S::kDig, reinterpret_cast<const float *>(strips + at + S::kDx), l16, kq, last_row, nb, b);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the strips have been read
            if (b + 1 < nb) issue_w(b + 1);
            blk.template multiply<true>(acc, kq);
        }
        const uint32_t row = row0 + l16;
#pragma unroll
        for (int t = 0; t < kLive; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t tok = 16 * t + 4 * kq + r;
                if (tok < live && row < rows) {
                    const uint32_t slot = out_rows[start + tok];
                    // fanout.rs:306-308: the expert's output times the slot's route weight
                    out[static_cast<size_t>(slot) * rows + row] =
                        kMats == 2 ? act_mul<false>(acc[0][0][t][r], acc[kMats - 1][0][t][r]) : acc[0][0][t][r] * out_scale[slot];
                }
            }
    };
    if constexpr (kMT > 1) {
        if (live <= 16) {  // workgroup-uniform
            run(std::integral_constant<int, 1>{});
            return;
        }
    }
    run(std::integral_constant<int, kMT>{});
}

template <uint32_t kFmt, int kMT, int kMats>
void launch_moe_few(const uint8_t *w, const uint8_t *w2, const uint8_t *ws, const uint8_t *ws2, uint32_t n_routed, const ActView &act,
                    const MoeGroups &g, const uint32_t *act_rows, const float *scale, float *out, uint32_t rows, uint32_t nb,
                    hipStream_t stream) {
    static bool configured = false;
    constexpr size_t lds = MfLds<kFmt, kMT, kMats>::kBytes;
    if (!allow_dynamic_lds(reinterpret_cast<const void *>(moe_few_kernel<kFmt, kMT, kMats>), lds, &configured, "moe_few_kernel")) return;
    for (uint32_t u = 0; u < g.n_units; u += 65535)  // grid rows that a device is sure to take
        hipLaunchKernelGGL((moe_few_kernel<kFmt, kMT, kMats>), dim3((rows + 16 * kMfWaves - 1) / (16 * kMfWaves), std::min(g.n_units - u, 65535u)),
                           dim3(kWave * kMfWaves), lds, stream, w, w2, ws, ws2, n_routed, act.qs, act.d, act.digits, g.units, act_rows,
                           g.sorted_slot, scale, out, rows, nb, u);
}

}  // namespace

// us a call with tiles of 16 : of 32: 15.7 slots a group on average (64 x top-8 of 1792 x 1792 at 120 tokens) 139 : 126, 15 (32 x top-4 of
// 768 x 2048 at 120) 51.0 : 49.6; 12.5 (64 x top-8 of 512 x 2816 at 100) 61.9 : 65.4, (16 x top-2 of 1536 x 1536 at 100) 36.3 : 39.9.  Tiles of
// 64 (200 registers, two waves a SIMD) against 32: 128 x top-8 of 768 x 2048 at 512 tokens 191 : 175, at 1024 275 : 273, at 2048 455 : 472, 16 x
// top-2 of 1024 x 2304 at 400 72 : 66; only 8 x top-2 of 2048 x 4096 at 400 gained much (115 : 135).
uint32_t moe_few_tile(size_t n_slots, size_t n_groups) { return n_slots <= 14 * n_groups ? 16 : 32; }

// 32-bit offsets into the activations.  (The last piece of every other Q6_K block ends two bytes behind it, gemm_few.h: inside the
// expert's matrix, whose n_embd rows, a multiple of 256, make an even number of blocks.)
bool moe_few_supported(size_t nb_in, size_t nb_mid, size_t token_count, size_t n_slots, size_t n_ff, size_t n_embd) {
    return nb_in <= kFewMaxBlocks && nb_mid <= kFewMaxBlocks && token_count * n_embd < (size_t(1) << 32) && n_slots * n_ff < (size_t(1) << 32);
}

void launch_moe_few_gate_up(const uint8_t *gate_all, const uint8_t *up_all, const MoeShared &shared, ActView act, const MoeGroups &g,
                            float *mid, uint32_t n_ff, uint32_t nb_in, hipStream_t stream) {
    if (g.n_units == 0 || n_ff == 0) return;
    if (g.unit_tokens == 16)
        launch_moe_few<kQ4K, 1, 2>(gate_all, up_all, shared.gate, shared.up, shared.n_routed, act, g, g.sorted_token, nullptr, mid, n_ff,
                                   nb_in, stream);
    else
        launch_moe_few<kQ4K, 2, 2>(gate_all, up_all, shared.gate, shared.up, shared.n_routed, act, g, g.sorted_token, nullptr, mid, n_ff,
                                   nb_in, stream);
}

template <uint32_t kFmt>
static void moe_few_down(const uint8_t *down_all, const MoeShared &shared, const ActView &act, const MoeGroups &g, const float *slot_route,
                         float *slot_out, uint32_t n_embd, uint32_t nb_mid, hipStream_t stream) {
    if (g.unit_tokens == 16)
        launch_moe_few<kFmt, 1, 1>(down_all, down_all, shared.down, shared.down, shared.n_routed, act, g, g.sorted_slot, slot_route, slot_out,
                                   n_embd, nb_mid, stream);
    else
        launch_moe_few<kFmt, 2, 1>(down_all, down_all, shared.down, shared.down, shared.n_routed, act, g, g.sorted_slot, slot_route, slot_out,
                                   n_embd, nb_mid, stream);
}

void launch_moe_few_down(const uint8_t *down_all, const MoeShared &shared, uint32_t down_quant, ActView mid_act, const MoeGroups &g,
                         const float *slot_route, float *slot_out, uint32_t n_embd, uint32_t nb_mid, hipStream_t stream) {
    if (g.n_units == 0 || n_embd == 0) return;
    if (down_quant == kQ4K)
        moe_few_down<kQ4K>(down_all, shared, mid_act, g, slot_route, slot_out, n_embd, nb_mid, stream);
    else if (down_quant == kQ5K)
        moe_few_down<kQ5K>(down_all, shared, mid_act, g, slot_route, slot_out, n_embd, nb_mid, stream);
    else
        moe_few_down<kQ6K>(down_all, shared, mid_act, g, slot_route, slot_out, n_embd, nb_mid, stream);
}

}  // namespace rnb
