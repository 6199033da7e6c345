// Batched GEMM of Q6_K above 80 activation rows where its plan prefers it to the int8 tile kernel
// (mmq6_plan), on fp16 MFMA with whole-number operands: kai_fused_mmq_run's and the legacy op's product
// over the int8 activation plane.
//
// Arithmetic. Per 32-value block the reference takes the integer dot of the activation codes q with
// the weight codes (c - 32) times their int8 scales (one per 16 values), times the activation scale
// d8 and the superblock's d (vecdotq.cuh:447-465). sc (c - 32) is a 13-bit integer, more than fp16
// holds, but its two parts are exact: c - 32 = 16 (h - 2) + l with h the two high and l the four low
// bits, hi = 16 sc (h - 2) (multiples of 16 up to 4096) and lo = sc l (up to 1920). Activation codes are
// exact too, and every partial sum of a block is a whole number below 32 * 127 * 4096 < 2^24, so
// four MFMAs leave the block's integer dot in fp32, exactly, with no conversion left to do:
//   y += d * sum over the superblock's blocks of d8 * dot.
// The int8 tile kernel spends 20 VALU instructions per int8 MFMA on the
// two scales' combination and conversion; here a 32 x 32 x 32 block takes 128 cycles of the matrix pipe
// and about 40 VALU instructions (16 for d8, 2 for d, the rest the weights' and activation's share).
// 5120 x 17408, kernel alone: 160 rows 232 -> 133 us, 512 rows 412 -> 281 us, 2048 rows 1270 -> 975 us.
// VALU issue (conversions of weights and activation, d8) takes 41 % of the time at 512 rows and the
// matrix pipe 29 %; the rest are waits.
//
// Layout and pipeline as in kai_mmqh.cuh: D[j][i] with A = 32 weight rows per wave, B = activation
// rows; lane (col, kh) holds row col's values 16 kh .. + 16 of each block; the weights go from the
// row's wire bytes to operands in registers. The activation is staged by the whole workgroup from the
// plane: a thread loads 16 codes two stages (of 64 values) ahead, converts them to fp16 once for all
// waves and writes them to LDS a stage ahead. GK groups of waves take a part of K each and add their
// sums in LDS: the plane leaves the call no scratch for K pieces.
#pragma once

#include "kai_mmqh.cuh"

namespace kai {

constexpr int MMQ6_SB = 210;  // bytes of a superblock: ql[128], qh[64], scales[16], d

template <int CT, int GN, int GK>
struct Mmq6Tile {
    static constexpr int GROUP = 64 * GN, THREADS = GROUP * GK, BN = 32 * GN, BM = 32 * CT;
    static constexpr int CODES = 128 * BM, SCALES = 8 * BM;  // one stage: fp16 codes, two d8 per row
    static constexpr int STAGE = CODES + SCALES, DROW = 128;  // a wave's 32 superblock scales
    static constexpr int USED = GK * 2 * STAGE + GK * GN * DROW, SUMS = GK > 1 ? GK * GN * CT * 4096 : 0;
    static constexpr int TURN = GK * GN * MMQH_TURN;
    static constexpr int LDS = USED > SUMS ? (USED > TURN ? USED : TURN) : (SUMS > TURN ? SUMS : TURN);
    static constexpr int UNITS = 4 * BM;  // 16-code units of a stage
    static constexpr int PER = (UNITS + GROUP - 1) / GROUP;
    static_assert(LDS <= 160 * 1024, "LDS");
};

template <int CT, int GN, int GK, int WPE>
__global__ __launch_bounds__(64 * GN * GK) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void mmq6_kernel(
    const uint8_t *__restrict__ weight, int64_t row_bytes, int n, int k, const uint8_t *__restrict__ plane, int m,
    const float *__restrict__ inverse, void *__restrict__ dst, int64_t stride_dst, int dst_bf16, int tiles_n) {
    using T = Mmq6Tile<CT, GN, GK>;
    constexpr int GROUP = T::GROUP, BM = T::BM, PER = T::PER;
    __shared__ __align__(1024) uint8_t lds[T::LDS];
    const int lane = threadIdx.x % WAVE, wg_wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int kz = wg_wave / GN, wave = wg_wave % GN, gtid = WAVE * wave + lane;
    lds_u8 *const act = (lds_u8 *)lds + kz * 2 * T::STAGE;
    lds_u8 *const drow_lds = (lds_u8 *)lds + GK * 2 * T::STAGE + wg_wave * T::DROW;

    // each XCD (workgroups dealt round-robin over 8) gets a contiguous range of the tiles, weight
    // tiles fastest
    int t = blockIdx.x;
    if (gridDim.x % 8 == 0) t = (t % 8) * (gridDim.x / 8) + t / 8;
    const int n0 = t % tiles_n * T::BN, m0 = t / tiles_n * BM;
    const int steps = k / 256, turns = (steps + GK - 1) / GK;
    const int first = min(steps, turns * kz), count = min(steps - first, turns), last = max(4 * (first + count) - 1, 0);

    const int col = lane & 31, kh = lane >> 5, wrow0 = 32 * wave;
    const uint8_t *const wrow = weight + int64_t(min(n0 + wrow0 + col, n - 1)) * row_bytes;

    // ---- activation: unit u of a stage is 16-value group u / BM of row u % BM
    uint4 codes[PER];
    float2 scales;
    const bool scaler = gtid < BM;
    auto act_load = [&](int s) __attribute__((always_inline)) {
        const uint8_t *const block = plane + int64_t(s >> 1) * m * MMQ_BLOCK_BYTES;
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            const int u = min(gtid + p * GROUP, T::UNITS - 1);
            codes[p] = *reinterpret_cast<const uint4 *>(block + int64_t(min(m0 + u % BM, m - 1)) * MMQ_BLOCK_BYTES + 16 +
                                                        64 * (s & 1) + 16 * (u / BM));
        }
        scales = *reinterpret_cast<const float2 *>(block + int64_t(min(m0 + gtid % BM, m - 1)) * MMQ_BLOCK_BYTES + 8 * (s & 1));
    };
    auto act_store = [&](int buf) __attribute__((always_inline)) {
        lds_u8 *const at = act + buf * T::STAGE;
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            const int u = gtid + p * GROUP, row = u % BM, g = u / BM;
            if (T::UNITS % GROUP != 0 && u >= T::UNITS) continue;
            const uint32_t f = 0x80808080u;  // int8 -> x + 128
            const v8h_t a = bytes8_to_h(codes[p].x ^ f, codes[p].y ^ f, 128.0f, h2_t{1, 1});
            const v8h_t b = bytes8_to_h(codes[p].z ^ f, codes[p].w ^ f, 128.0f, h2_t{1, 1});
            store16(at + g * BM * 32 + mmqh_swz(row, 0), __builtin_bit_cast(uint4, a));
            store16(at + g * BM * 32 + mmqh_swz(row, 1), __builtin_bit_cast(uint4, b));
        }
        if (scaler) {
            store_unaligned(at + T::CODES + 4 * gtid, scales.x);
            store_unaligned(at + T::CODES + 4 * (BM + gtid), scales.y);
        }
    };

    // ---- weights: the lane's half kh of every 32-value block; half a superblock's codes are reloaded
    // when its last block has been converted
    uint4 ql[4], qh[2], sc, sc_next;
    uint32_t d, d_next;
    auto wload = [&](int h, int step) __attribute__((always_inline)) {
        const uint8_t *const p = wrow + int64_t(MMQ6_SB) * step;
        ql[2 * h] = load_unaligned<uint4>(p + 64 * h + 16 * kh);
        ql[2 * h + 1] = load_unaligned<uint4>(p + 64 * h + 32 + 16 * kh);
        qh[h] = load_unaligned<uint4>(p + 128 + 32 * h + 16 * kh);
    };
    auto wscales = [&](int step) __attribute__((always_inline)) {
        const uint8_t *const p = wrow + int64_t(MMQ6_SB) * step;
        sc_next = load_unaligned<uint4>(p + 192);
        d_next = load_unaligned<uint16_t>(p + 208);
    };
    // operands of block kb: hi and lo of its two MFMAs
    auto convert = [&](auto kbtag, v8h_t (&hi)[2], v8h_t (&lo)[2]) __attribute__((always_inline)) {
        constexpr int kb = decltype(kbtag)::value, h = kb / 4, s = kb % 4;
        const uint32_t word = kb < 2 ? sc.x : kb < 4 ? sc.y : kb < 6 ? sc.z : sc.w;  // scales 2 kb, 2 kb + 1
        const int scale = static_cast<int8_t>(word >> (16 * (kb & 1) + 8 * kh));
        const _Float16 f = static_cast<_Float16>(static_cast<float>(scale));
        const h2_t sf = {f, f}, s16 = sf * h2_t{16, 16}, off = sf * h2_t{-32, -32};
        const uint4 l = ql[2 * h + (s & 1)], u = qh[h];
        const uint32_t lw[4] = {l.x, l.y, l.z, l.w}, uw[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            hi[i] = nibbles8_to_h((uw[2 * i] >> (2 * s)) & 0x03030303u, (uw[2 * i + 1] >> (2 * s)) & 0x03030303u, s16, off);
            lo[i] = nibbles8_to_h((lw[2 * i] >> (4 * (s >> 1))) & 0x0f0f0f0fu, (lw[2 * i + 1] >> (4 * (s >> 1))) & 0x0f0f0f0fu,
                                  sf, h2_t{0, 0});
        }
    };

    float acc[CT][16], sum[CT][16];
#pragma unroll
    for (int b = 0; b < CT; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[b][r] = 0.0f;
    v8h_t hi[2], lo[2], hi_next[2], lo_next[2];
    lds_u8 *const b_at[2] = {act + 2 * BM * 16 * kh + mmqh_swz(col, 0), act + 2 * BM * 16 * kh + mmqh_swz(col, 1)};

    // Stage J of step i (LDS buffer J % 2): the activation of stage s + 1 (loaded a stage before) goes to
    // the other buffer, whose last reader was stage s - 1, that of stage s + 2 is loaded; the weights'
    // halves half a superblock ahead. Block by block the products, the next block's weights converted
    // meanwhile.
    auto stage = [&](int i, auto jtag) __attribute__((always_inline)) {
        constexpr int J = decltype(jtag)::value;
        const int step = first + i, s = 4 * step + J;
        act_store((J + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);
        act_load(min(s + 2, last));
        if constexpr (J == 0) wload(1, step);
        if constexpr (J == 2) {
            wload(0, min(step + 1, last >> 2));
            wscales(min(step + 1, last >> 2));
        }
        if constexpr (J == 3) {  // the superblock's scales of the wave's rows
            if (kh == 0) store_unaligned(drow_lds + 4 * col, half_bits_to_float(d));
        }
        auto block = [&](auto btag) __attribute__((always_inline)) {
            constexpr int B = decltype(btag)::value, KB = 2 * J + B;
            if constexpr (KB == 7) {
                sc = sc_next;
                d = d_next;
            }
            lds_u8 *const at = act + (J & 1) * T::STAGE + T::CODES + 4 * (B * BM + col);
            v16f_t dot[2];
            float d8[2];
            // a tile's products run while the tile before is scaled
            auto tile = [&](int tm) __attribute__((always_inline)) {
                const v8h_t x0 = load_unaligned<v8h_t>(b_at[0] + (J & 1) * T::STAGE + B * 2 * BM * 32 + 1024 * tm);
                const v8h_t x1 = load_unaligned<v8h_t>(b_at[1] + (J & 1) * T::STAGE + B * 2 * BM * 32 + 1024 * tm);
                d8[tm & 1] = load_unaligned<float>(at + 128 * tm);
                v16f_t v = {};
                v = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi[0], x0, v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi[1], x1, v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo[0], x0, v, 0, 0, 0);
                dot[tm & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo[1], x1, v, 0, 0, 0);
            };
            tile(0);
            convert(std::integral_constant<int, (KB + 1) % 8>{}, hi_next, lo_next);
#pragma unroll
            for (int tm = 0; tm < CT; ++tm) {
                __builtin_amdgcn_sched_barrier(0);
                if (tm + 1 < CT) tile(tm + 1);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    sum[tm][r] = KB == 0 ? d8[tm & 1] * dot[tm & 1][r] : fmaf(d8[tm & 1], dot[tm & 1][r], sum[tm][r]);
                    asm volatile("" : "+v"(sum[tm][r]));  // here: left to its use, every block's dots stay live
                }
            }
#pragma unroll
            for (int p = 0; p < 2; ++p) hi[p] = hi_next[p], lo[p] = lo_next[p];
            __builtin_amdgcn_sched_barrier(0);
        };
        __builtin_amdgcn_sched_barrier(0);
        block(std::integral_constant<int, 0>{});
        block(std::integral_constant<int, 1>{});
        if constexpr (J == 3) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                __builtin_amdgcn_sched_barrier(0);
                const float4 f = __builtin_bit_cast(float4, load_unaligned<uint4>(drow_lds + 32 * q + 16 * kh));
                const float df[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
                for (int tm = 0; tm < CT; ++tm)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[tm][4 * q + e] = fmaf(df[e], sum[tm][4 * q + e], acc[tm][4 * q + e]);
            }
        }
        mmqh_barrier();
    };
    if (count > 0) {
        act_load(4 * first);
        act_store(0);
        act_load(min(4 * first + 1, last));
        wload(0, first);
        wscales(first);
        sc = sc_next;
        d = d_next;
        convert(std::integral_constant<int, 0>{}, hi, lo);
    }
    mmqh_barrier();
    for (int i = 0; i < turns; ++i) {
        if (GK == 1 || i < count) {
            stage(i, std::integral_constant<int, 0>{});
            stage(i, std::integral_constant<int, 1>{});
            stage(i, std::integral_constant<int, 2>{});
            stage(i, std::integral_constant<int, 3>{});
        } else {  // a group whose run is a step shorter meets the others at their barriers
#pragma unroll
            for (int j = 0; j < 4; ++j) mmqh_barrier();
        }
    }
    v16f_t out[CT];
#pragma unroll
    for (int tm = 0; tm < CT; ++tm)
#pragma unroll
        for (int r = 0; r < 16; ++r) out[tm][r] = acc[tm][r];
    if constexpr (GK > 1) mmqh_add_groups<CT, GK>(out, (lds_u8 *)lds, GN, kz, wave, lane);
    lds_u8 *const mine = (lds_u8 *)lds + wg_wave * MMQH_TURN;
    if (dst_bf16) mmqh_store<2, CT, GK>(out, mine, dst, stride_dst, inverse, m0, n0 + wrow0, m, n, kz, lane);
    else mmqh_store<1, CT, GK>(out, mine, dst, stride_dst, inverse, m0, n0 + wrow0, m, n, kz, lane);
}

// The product on its plan's configuration; false: the int8 tile kernel is to take it.
bool launch_mmq6(const void *weight, int64_t n, int64_t k, int64_t m, const uint8_t *plane, const float *inverse, void *dst,
                 bool dst_bf16, int64_t stride_dst, hipStream_t stream);

}  // namespace kai
