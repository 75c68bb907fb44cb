// Dense W4A8 GEMM on wide streamed-K tiles (gfx950 fp8 MFMA): the dense op above the GEMV's rows.
//
// Replaces the reference's tiled WMMA GEMM (moe_gemm_tiled.h:29-350) for op-layout int4 weights
// of group 128 and any K. The schedule is this file's own:
//
//   * a work-group owns BM x BN outputs, its waves WM x WN pieces of 16 MT x 16 NT; per
//     128-wide K group the e4m3 rows (BM x 128 bytes) and the weights, decoded to e4m3(n - z)
//     (BN x 128 bytes), pass through LDS (two slots, one barrier a group), so that every byte is
//     loaded once per work-group, along its row (four or eight lanes a row: whole cache accesses;
//     the MFMA operand order touches a row per lane), and every nibble is decoded once per BM rows;
//   * the decode of group g + 1 (registers to LDS) stands between the MFMAs of group g. Raw nibbles
//     with the zero-point term taken off the sums are cheaper to make (12 operations a piece
//     instead of 52), but what cancels later is rounded first: at K = 12288 that put 4.8 in 100
//     fp16 results off the rounded exact value instead of 2.6 with normal rows, 1.1 instead of 0.09
//     with non-negative ones (the general tiles, which this file replaces there, decode too);
//   * operands go in weights first, so a lane holds one row's four adjacent columns; the fold
//     run += partial * scale of row fragment i follows the MFMAs of i + 1, its fp16 scales from an
//     LDS table of 16 groups;
//   * XCD-aware order: an XCD takes a contiguous run of tiles, eight row tiles by as many column
//     tiles as there are, so its L2 serves every row and weight several times.
//
// The largest tile is bound by its LDS reads and VALU work (decode 3.25, fold 4 an MFMA) beside the
// MFMAs, the small ones by the operations of one wave a SIMD: about 0.5 us a K group. Measured (us
// a call of the op, zero-points, act-quant included; general or 64 x 256 tiles or GEMV -> these):
// (N, K) = (4096, 12288) M = 2048 351 -> 148 (1.4 PF/s); (12288, 4096) M = 2048 267 -> 158, M = 48
// 34 -> 26; (4096, 4096) M = 512 58 -> 33; (8192, 8192) M = 1 67 -> 39. On raw nibbles, with 32 x
// 128 to 128 x 256 tiles: 155, 153, 26, 31, 40.
#include <algorithm>
#include <type_traits>

#include "grouped_params.h"

namespace w4a8 {
namespace {

constexpr int kWtChunk = 16;      // K groups per table
constexpr int kWtSlots = 2;       // K groups in LDS
constexpr int kWtXcds = 8;
constexpr int kWtRunRows = 8;     // row tiles of an XCD's run

template <int WM_, int WN_, int MT_, int NT_>
struct WtCfg {
    static constexpr int WM = WM_, WN = WN_, MT = MT_, NT = NT_;
    static constexpr int kThreads = 64 * WM * WN;
    static constexpr int BM = WM * MT * 16, BN = WN * NT * 16;
    static constexpr int ACH = BM * 8 / kThreads;      // 16-byte row pieces per thread and group
    static constexpr int BCH = BN * 4 / kThreads;      // 16-byte weight pieces
    static_assert(ACH * kThreads == BM * 8 && BCH * kThreads == BN * 4, "pieces must divide");
    static_assert(BCH <= MT, "a row fragment's MFMAs cover the decode of one piece");
    // LDS (bytes): kWtSlots slots of rows and decoded weights, the scales of a chunk of groups,
    // the decode tables
    static constexpr int B = BM * kGroup;                       // weights behind a slot's rows
    static constexpr int kSlot = B + BN * kGroup;
    static constexpr int SC = kWtSlots * kSlot;                 // [16][BN] fp16
    static constexpr int LUT = SC + kWtChunk * BN * 2;          // [16] 16-byte tables
    static constexpr int kLds = LUT + 16 * 16;
};

// ZP: weights with zero-points (else the zero point is 8)
template <typename C, bool ZP>
__global__ void __launch_bounds__(C::kThreads, 2) wide_tiles_kernel(Params p, int mtiles, int ntiles) {
    constexpr int MT = C::MT, NT = C::NT, BM = C::BM, BN = C::BN;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int items = mtiles * ntiles;
    const int per = (items + kWtXcds - 1) / kWtXcds;
    const int jx = blockIdx.x / kWtXcds;
    const int item = (int)(blockIdx.x % kWtXcds) * per + jx;
    if (jx >= per || item >= items) return;
    // runs of kWtRunRows row tiles (the last run may be shorter), column tiles inside a run
    const int run_items = kWtRunRows * ntiles;
    const int m0 = item / run_items * kWtRunRows;
    const int rows_here = std::min(kWtRunRows, mtiles - m0);
    const int rem = item % run_items;
    const int m_tile = m0 + rem % rows_here, n_tile = rem / rows_here;

    const int row0 = m_tile * BM, col0 = n_tile * BN;
    const int M = (int)p.P, N = p.N;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / C::WN, wn = wave % C::WN;
    const int q = lane >> 4, c16 = lane & 15;
    const int K = p.K, G = p.G;
    // rows and columns past the end read the last one (never stored)
    auto xrow = [&](int m) __attribute__((always_inline)) { return std::min(row0 + m, M - 1); };
    auto wrow = [&](int n) __attribute__((always_inline)) { return std::min(col0 + n, N - 1); };
    const uint8_t* we = reinterpret_cast<const uint8_t*>(p.w);
    const uint16_t* se = reinterpret_cast<const uint16_t*>(p.scales);

    // ---- staging: 32-bit byte offsets from the rows and the expert's slice ----
    // place of row r in LDS: with the piece swizzle, equal pieces of sixteen rows lie in different
    // banks (without it a third of the LDS cycles were conflicts: (12288, 4096) M = 2048 169 -> 158 us)
    auto lrow = [](int r) __attribute__((always_inline)) { return r ^ ((r >> 3) & 1); };
    uint32_t aoff[C::ACH], boff[C::BCH], zoff[C::BCH];
    int adst[C::ACH], bdst[C::BCH][2], zsh[C::BCH];
#pragma unroll
    for (int i = 0; i < C::ACH; ++i) {
        const int c = tid + i * C::kThreads, r = c >> 3, ch = c & 7;
        aoff[i] = (uint32_t)xrow(r) * (uint32_t)K + (uint32_t)ch * 16u;
        adst[i] = lrow(r) * kGroup + ((ch ^ (r & 7)) << 4);
    }
#pragma unroll
    for (int i = 0; i < C::BCH; ++i) {
        // piece pc (32 nibbles) of weight row r becomes pieces 2 pc and 2 pc + 1 of its LDS row
        const int c = tid + i * C::kThreads, r = c >> 2, pc = c & 3, n = wrow(r);
        boff[i] = (uint32_t)n * (uint32_t)(K / 2) + (uint32_t)pc * 16u;
        zoff[i] = (uint32_t)(n >> 3) * (uint32_t)G * 4u;
        zsh[i] = 4 * (n & 7);
#pragma unroll
        for (int h = 0; h < 2; ++h) bdst[i][h] = C::B + lrow(r) * kGroup + (((2 * pc + h) ^ (r & 7)) << 4);
    }
    u32x4 ar[2][C::ACH], br[2][C::BCH];
    uint32_t zr[2][ZP ? C::BCH : 1];
    auto issue = [&](int g, auto setc) __attribute__((always_inline)) {
        constexpr int s = decltype(setc)::value;
        const int gg = std::min(g, G - 1);                     // past the end: never used
        const uint8_t* ab = p.xq + (uint32_t)gg * kGroup;
        const uint8_t* bb = we + (uint32_t)gg * 64u;
        if constexpr (ZP) {
            const uint8_t* zb = reinterpret_cast<const uint8_t*>(p.zeros) + (uint32_t)gg * 4u;
#pragma unroll
            for (int i = 0; i < C::BCH; ++i) zr[s][i] = *reinterpret_cast<const uint32_t*>(zb + opaque_u32(zoff[i]));
        }
#pragma unroll
        for (int i = 0; i < C::BCH; ++i) br[s][i] = *reinterpret_cast<const u32x4*>(bb + opaque_u32(boff[i]));
#pragma unroll
        for (int i = 0; i < C::ACH; ++i) ar[s][i] = *reinterpret_cast<const u32x4*>(ab + opaque_u32(aoff[i]));
    };
    const DecodeMasks masks = decode_masks();
    uint4 lut[ZP ? C::BCH : 1];
    auto read_luts = [&](auto setc) __attribute__((always_inline)) {
        constexpr int s = decltype(setc)::value;
        if constexpr (ZP) {
#pragma unroll
            for (int i = 0; i < C::BCH; ++i)
                lut[i] = *reinterpret_cast<const uint4*>(lds + C::LUT + ((zr[s][i] >> zsh[i]) & 0xF) * 16);
        } else {
            (void)s;
        }
    };
    auto store_w = [&](int slot, int i, auto setc) __attribute__((always_inline)) {   // slot: byte offset
        constexpr int s = decltype(setc)::value;
        const u32x4 w = br[s][i];
        const v8i d = decode_frag(w, lut[ZP ? i : 0], masks);
        *reinterpret_cast<uint4*>(lds + slot + bdst[i][0]) = make_uint4(d[0], d[1], d[2], d[3]);
        *reinterpret_cast<uint4*>(lds + slot + bdst[i][1]) = make_uint4(d[4], d[5], d[6], d[7]);
    };
    auto store_a = [&](int slot, auto setc) __attribute__((always_inline)) {
        constexpr int s = decltype(setc)::value;
#pragma unroll
        for (int i = 0; i < C::ACH; ++i) *reinterpret_cast<u32x4*>(lds + slot + adst[i]) = ar[s][i];
    };

    // ---- scales of the 16 groups from g0: eight groups an item, loads first, clamped ----
    uint16_t* s_sc = reinterpret_cast<uint16_t*>(lds + C::SC);
    auto build = [&](int g0) __attribute__((always_inline)) {
        for (int it = tid; it < BN * 2; it += C::kThreads) {
            const int n = it % BN, h = it / BN;
            const uint16_t* sp = se + (int64_t)wrow(n) * G;
            uint16_t sv[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) sv[t] = sp[std::min(g0 + 8 * h + t, G - 1)];
#pragma unroll
            for (int t = 0; t < 8; ++t) s_sc[(8 * h + t) * BN + n] = sv[t];
        }
    };

    v4f run[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) run[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    // One K group from its LDS slot (byte offset), gl its index in the chunk. The pieces of the
    // next group are decoded and stored between the MFMAs of the row fragments.
    const int a_lane = (wm * MT * 16 + lrow(c16)) * kGroup;
    const int b_lane = C::B + (wn * NT * 16 + lrow(c16)) * kGroup;
    const int p0 = ((2 * q) ^ (c16 & 7)) << 4, p1 = ((2 * q + 1) ^ (c16 & 7)) << 4;
    auto frag = [&](const uint8_t* r) __attribute__((always_inline)) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(r + p0), hi = *reinterpret_cast<const u32x4*>(r + p1);
        return v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
    };
    auto compute = [&](int slot, int gl, int next_slot, auto nextc) __attribute__((always_inline)) {
        v8i bf[NT];
        uint2 sc[NT];                                          // scales of the lane's four columns
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            bf[j] = frag(lds + slot + b_lane + j * 16 * kGroup);
            sc[j] = *reinterpret_cast<const uint2*>(s_sc + gl * BN + (wn * NT + j) * 16 + 4 * q);
        }
        read_luts(nextc);
        v4f pend[2][NT];
        auto fold = [&](int i, const v4f (&t)[NT]) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t w = r < 2 ? sc[j].x : sc[j].y;
                    run[i][j][r] = fmaf(t[j][r], __half2float(__ushort_as_half((uint16_t)((r & 1) ? w >> 16 : w & 0xFFFF))),
                                        run[i][j][r]);
                }
        };
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const v8i af = frag(lds + slot + a_lane + i * 16 * kGroup);
#pragma unroll
            for (int j = 0; j < NT; ++j) pend[i & 1][j] = mfma_16x16x128(bf[j], af, v4f{0.f, 0.f, 0.f, 0.f});
            if (i < C::BCH) store_w(next_slot, i, nextc);
            if (i > 0) fold(i - 1, pend[(i - 1) & 1]);
        }
        fold(MT - 1, pend[(MT - 1) & 1]);
        store_a(next_slot, nextc);
    };

    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    // group g is computed from slot g & 1 while groups g + 1 and g + 2 are in registers or in
    // flight; group g + 1 goes to the other slot, read last before the previous barrier
    auto group = [&](int g, auto setc, auto nextc) __attribute__((always_inline)) {
        issue(g + 2, setc);
        __builtin_amdgcn_sched_barrier(0);
        compute(decltype(setc)::value * C::kSlot, g & (kWtChunk - 1), decltype(nextc)::value * C::kSlot, nextc);
        lds_barrier();
    };
    issue(0, S0{});
    issue(1, S1{});
    if (tid < 16) *reinterpret_cast<uint4*>(lds + C::LUT + tid * 16) = load_table(tid);
    if constexpr (!ZP) lut[0] = load_table(8);
    build(0);
    lds_barrier();
    read_luts(S0{});
#pragma unroll
    for (int i = 0; i < C::BCH; ++i) store_w(0, i, S0{});
    store_a(0, S0{});
    lds_barrier();
    for (int g = 0; g < G; g += 2) {
        if (g > 0 && (g & (kWtChunk - 1)) == 0) {
            build(g);                                          // (every wave is past the old ones)
            lds_barrier();
        }
        group(g, S0{}, S1{});
        if (g + 1 < G) group(g + 1, S1{}, S0{});
    }

    // ---- epilogue: lane (q, c16) holds row 16 i + c16, columns 4 q .. 4 q + 3 ----
    const bool vec = N % 4 == 0;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = row0 + (wm * MT + i) * 16 + c16;
        if (m >= M) continue;
        const float a = p.asc[m];
        __half* orow = reinterpret_cast<__half*>(p.out) + (int64_t)m * N;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int col = col0 + (wn * NT + j) * 16 + 4 * q;
            if (col >= N) continue;
            __half v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = __float2half(as_f32(run[i][j][r] * a));
            if (vec) {
                const __half2 v01 = __halves2half2(v[0], v[1]), v23 = __halves2half2(v[2], v[3]);
                *reinterpret_cast<uint2*>(orow + col) = make_uint2(__builtin_bit_cast(uint32_t, v01),
                                                                   __builtin_bit_cast(uint32_t, v23));
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (col + r < N) orow[col + r] = v[r];
            }
        }
    }
}

template <typename C, bool ZP>
int launch_wide_z(const Params& p, hipStream_t s) {
    const int ntiles = (p.N + C::BN - 1) / C::BN;
    const int mtiles = (int)((p.P + C::BM - 1) / C::BM);
    const int64_t items = (int64_t)mtiles * ntiles;
    const void* fn = reinterpret_cast<const void*>(&wide_tiles_kernel<C, ZP>);
    if (int rc = reserve_dyn_lds(fn, C::kLds, "wide_tiles_kernel")) return rc;
    launch_kernel(&wide_tiles_kernel<C, ZP>, dim3((unsigned)((items + kWtXcds - 1) / kWtXcds * kWtXcds)),
                  dim3(C::kThreads), (size_t)C::kLds, s, p, mtiles, ntiles);
    return check_launch("wide_tiles_kernel");
}

template <typename C>
int launch_wide_t(const Params& p, hipStream_t s) {
    return p.zeros ? launch_wide_z<C, true>(p, s) : launch_wide_z<C, false>(p, s);
}

using Wt32x64 = WtCfg<1, 4, 2, 1>;     // four waves
using Wt64x64 = WtCfg<1, 4, 4, 1>;
using Wt64x128 = WtCfg<2, 4, 2, 2>;    // eight waves
using Wt128x128 = WtCfg<2, 2, 4, 4>;   // four
using Wt256x128 = WtCfg<4, 2, 4, 4>;   // eight

}  // namespace

bool wide_tiles_supported(int64_t x_rows, int64_t K, int64_t N, int64_t group_size, bool e2m1) {
    return !e2m1 && group_size == kGroup && K % kGroup == 0 && x_rows * K < (int64_t)1 << 31 &&
           N * (K / 2) < (int64_t)1 << 31;
}

int launch_wide_tiles(const GroupedArgs& a, hipStream_t s) {
    const Params p = make_params(a);
    if (p.P == 0) return W4A8_OK;
    if (!wide_tiles_supported(a.x_rows, a.K, a.N, a.group_size, a.e2m1) || a.w_frag || p.xq == nullptr ||
        p.asc == nullptr || a.epi != Epi::kHalf || a.expert_ids != nullptr) {
        set_error("wide tiles: need op-layout int4 weights of group 128, prequantised rows with group "
                  "sums, expert slices and rows below 2 GiB, fp16 out");
        return W4A8_ERR_INVALID;
    }
    // us at K = 4096, act-quant included, of r work-groups a CU (at once or in rounds): a + b r. A
    // small tile's K step takes less time, a large one's multiplies more. Against the fastest tile of
    // each size, over (N, K) = (4096, 1024), (6144, 2048), (16384, 512), (4096, 4096), (12288, 4096),
    // (28672, 4096), (2048, 6144), (8192, 8192), (4096, 12288) at M = 17 .. 2048: the choice is
    // within 6% of it, within 12% at K <= 1024.
    const int64_t cus = device_cu_count();
    auto cost = [&](int bm, int bn, double a0, double b) {
        const int64_t t = (a.P + bm - 1) / bm * ((a.N + bn - 1) / bn);
        return a0 + b * (double)((t + cus - 1) / cus);
    };
    const double c[5] = {cost(32, 64, 16, 6.5), cost(64, 64, 18, 9.3), cost(64, 128, 14, 18),
                         cost(128, 128, 20, 27), cost(256, 128, 5, 52)};
    switch (std::min_element(c, c + 5) - c) {
        case 0: return launch_wide_t<Wt32x64>(p, s);
        case 1: return launch_wide_t<Wt64x64>(p, s);
        case 2: return launch_wide_t<Wt64x128>(p, s);
        case 3: return launch_wide_t<Wt128x128>(p, s);
        default: return launch_wide_t<Wt256x128>(p, s);
    }
}

}  // namespace w4a8
