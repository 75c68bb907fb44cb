// Dense W4A8 GEMM on wide streamed-K tiles (gfx950 fp8 MFMA): the dense op above the GEMV's rows.
//
// Replaces the reference's tiled WMMA GEMM (moe_gemm_tiled.h:29-350) for op-layout int4 weights
// of group 128 and any K. Arithmetic as in w4a8_common.h (raw-nibble operands, per-group fold,
// zero-point term from row group sums). The schedule is this file's own:
//
//   * a work-group owns BM x BN outputs, its waves WM x WN pieces of 16 MT x 16 NT; per
//     128-wide K group the e4m3 rows (BM x 128 bytes) and the raw int4 rows (BN x 64 bytes)
//     pass through LDS (two slots, one barrier a group), so that every byte is loaded once
//     per work-group, along its row (four or eight lanes a row: whole cache accesses; the
//     MFMA operand order touches a row per lane), and both pieces of a wave are read from LDS;
//   * a wave spreads its NT weight fragments once a group (two ANDs and a shift a word) for MT
//     row fragments; operands go in weights first, so a lane holds one row's four adjacent
//     columns; the fold run += partial * scale of row fragment i follows the MFMAs of i + 1;
//   * scales and zero-points come 16 groups at a time into LDS tables: fp16 scales [group][row],
//     s * z as bf16 hi / lo, the rows' group sums as bf16 hi / lo (scaled by -2^-9), and the
//     zero-point term of the 16 groups is two bf16 MFMAs a block on the accumulators
//     themselves;
//   * XCD-aware order: an XCD takes a contiguous run of tiles, eight row tiles by as many column
//     tiles as there are, so its L2 serves every row and weight several times.
//
// Bound by its LDS reads and VALU work beside the MFMAs: a 64 x 64 wave piece reads 12 KB of LDS
// for 16 MFMAs (the four SIMDs' reads alone take about as long as the MFMAs), and spread plus fold
// are 7 VALU an MFMA (a loop of just these reaches 2.7 PF/s). Tried without gain: three slots
// with the next group's weights read and spread ahead, one MFMA to four folds in program order,
// two 128 x 128 work-groups a CU. Measured (us a call, GEMV / tiles before -> now, act-quant
// included): (N, K) = (4096, 12288) M = 2048 - / 342 -> 143 (1.4 PF/s), M = 64 92 / 121 -> 53;
// (12288, 4096) M = 2048 590 / 265 -> 155, M = 48 35 / 57 -> 23; (3008, 7040) M = 512 99 / 84 -> 51.
#include <algorithm>
#include <type_traits>

#include "grouped_params.h"

namespace w4a8 {
namespace {

constexpr int kWtChunk = 16;      // K groups per table
constexpr int kWtSlots = 2;       // K groups in LDS
constexpr int kWtXcds = 8;
constexpr int kWtRunRows = 8;     // row tiles of an XCD's run

using bf16x8 = __bf16 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bf16x8 wt_bf16x8(const __bf16* ptr) {
    const uint4 v = *reinterpret_cast<const uint4*>(ptr);
    bf16x8 r;
    __builtin_memcpy(&r, &v, 16);
    return r;
}

template <int WM_, int WN_, int MT_, int NT_>
struct WtCfg {
    static constexpr int WM = WM_, WN = WN_, MT = MT_, NT = NT_;
    static constexpr int kThreads = 64 * WM * WN;
    static constexpr int BM = WM * MT * 16, BN = WN * NT * 16;
    static constexpr int ACH = BM * 8 / kThreads;      // 16-byte row pieces per thread and group
    static constexpr int BCH = BN * 4 / kThreads;      // 16-byte weight pieces
    static_assert(ACH * kThreads == BM * 8 && BCH * kThreads == BN * 4, "pieces must divide");
    // LDS (bytes): kWtSlots slots of rows and weights, then the tables of a chunk of groups
    static constexpr int B = BM * kGroup;                       // weights behind a slot's rows
    static constexpr int kSlot = B + BN * 64;
    static constexpr int SC = kWtSlots * kSlot;                 // [16][BN] fp16
    static constexpr int SZ = SC + kWtChunk * BN * 2;           // [2][BN][16] bf16 (hi, lo)
    static constexpr int SA = SZ + 2 * BN * kWtChunk * 2;       // [2][BM][16] bf16
    static constexpr int kLds = SA + 2 * BM * kWtChunk * 2;
};

template <typename C>
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
    uint32_t aoff[C::ACH], boff[C::BCH];
    int adst[C::ACH];
#pragma unroll
    for (int i = 0; i < C::ACH; ++i) {
        const int c = tid + i * C::kThreads, r = c >> 3, ch = c & 7;
        aoff[i] = (uint32_t)xrow(r) * (uint32_t)K + (uint32_t)ch * 16u;
        adst[i] = r * kGroup + ((ch ^ (r & 7)) << 4);
    }
#pragma unroll
    for (int i = 0; i < C::BCH; ++i) {
        // piece c & 3 of the LDS row holds the row's piece (c & 3) ^ ((row / 4) & 3)
        const int c = tid + i * C::kThreads, r = c >> 2, pc = (c & 3) ^ ((r >> 2) & 3);
        boff[i] = (uint32_t)wrow(r) * (uint32_t)(K / 2) + (uint32_t)pc * 16u;
    }
    u32x4 ar[2][C::ACH], br[2][C::BCH];
    auto issue = [&](int g, auto setc) __attribute__((always_inline)) {
        constexpr int s = decltype(setc)::value;
        const int gg = std::min(g, G - 1);                     // past the end: never used
        const uint8_t* ab = p.xq + (uint32_t)gg * kGroup;
        const uint8_t* bb = we + (uint32_t)gg * 64u;
#pragma unroll
        for (int i = 0; i < C::BCH; ++i) br[s][i] = *reinterpret_cast<const u32x4*>(bb + opaque_u32(boff[i]));
#pragma unroll
        for (int i = 0; i < C::ACH; ++i) ar[s][i] = *reinterpret_cast<const u32x4*>(ab + opaque_u32(aoff[i]));
    };
    auto store = [&](int slot, auto setc) __attribute__((always_inline)) {   // slot: byte offset
        constexpr int s = decltype(setc)::value;
#pragma unroll
        for (int i = 0; i < C::BCH; ++i)
            *reinterpret_cast<u32x4*>(lds + slot + C::B + (tid + i * C::kThreads) * 16) = br[s][i];
#pragma unroll
        for (int i = 0; i < C::ACH; ++i) *reinterpret_cast<u32x4*>(lds + slot + adst[i]) = ar[s][i];
    };

    // ---- tables of the 16 groups from g0 ----
    uint16_t* s_sc = reinterpret_cast<uint16_t*>(lds + C::SC);
    __bf16* s_sz = reinterpret_cast<__bf16*>(lds + C::SZ);
    __bf16* s_sa = reinterpret_cast<__bf16*>(lds + C::SA);
    auto build = [&](int g0) __attribute__((always_inline)) {
        // weight rows: eight groups an item; loads first, clamped (groups past G count as 0)
        for (int it = tid; it < BN * 2; it += C::kThreads) {
            const int n = it % BN, h = it / BN, row = wrow(n);
            const uint16_t* sp = se + (int64_t)row * G;
            const int32_t* zp = p.zeros ? p.zeros + (int64_t)(row >> 3) * G : nullptr;
            uint16_t sv[8];
            int32_t zv[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int g = std::min(g0 + 8 * h + t, G - 1);
                sv[t] = sp[g];
                zv[t] = zp ? zp[g] : 0;
            }
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int t = 0; t < 8; t += 2) {
                uint32_t hb[2], lb[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int g = g0 + 8 * h + t + u;
                    const float z = zp ? (float)((zv[t + u] >> ((row & 7) * 4)) & 0xF) : 8.0f;
                    const float sz = g < G ? __half2float(__ushort_as_half(sv[t + u])) * z : 0.f;   // exact
                    const __bf16 b = (__bf16)sz;
                    hb[u] = __builtin_bit_cast(uint16_t, b);
                    lb[u] = __builtin_bit_cast(uint16_t, (__bf16)(sz - (float)b));
                    s_sc[(8 * h + t + u) * BN + n] = sv[t + u];
                }
                hi[t / 2] = hb[0] | (hb[1] << 16);
                lo[t / 2] = lb[0] | (lb[1] << 16);
            }
            *reinterpret_cast<uint4*>(s_sz + n * kWtChunk + 8 * h) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
            *reinterpret_cast<uint4*>(s_sz + (BN + n) * kWtChunk + 8 * h) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        }
        // the rows' group sums, times -2^-9 (the accumulators hold sums of n * 2^-9)
        for (int it = tid; it < BM * 4; it += C::kThreads) {
            const int r = it >> 2, t0 = 4 * (it & 3);
            const float* ap = p.asum + (int64_t)xrow(r) * G;
            float v[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) v[t] = ap[std::min(g0 + t0 + t, G - 1)];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float a = g0 + t0 + t < G ? v[t] * (-1.0f / kNibbleScale) : 0.f;
                const __bf16 b = (__bf16)a;
                s_sa[r * kWtChunk + t0 + t] = b;
                s_sa[(BM + r) * kWtChunk + t0 + t] = (__bf16)(a - (float)b);
            }
        }
    };

    v4f run[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) run[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    // zero-point term of the chunk's 16 groups on the accumulators: lane (q, c16), K slot
    // 8 q + t is group 8 (q & 1) + t; rows' operand hi (q < 2) or lo half, weights' operand hi,
    // then lo (slots 16 .. 31 repeat 0 .. 15), so the two MFMAs add (sa_hi + sa_lo)(sz_hi + sz_lo)
    auto zero_term = [&]() __attribute__((always_inline)) {
        const int go = 8 * (q & 1);
        bf16x8 zh[NT], zl[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int n = (wn * NT + j) * 16 + c16;
            zh[j] = wt_bf16x8(s_sz + n * kWtChunk + go);
            zl[j] = wt_bf16x8(s_sz + (BN + n) * kWtChunk + go);
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int m = (wm * MT + i) * 16 + c16;
            const bf16x8 sa = wt_bf16x8(s_sa + ((q < 2 ? 0 : BM) + m) * kWtChunk + go);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                run[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(zh[j], sa, run[i][j], 0, 0, 0);
                run[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(zl[j], sa, run[i][j], 0, 0, 0);
            }
        }
    };

    // one K group from its LDS slot (byte offset), gl its index in the chunk
    const int a_lane = (wm * MT * 16 + c16) * kGroup;
    const int b_lane = C::B + (wn * NT * 16 + c16) * 64 + ((q ^ ((c16 >> 2) & 3)) << 4);
    const int a0 = ((2 * q) ^ (c16 & 7)) << 4, a1 = ((2 * q + 1) ^ (c16 & 7)) << 4;
    auto compute = [&](int slot, int gl) __attribute__((always_inline)) {
        v8i bf[NT];
        uint2 sc[NT];                                          // scales of the lane's four columns
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            bf[j] = spread_nibbles(*reinterpret_cast<const uint4*>(lds + slot + b_lane + j * 16 * 64));
            sc[j] = *reinterpret_cast<const uint2*>(s_sc + gl * BN + (wn * NT + j) * 16 + 4 * q);
        }
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
            const uint8_t* A = lds + slot + a_lane + i * 16 * kGroup;
            const u32x4 lo = *reinterpret_cast<const u32x4*>(A + a0);
            const u32x4 hi = *reinterpret_cast<const u32x4*>(A + a1);
            const v8i af = {(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
#pragma unroll
            for (int j = 0; j < NT; ++j) pend[i & 1][j] = mfma_16x16x128(bf[j], af, v4f{0.f, 0.f, 0.f, 0.f});
            if (i > 0) fold(i - 1, pend[(i - 1) & 1]);
        }
        fold(MT - 1, pend[(MT - 1) & 1]);
    };

    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    // group g is computed from slot g & 1 while groups g + 1 and g + 2 are in registers or in
    // flight; group g + 1 goes to the other slot, read last before the previous barrier
    issue(0, S0{});
    issue(1, S1{});
    build(0);
    store(0, S0{});
    lds_barrier();
    auto group = [&](int g, auto setc, auto nextc) __attribute__((always_inline)) {
        issue(g + 2, setc);
        __builtin_amdgcn_sched_barrier(0);
        compute(decltype(setc)::value * C::kSlot, g & (kWtChunk - 1));
        store(decltype(nextc)::value * C::kSlot, nextc);
        lds_barrier();
    };
    for (int g = 0; g < G; g += 2) {
        if (g > 0 && (g & (kWtChunk - 1)) == 0) {
            zero_term();
            lds_barrier();                                     // every wave past the old tables
            build(g);
            lds_barrier();
        }
        group(g, S0{}, S1{});
        if (g + 1 < G) group(g + 1, S1{}, S0{});
    }
    zero_term();

    // ---- epilogue: lane (q, c16) holds row 16 i + c16, columns 4 q .. 4 q + 3 ----
    const bool vec = N % 4 == 0;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = row0 + (wm * MT + i) * 16 + c16;
        if (m >= M) continue;
        const float a = p.asc[m] * kNibbleScale;               // exact: a power of two
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

template <typename C>
int launch_wide_t(const Params& p, hipStream_t s) {
    const int ntiles = (p.N + C::BN - 1) / C::BN;
    const int mtiles = (int)((p.P + C::BM - 1) / C::BM);
    const int64_t items = (int64_t)mtiles * ntiles;
    const void* fn = reinterpret_cast<const void*>(&wide_tiles_kernel<C>);
    if (int rc = reserve_dyn_lds(fn, C::kLds, "wide_tiles_kernel")) return rc;
    launch_kernel(&wide_tiles_kernel<C>, dim3((unsigned)((items + kWtXcds - 1) / kWtXcds * kWtXcds)),
                  dim3(C::kThreads), (size_t)C::kLds, s, p, mtiles, ntiles);
    return check_launch("wide_tiles_kernel");
}

using Wt32x128 = WtCfg<1, 4, 2, 2>;    // four waves, up to four work-groups on a CU
using Wt64x128 = WtCfg<1, 4, 4, 2>;
using Wt128x128 = WtCfg<2, 2, 4, 4>;
using Wt128x256 = WtCfg<2, 4, 4, 4>;   // eight waves

}  // namespace

bool wide_tiles_supported(int64_t x_rows, int64_t K, int64_t N, int64_t group_size, bool e2m1) {
    return !e2m1 && group_size == kGroup && K % kGroup == 0 && x_rows * K < (int64_t)1 << 31 &&
           N * (K / 2) < (int64_t)1 << 31;
}

int launch_wide_tiles(const GroupedArgs& a, hipStream_t s) {
    const Params p = make_params(a);
    if (p.P == 0) return W4A8_OK;
    if (!wide_tiles_supported(a.x_rows, a.K, a.N, a.group_size, a.e2m1) || a.w_frag || p.xq == nullptr ||
        p.asum == nullptr || p.asc == nullptr || a.epi != Epi::kHalf || a.expert_ids != nullptr) {
        set_error("wide tiles: need op-layout int4 weights of group 128, prequantised rows with group "
                  "sums, expert slices and rows below 2 GiB, fp16 out");
        return W4A8_ERR_INVALID;
    }
    // The smallest tile whose grid does not pass the CUs: a group takes a work-group 0.6, 0.75,
    // 1.1 or 1.25 us by itself (the four sizes), so while CUs are free a smaller tile ends first;
    // three rounds of 64 x 128 (several of them share a CU) still lead, e.g. (N, K) = (4096, 4096),
    // us for 32 x 128 / 64 x 128 / 128 x 128 / 128 x 256: M = 256 24.6 / 28.7 / 40 / 50, M = 384
    // 30.6 / 29.7 / 41 / 51, M = 1024 50 / 43 / 45 / 54. Past that the largest tile, unless its
    // last round would be mostly empty: M = 2048 91 / 71 / 62 / 58 (256 tiles), (8192, 4096) at
    // M = 1536 129 / 102 / 91 / 102 (384 tiles).
    const int64_t cus = device_cu_count();
    auto tiles = [&](int bm, int bn) { return (a.P + bm - 1) / bm * ((a.N + bn - 1) / bn); };
    if (tiles(32, 128) <= cus) return launch_wide_t<Wt32x128>(p, s);
    if (tiles(64, 128) <= 3 * cus) return launch_wide_t<Wt64x128>(p, s);
    const int64_t big = tiles(128, 256), rounds = (big + cus - 1) / cus;
    if (20 * big >= 17 * rounds * cus) return launch_wide_t<Wt128x256>(p, s);
    return launch_wide_t<Wt128x128>(p, s);
}

}  // namespace w4a8
