// Grouped GEMM on E2M1 (mxfp4) weights with block scales of 32: gfx950 fp8 x fp4 MFMA.
//
// Replaces the reference's E2M1 tiles (moe_gemm_tiled.h:192-350 with weight_is_e2m1,
// tile_config.h:59-71) for group size 32. The schedule is this file's own:
//
//   * the int32 words go into the MFMA as they are: a lane's 16 bytes are 32 E2M1 codes, the
//     f8f6f4 MFMA's own fp4 operand, against e4m3 activations in natural k order;
//   * scales that are powers of two (an MX checkpoint's: E8M0 converted to fp16 at load, exponents
//     -14 to 15) become the MFMA's own block-scale operand, so a 128-wide K step is one MFMA per 16 x 16
//     block that accumulates in place: no fold, no masked operands. A wave looks at the fp16
//     scales as they come; a column with one that is not a normal positive power of two
//     is taken through the general form as well, which replaces its sums (one masked MFMA per
//     group and the fp32 fold run += partial * scale, the arithmetic of the scalar kernel);
//   * loads are coalesced along the weight rows (four lanes a row's 64 bytes of a step; 32
//     bytes of scales a row and four steps) and reach the MFMA's lane order through LDS, per
//     wave; the scales as E8M0 bytes, the MFMAs taking a step's byte by op_sel;
//   * operands go in weights first, so a lane ends with four adjacent output columns of one
//     row: bias, SiLU or swigluoai (gate and up interleaved) are applied in registers and
//     the row piece leaves in one store;
//   * the e4m3 rows of the tile (BM = 64 or 32) pass through LDS, two slots and one barrier
//     per 128-wide step; with BM = 16 (decode) each wave brings them itself and the loop has no
//     barrier. Four steps of weights and rows are in flight per wave;
//   * XCD-aware order: an XCD takes a contiguous run of (column tile, row block) items, so
//     the row blocks of one expert read its weights from one L2.
//
// Bound by HBM while an expert has few rows; with many, by each wave's LDS reads, MFMAs and
// barrier following one another. Measured at hidden = intermediate = 2880, 32 experts, top-4:
// gemm1 alone (16- and 64-row blocks, before: a masked MFMA and a fold per group of 32) T = 8
// 103 / 132 -> 46 / 52 us, T = 256 346 / 246 -> 158 / 106, T = 1000 925 / 515 -> 422 / 190; the
// layer with biases and swigluoai in one call (before: op by op) T = 8 380 -> 112 us, T = 1000
// 967 -> 329. Scales that are no powers of two, gemm1 in 16- / 32- / 64-row blocks: T = 8
// 102 / 114 / 133 -> 85 / 92 / 132 us, T = 1000 926 / 746 / 515 -> 645 / 428 / 536, but T = 1
// 35 / 41 / 52 -> 32 / 50 / 104: fewer, larger work-groups than before, and their loads wait. With
// such a scale in 2 of 100 columns both forms run: T = 1 35 / 41 / 52 -> 46 / 82 / 110, T = 1000
// 925 / 738 / 506 -> 674 / 500 / 439.
#include <algorithm>
#include <type_traits>

#include "grouped_params.h"

namespace w4a8 {
namespace {

constexpr int kF4Group = 32;       // weights per scale
constexpr int kF4Steps = 4;        // K steps of 128 per super-step (ring of weight loads)
constexpr int kF4Xcds = 8;
constexpr uint32_t kF4OnesHalf2 = 0x3C003C00u;   // two fp16 1.0
constexpr int kF4ScaleOne = 0x7F7F7F7F;          // E8M0 1.0

using u16x2 = unsigned short __attribute__((ext_vector_type(2)));

// 8 bytes at a 2-byte aligned address
struct __attribute__((packed, aligned(2))) F4Scales {
    uint32_t lo, hi;
};

// Block-scaled MFMA of one step: weights (fp4, E8M0 byte S of sw per lane) x rows (e4m3).
template <int S>
__device__ __forceinline__ v4f f4_mfma(const v8i& w, const v8i& a, const v4f& c, int sw) {
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, a, c, 4, 0, S, sw, 0, kF4ScaleOne);
}

template <Epi EPI, int MT, int NT>
__global__ void __launch_bounds__(256, 2) fp4_tiles_kernel(Params p, int nblocks, int ntiles) {
    constexpr bool kSilu = EPI == Epi::kSiluHalf;
    constexpr int BM = 16 * MT;
    // one row fragment (decode): each wave brings the rows it needs itself, without barriers
    constexpr bool kOwnRows = MT == 1;
    constexpr int kOutFrags = kSilu ? NT / 2 : NT;        // output fragments of a wave
    constexpr int kLoaders = kOwnRows ? 64 : 256;         // threads that share a step's rows
    constexpr int kCh = BM * 8 / kLoaders;                // 16-byte row pieces per thread and step
    static_assert(!kSilu || NT % 2 == 0, "gate and up fragments come in pairs");
    __shared__ __attribute__((aligned(16))) uint8_t s_a[(kOwnRows ? 4 : 2) * BM * kGroup];
    __shared__ uint4 s_w[4][NT][64];                      // a step's weights, per wave
    __shared__ uint4 s_s[4][NT][16];                      // a super-step's E8M0 bytes, per wave

    const int ntp = p.ntp ? p.ntp[0] : (int)p.P;
    const int live = std::min(nblocks, (int)((std::min<int64_t>(ntp, p.P) + BM - 1) / BM));
    const int items = live * ntiles;
    const int per = (items + kF4Xcds - 1) / kF4Xcds;
    const int jx = blockIdx.x / kF4Xcds;
    const int item = (int)(blockIdx.x % kF4Xcds) * per + jx;
    if (jx >= per || item >= items) return;
    const int n_tile = item / live;
    const int64_t row0 = (int64_t)(item % live) * BM;
    const int e = __builtin_amdgcn_readfirstlane(p.expert_ids ? p.expert_ids[row0 / p.block_m] : 0);
    if (e < 0 || e >= p.E) return;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, c16 = lane & 15;
    const int K = p.K, G = p.G;
    const int ncols = kSilu ? p.N / 2 : p.N;

    // lane l < BM of every wave resolves tile row l
    int slot = -1;
    const int src = lane < BM ? resolve_row(p, row0 + lane, ntp, slot) : -1;
    const uint64_t vmask = __ballot(src >= 0);
    if (vmask == 0) return;
    const int nfl = __builtin_amdgcn_readfirstlane((63 - __clzll(vmask)) / 16 + 1);   // live 16-row fragments
    const int fallback = __shfl(src, __ffsll((long long)vmask) - 1, 64);
    auto src_of = [&](int r) __attribute__((always_inline)) {   // every lane takes part
        const int s = __shfl(src, r, 64);
        return s >= 0 ? s : fallback;      // padding rows read a real row; they are not stored
    };

    // ---- weights. Lane l loads row l / 4 of fragment j, 16 of its step's 64 bytes: four lanes
    // a contiguous 64 bytes, one cache access, where the operand's own order (lane (q, c16):
    // row c16, piece q) touches a row per lane. They reach that order through LDS, the piece
    // index swizzled by the row so that the reads meet no bank conflict. ----
    const int out0 = (n_tile * 4 + wave) * kOutFrags * 16;   // first output column of the wave
    const uint8_t* we = reinterpret_cast<const uint8_t*>(p.w) + (int64_t)e * p.N * (K / 2);
    const uint8_t* se = reinterpret_cast<const uint8_t*>(p.scales + (int64_t)e * p.N * G);
    const int lrow = lane >> 2, lblk = (lane & 3) ^ ((lane >> 4) & 3);   // row, K block of the step
    // weight row of fragment j, row r of it (edge columns read row 0: never stored)
    auto wrow = [&](int j, int r) __attribute__((always_inline)) {
        const int col = out0 + 16 * (kSilu ? j % kOutFrags : j) + r;
        return col >= ncols ? 0 : (kSilu && j >= kOutFrags) ? col + ncols : col;
    };
    // (32-bit byte offsets from the expert's slices, which are below 2 GiB)
    uint32_t wp[NT], sp[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        wp[j] = (uint32_t)wrow(j, lrow) * (uint32_t)(K / 2) + (uint32_t)lblk * 16u;
        sp[j] = (uint32_t)wrow(j, lrow) * (uint32_t)G * 2u;
    }
    const int nst = (K + kGroup - 1) / kGroup;             // K steps; the last may be partial
    const int nsuper = (nst + kF4Steps - 1) / kF4Steps;

    u32x4 bw[kF4Steps][NT];
    // loads of step g; blocks past K (and steps past the last) re-read step 0: finite codes
    // against rows that are zero there
    auto issue_w = [&](int g, auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
        const uint32_t off = 4 * g + lblk < G ? (uint32_t)g * 64u : 0u;
#pragma unroll
        for (int j = 0; j < NT; ++j) bw[s][j] = *reinterpret_cast<const u32x4*>(we + opaque_u32(wp[j] + off));
    };
    auto store_w = [&](auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
#pragma unroll
        for (int j = 0; j < NT; ++j) *reinterpret_cast<u32x4*>(&s_w[wave][j][lane]) = bw[s][j];
    };
    const int wslot = 4 * c16 + (q ^ ((c16 >> 2) & 3));
    // scales of a super-step: lane l row l / 4, the four groups of step l % 4
    F4Scales raw[NT];
    auto issue_s = [&](int su) __attribute__((always_inline)) {
        const uint32_t start = 2u * (uint32_t)std::min(4 * (kF4Steps * su + (lane & 3)), G - 4);
#pragma unroll
        for (int j = 0; j < NT; ++j) raw[j] = *reinterpret_cast<const F4Scales*>(se + opaque_u32(sp[j] + start));
    };

    // ---- rows ----
    u32x4 ar[kF4Steps][kCh];
    uint32_t ap[kCh];                  // byte offsets (the rows are below 2 GiB)
    int adst[kCh];
#pragma unroll
    for (int i = 0; i < kCh; ++i) {
        const int c = (kOwnRows ? lane : tid) + i * kLoaders, r = c >> 3, ch = c & 7;
        ap[i] = (uint32_t)src_of(r) * (uint32_t)K + (uint32_t)ch * 16u;
        adst[i] = r * kGroup + ((ch ^ (r & 7)) << 4);
    }
    // step g's rows in LDS: two slots of the work-group, or one of the wave (whose LDS
    // operations stay in order)
    auto a_slot = [&](int g) __attribute__((always_inline)) { return s_a + (kOwnRows ? wave : g & 1) * BM * kGroup; };
    auto issue_a = [&](int g, auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
#pragma unroll
        for (int i = 0; i < kCh; ++i) {
            const int k0 = g * kGroup + (tid & 7) * 16;
            ar[s][i] = *reinterpret_cast<const u32x4*>(p.xq + opaque_u32(ap[i] + (k0 < K ? g * kGroup : 0)));
        }
    };
    auto store_a = [&](int g, auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
#pragma unroll
        for (int i = 0; i < kCh; ++i) {
            const int k0 = g * kGroup + (tid & 7) * 16;
            const u32x4 v = k0 < K ? ar[s][i] : u32x4{0u, 0u, 0u, 0u};
            *reinterpret_cast<u32x4*>(a_slot(g) + adst[i]) = v;
        }
    };

    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    auto row_frag = [&](int i, int g) __attribute__((always_inline)) {
        const uint8_t* A = a_slot(g) + (16 * i + c16) * kGroup;
        const u32x4 lo = *reinterpret_cast<const u32x4*>(A + ((q ^ (c16 & 7)) << 4));
        const u32x4 hi = *reinterpret_cast<const u32x4*>(A + (((4 + q) ^ (c16 & 7)) << 4));
        return v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
    };

    // one super-step: the E8M0 bytes of the lane's K block for its four steps are in sw, its
    // weights and rows in the ring
    int sw[NT];
    auto super = [&](int su, auto lastc) __attribute__((always_inline)) {
        constexpr bool last = decltype(lastc)::value;
        auto step = [&](auto sc) __attribute__((always_inline)) {
            constexpr int s = decltype(sc)::value;
            const int g = kF4Steps * su + s;
            if (last && g >= nst) return;                  // uniform over the work-group
            // The rows go out four steps ahead, before the step's weights (and kept there by the
            // barrier): the wait for the rows of step g + 1 below then leaves three steps of
            // weights in flight (loads return in order).
            issue_a(g + kF4Steps, sc);
            __builtin_amdgcn_sched_barrier(0);
            v8i wf[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const uint4 v = s_w[wave][j][wslot];
                wf[j] = v8i{(int)v.x, (int)v.y, (int)v.z, (int)v.w, 0, 0, 0, 0};
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                if (i >= nfl) break;                       // uniform
                const v8i af = row_frag(i, g);
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = f4_mfma<s>(wf[j], af, acc[i][j], sw[j]);
            }
            using Next = std::integral_constant<int, (s + 1) % kF4Steps>;
            issue_w(g + kF4Steps, sc);
            store_a(g + 1, Next{});
            store_w(Next{});
            if constexpr (!kOwnRows) lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
    };
    // The super-step's scales out of raw, as E8M0 bytes through LDS; blocks past K count as
    // 1.0. other and emin collect whether every scale so far of the lane's row was a normal
    // positive power of two.
    uint32_t other[NT];
    u16x2 emin[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        other[j] = 0;
        emin[j] = u16x2{0x1E, 0x1E};
    }
    const uint32_t selq = (uint32_t)(q | ((4 + q) << 8));
    auto take_scales = [&](int su) __attribute__((always_inline)) {
        const int past = std::min(std::max(4 * (kF4Steps * su + (lane & 3)) - (G - 4), 0), 4);   // leading halves to drop
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            uint64_t v = (uint64_t)raw[j].lo | ((uint64_t)raw[j].hi << 32);
            const uint64_t ones = (uint64_t)kF4OnesHalf2 | ((uint64_t)kF4OnesHalf2 << 32);
            if (past > 0) v = past == 4 ? ones : (v >> (16 * past)) | (ones << (64 - 16 * past));
            const uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
            other[j] |= (lo | hi) & 0x83FF83FFu;            // sign or fraction bits
            const uint32_t e0 = (lo >> 10) & 0x001F001Fu, e1 = (hi >> 10) & 0x001F001Fu;
            // exponent 0 (zero, subnormal) and 31 (inf, NaN) give 0 here
            emin[j] = __builtin_elementwise_min(emin[j], __builtin_bit_cast(u16x2, (e0 + 0x00010001u) & 0x001E001Eu));
            emin[j] = __builtin_elementwise_min(emin[j], __builtin_bit_cast(u16x2, (e1 + 0x00010001u) & 0x001E001Eu));
            // bytes of K blocks 0..3 of the lane's step; row r's sixteen bytes lie together
            reinterpret_cast<uint32_t*>(&s_s[wave][j][0])[lane] =
                __builtin_amdgcn_perm(e1 + 0x00700070u, e0 + 0x00700070u, 0x06040200u);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {                      // byte s of sw: block q of step s, row c16
            const uint4 t = s_s[wave][j][c16];
            sw[j] = (int)__builtin_amdgcn_perm(__builtin_amdgcn_perm(t.w, t.z, selq),
                                               __builtin_amdgcn_perm(t.y, t.x, selq), 0x05040100u);
        }
    };
    // bit r: weight row r of fragment j has a scale that the block-scaled form cannot take
    auto general_rows = [&](int j) __attribute__((always_inline)) {
        const uint64_t m = __ballot(other[j] != 0 || emin[j].x == 0 || emin[j].y == 0);
        return (uint32_t)(__ballot(((m >> (4 * c16)) & 15) != 0) & 0xFFFFu);
    };
    // The general form: one masked MFMA per group and the fold run += partial * scale, for
    // fragments J0 .. J0 + NJ - 1 into run. Each wave reads the rows itself, without LDS: some
    // waves of the work-group may be past their work. Every row fragment takes part, live or
    // not: with a uniform branch around each fragment's MFMAs the compiler moved the folds past
    // the branches, where it can leave out the wait between an MFMA and the next use of its
    // result's registers (tests/test_cpu_mfma_waits.py walks the built code for that; the ring's
    // branches guard MFMAs alone, whose results are read after its barriers).
    auto general_form = [&](auto j0c, auto njc, auto& run) __attribute__((always_inline)) {
        constexpr int J0 = decltype(j0c)::value, NJ = decltype(njc)::value;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) run[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        const uint8_t *rp[MT], *wr[NJ], *sr[NJ];
#pragma unroll
        for (int i = 0; i < MT; ++i) rp[i] = p.xq + (int64_t)src_of(16 * i + c16) * K + q * 16;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            wr[j] = we + (int64_t)wrow(J0 + j, c16) * (K / 2) + q * 16;
            sr[j] = se + (int64_t)wrow(J0 + j, c16) * G * 2;
        }
#pragma unroll 1
        for (int g = 0; g < nst; ++g) {
            const bool in = 4 * g + q < G;
            u32x4 w[NJ];
            int sb[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                w[j] = *reinterpret_cast<const u32x4*>(wr[j] + (in ? g * 64 : 0));
                sb[j] = *reinterpret_cast<const uint16_t*>(sr[j] + (in ? 2 * (4 * g + q) : 0));
            }
            const int k0 = g * kGroup + q * 16;
            v8i af[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                u32x4 lo = *reinterpret_cast<const u32x4*>(rp[i] + (k0 < K ? g * kGroup : 0));
                u32x4 hi = *reinterpret_cast<const u32x4*>(rp[i] + (k0 + 64 < K ? g * kGroup + 64 : 0));
                if (k0 >= K) lo = u32x4{0u, 0u, 0u, 0u};
                if (k0 + 64 >= K) hi = u32x4{0u, 0u, 0u, 0u};
                af[i] = v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
            }
#pragma unroll 1
            for (int sg = 0; sg < 4 && 4 * g + sg < G; ++sg) {
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const v8i wm = {q == sg ? (int)w[j].x : 0, q == sg ? (int)w[j].y : 0, q == sg ? (int)w[j].z : 0,
                                    q == sg ? (int)w[j].w : 0, 0, 0, 0, 0};
                    float f[4];                            // scales of weight rows 4 q .. 4 q + 3
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        f[r] = __half2float(__ushort_as_half((uint16_t)__shfl(sb[j], 16 * sg + 4 * q + r, 64)));
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        const v4f t = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                            wm, af[i], v4f{0.f, 0.f, 0.f, 0.f}, 4, 0, 0, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; ++r) run[i][j][r] = fmaf(t[r], f[r], run[i][j][r]);
                    }
                }
            }
        }
    };

    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    using S3 = std::integral_constant<int, 3>;
    issue_s(0);
    auto fill = [&](auto sc) __attribute__((always_inline)) {
        issue_a(decltype(sc)::value, sc);
        issue_w(decltype(sc)::value, sc);
        __builtin_amdgcn_sched_barrier(0);
    };
    fill(S0{});
    fill(S1{});
    fill(S2{});
    fill(S3{});
    store_a(0, S0{});
    store_w(S0{});
    if constexpr (!kOwnRows) lds_barrier();
    // where the first super-step already sends every column of the work-group to the general
    // form, the ring is left out
    take_scales(0);
    uint32_t every = 0xFFFFu;
#pragma unroll
    for (int j = 0; j < NT; ++j) every &= general_rows(j);
    if (__syncthreads_and(every == 0xFFFFu) == 0) {
        for (int su = 0; su + 1 < nsuper; ++su) {
            issue_s(su + 1);
            super(su, std::false_type{});
            take_scales(su + 1);
        }
        super(nsuper - 1, std::true_type{});
        // the form is chosen per column, so a column's result does not depend on its tile
        auto replace = [&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            if constexpr (j < NT) {
                const uint32_t rows = general_rows(j);
                if (rows == 0) return;
                v4f run[MT][1];
                general_form(jc, std::integral_constant<int, 1>{}, run);
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if ((rows >> (4 * q + r)) & 1) acc[i][j][r] = run[i][0][r];
            }
        };
        replace(S0{});
        replace(S1{});
        replace(S2{});
        replace(S3{});
    } else {
        // two fragments at a time where four would not fit the registers
        if constexpr (MT == 4) {
            v4f run[MT][2];
            auto half = [&](auto j0c) __attribute__((always_inline)) {
                general_form(j0c, std::integral_constant<int, 2>{}, run);
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    acc[i][decltype(j0c)::value] = run[i][0];
                    acc[i][decltype(j0c)::value + 1] = run[i][1];
                }
            };
            half(S0{});
            half(S2{});
        } else {
            general_form(S0{}, std::integral_constant<int, NT>{}, acc);
        }
    }

    // ---- epilogue: lane (q, c16) holds row 16 i + c16, columns 4 q .. 4 q + 3 ----
    const __half* be = p.bias ? p.bias + (int64_t)e * p.N : nullptr;
    const bool vec = p.N % 8 == 0;      // whole four-column pieces at aligned addresses
    constexpr bool kHalves = EPI == Epi::kHalf || kSilu || EPI == Epi::kSwigluHalf;
    __half bv[kHalves ? NT : 1][4];     // the lane's bias values (0 without a bias; unused rows of edge columns)
    if constexpr (kHalves) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int c0 = out0 + 16 * (kSilu ? j % kOutFrags : j) + 4 * q;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                bv[j][r] = be == nullptr ? __float2half(0.f)
                                         : be[std::min(c0 + r, ncols - 1) + (kSilu && j >= kOutFrags ? ncols : 0)];
        }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = 16 * i + c16;
        const int sl = __shfl(slot, m, 64), sr = __shfl(src, m, 64);
        if (sr < 0) continue;
        const float a = p.asc[sr];
        const int64_t orow = row0 + m;
#pragma unroll
        for (int j = 0; j < kOutFrags; ++j) {
            const int col = out0 + 16 * j + 4 * q;
            if (col >= ncols) continue;
            if constexpr (EPI == Epi::kScatter || EPI == Epi::kSlotF32) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (col + r >= ncols) break;
                    if constexpr (EPI == Epi::kScatter)
                        atomicAdd(reinterpret_cast<float*>(p.out) + (int64_t)(sl / p.out_top_k) * p.N + col + r,
                                  p.tw[sl] * acc[i][j][r] * a);
                    else
                        reinterpret_cast<float*>(p.out)[(int64_t)sl * p.N + col + r] = acc[i][j][r] * a;
                }
            } else {
                __half v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    v[r] = __float2half(as_f32(acc[i][j][r] * a));
                    if (be != nullptr) v[r] = __hadd(v[r], bv[j][r]);
                }
                if constexpr (EPI == Epi::kSwigluHalf) {
                    __half* o = reinterpret_cast<__half*>(p.out) + orow * (p.N / 2) + col / 2;
                    const __half h0 = swigluoai_h(v[0], v[1], p.alpha, p.limit);
                    const __half h1 = swigluoai_h(v[2], v[3], p.alpha, p.limit);
                    if (vec) {
                        *reinterpret_cast<__half2*>(o) = __halves2half2(h0, h1);
                    } else {
                        o[0] = h0;
                        if (col + 2 < ncols) o[1] = h1;
                    }
                    continue;
                }
                if constexpr (kSilu) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        __half u = __float2half(as_f32(acc[i][j + (kSilu ? kOutFrags : 0)][r] * a));
                        if (be != nullptr) u = __hadd(u, bv[j + (kSilu ? kOutFrags : 0)][r]);
                        v[r] = silu_mul_h(v[r], u);
                    }
                }
                __half* o = reinterpret_cast<__half*>(p.out) + orow * ncols + col;
                if (vec && (!kSilu || ncols % 4 == 0)) {
                    const __half2 v01 = __halves2half2(v[0], v[1]), v23 = __halves2half2(v[2], v[3]);
                    *reinterpret_cast<uint2*>(o) = make_uint2(__builtin_bit_cast(uint32_t, v01),
                                                              __builtin_bit_cast(uint32_t, v23));
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (col + r < ncols) o[r] = v[r];
                }
            }
        }
    }
}

template <Epi EPI, int MT, int NT>
int launch_fp4_t(const Params& p, hipStream_t s) {
    constexpr int cols = 4 * 16 * (EPI == Epi::kSiluHalf ? NT / 2 : NT);
    const int ncols = EPI == Epi::kSiluHalf ? p.N / 2 : p.N;
    const int ntiles = (ncols + cols - 1) / cols;
    const int nblocks = (int)((p.P + 16 * MT - 1) / (16 * MT));
    const int64_t items = (int64_t)nblocks * ntiles;
    const unsigned grid = (unsigned)((items + kF4Xcds - 1) / kF4Xcds * kF4Xcds);
    launch_kernel(&fp4_tiles_kernel<EPI, MT, NT>, dim3(grid), dim3(256), 0, s, p, nblocks, ntiles);
    return check_launch("fp4_tiles_kernel");
}

template <Epi EPI>
int launch_fp4_e(const Params& p, hipStream_t s) {
    // the tile height divides block_m, so a tile lies in one expert's block
    if (p.block_m % 64 == 0) return launch_fp4_t<EPI, 4, 4>(p, s);
    if (p.block_m % 32 == 0) return launch_fp4_t<EPI, 2, 4>(p, s);
    return launch_fp4_t<EPI, 1, 2>(p, s);
}

}  // namespace

bool fp4_tiles_supported(int64_t x_rows, int64_t K, int64_t N, int64_t group_size, bool e2m1) {
    return e2m1 && group_size == kF4Group && K % kF4Group == 0 && K >= 4 * kF4Group &&
           N * (K / 2) < (int64_t)1 << 31 && x_rows * K < (int64_t)1 << 31;
}

int launch_grouped_fp4(const GroupedArgs& a, hipStream_t s) {
    const Params p = make_params(a);
    if (p.P == 0) return W4A8_OK;
    if (!fp4_tiles_supported(a.x_rows, a.K, a.N, a.group_size, a.e2m1) || a.w_frag || p.xq == nullptr ||
        p.asc == nullptr || a.block_m % 16 != 0) {
        set_error("fp4 tiles: need op-layout E2M1 weights with groups of 32, K >= 128, quantised "
                  "rows, expert slices and rows below 2 GiB and block_m a multiple of 16");
        return W4A8_ERR_INVALID;
    }
    switch (a.epi) {
        case Epi::kHalf: return launch_fp4_e<Epi::kHalf>(p, s);
        case Epi::kSiluHalf: return launch_fp4_e<Epi::kSiluHalf>(p, s);
        case Epi::kScatter: return launch_fp4_e<Epi::kScatter>(p, s);
        case Epi::kSlotF32: return launch_fp4_e<Epi::kSlotF32>(p, s);
        case Epi::kSwigluHalf: return launch_fp4_e<Epi::kSwigluHalf>(p, s);
    }
    return W4A8_ERR_INVALID;
}

}  // namespace w4a8
