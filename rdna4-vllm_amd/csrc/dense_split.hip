// Dense W4A8 GEMM for some tens of rows (gfx950 fp8 MFMA), K split over the waves of a
// work-group.
//
// Replaces the reference's small-M dense kernels (dense_kernel.hip's split-K and n-split forms
// behind mmq_fp8_gemm, vllm_adapter.py:296-324) on op-layout weights (N, K/8), group 128, any K.
// A work-group owns 16 MT rows x 16 columns; its eight waves take an eighth of the K groups
// each, so a dense GEMM whose output has few tiles still keeps every CU streaming weights, and
// no wave waits for another until the partial sums meet in LDS at the end (added in wave order).
// Rows come quantised (act_quant_kernel). Per group the weights are decoded to e4m3(n - z) (raw
// nibbles lose precision, see wide_tiles.hip), then one 16x16x128 MFMA a block and the fp16 scale
// fold. Two column fragments a work-group measured slower at every size (half the
// work-groups; registers): (4096, 12288) M = 64 53 -> 121 us on raw nibbles.
#include <algorithm>
#include <type_traits>

#include "grouped_params.h"

namespace w4a8 {
namespace {

constexpr int kDsWaves = 8;
constexpr int NT = 1;                       // column fragments of a work-group

struct SplitParams {
    const uint8_t* xq;     // (M, K) e4m3, k8-interleaved
    const float* asc;      // (M,)
    const int32_t* w;      // (N, K/8) op layout
    const __half* s;       // (N, G)
    const int32_t* z;      // (N/8, G) or null (zero point 8)
    __half* out;           // (M, N)
    int M, N, K, G;
};

// ZP: weights with zero-points (else the zero point is 8)
template <int MT, bool ZP>
__global__ void __launch_bounds__(64 * kDsWaves, 2) dense_split_kernel(SplitParams p) {
    __shared__ v4f s_part[kDsWaves][MT * NT][64];
    __shared__ uint4 s_lut[ZP ? 16 : 1];        // e4m3(n - z) tables
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, c16 = lane & 15;
    const int row0 = blockIdx.y * 16 * MT, col0 = blockIdx.x * 16 * NT;
    const int K = p.K, G = p.G;
    const int gb = G * wave / kDsWaves, ge = G * (wave + 1) / kDsWaves;

    // lane (q, c16): row / column c16 of a fragment, k in [128 g + 32 q, +32). Rows and columns
    // past the end read the last one (not stored).
    uint32_t aoff[MT], woff[NT], soff[NT], zoff[NT];
    int zsh[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
        aoff[i] = (uint32_t)min(row0 + 16 * i + c16, p.M - 1) * (uint32_t)K + (uint32_t)q * 32u;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int n = min(col0 + 16 * j + c16, p.N - 1);
        woff[j] = (uint32_t)n * (uint32_t)(K / 2) + (uint32_t)q * 16u;
        soff[j] = (uint32_t)n * (uint32_t)G * 2u;
        zoff[j] = (uint32_t)(n >> 3) * (uint32_t)G * 4u;
        zsh[j] = 4 * (n & 7);
    }
    const uint8_t* wb = reinterpret_cast<const uint8_t*>(p.w);
    const uint8_t* sb = reinterpret_cast<const uint8_t*>(p.s);
    const uint8_t* zb = reinterpret_cast<const uint8_t*>(p.z);

    constexpr int D = 4;                 // weight groups in flight
    constexpr int DA = MT > 2 ? 2 : 4;   // row groups in flight (their registers grow with MT)
    u32x4 bw[D][NT], ar[DA][MT][2];
    uint32_t sv[D][NT], zv[ZP ? D : 1][NT];
    auto issue_b = [&](int g, auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
        const uint32_t gg = (uint32_t)min(g, G - 1);         // past the end: never used
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            bw[s][j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wb + opaque_u32(woff[j] + gg * 64u)));
            sv[s][j] = *reinterpret_cast<const uint16_t*>(sb + opaque_u32(soff[j] + gg * 2u));
            if constexpr (ZP) zv[s][j] = *reinterpret_cast<const uint32_t*>(zb + opaque_u32(zoff[j] + gg * 4u));
        }
    };
    auto issue_a = [&](int g, auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value % DA;
        const uint32_t gg = (uint32_t)min(g, G - 1) * (uint32_t)kGroup;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const uint8_t* a = p.xq + opaque_u32(aoff[i] + gg);
            ar[s][i][0] = *reinterpret_cast<const u32x4*>(a);
            ar[s][i][1] = *reinterpret_cast<const u32x4*>(a + 16);
        }
    };
    v4f run[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) run[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    const DecodeMasks masks = decode_masks();
    const uint4 t8 = load_table(8);
    if (ZP && threadIdx.x < 16) s_lut[threadIdx.x] = load_table(threadIdx.x);
    auto step = [&](int g, auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value, sa_ = s % DA;
        v8i bf[NT];
        float sf[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const uint4 t = ZP ? s_lut[(zv[ZP ? s : 0][j] >> zsh[j]) & 0xFu] : t8;
            bf[j] = decode_frag(bw[s][j], t, masks);
            sf[j] = __half2float(__ushort_as_half((unsigned short)sv[s][j]));
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const u32x4 lo = ar[sa_][i][0], hi = ar[sa_][i][1];
            const v8i af = {(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const v4f acc = mfma_16x16x128(af, bf[j], v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                for (int r = 0; r < 4; ++r) run[i][j][r] = fmaf(acc[r], sf[j], run[i][j][r]);
            }
        }
        issue_a(g + DA, sc);
        issue_b(g + D, sc);
        __builtin_amdgcn_sched_barrier(0);
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    using S3 = std::integral_constant<int, 3>;
    auto fill = [&](auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
        if constexpr (s < DA) issue_a(gb + s, sc);
        issue_b(gb + s, sc);
        __builtin_amdgcn_sched_barrier(0);
    };
    fill(S0{});
    fill(S1{});
    fill(S2{});
    fill(S3{});
    if constexpr (ZP) lds_barrier();   // the tables are written
    const int nq = (ge - gb) / D, rem = (ge - gb) % D;
    int g = gb;
    for (int it = 0; it < nq; ++it, g += D) {
        step(g, S0{});
        step(g + 1, S1{});
        step(g + 2, S2{});
        step(g + 3, S3{});
    }
    if (rem > 0) step(g, S0{});
    if (rem > 1) step(g + 1, S1{});
    if (rem > 2) step(g + 2, S2{});

#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) s_part[wave][i * NT + j][lane] = run[i][j];
    __syncthreads();
    // wave w sums and stores blocks w, w + 8, ...: lane (q, c16) rows 4 q .. 4 q + 3, column c16
    for (int b = wave; b < MT * NT; b += kDsWaves) {
        v4f sum = s_part[0][b][lane];
#pragma unroll
        for (int w = 1; w < kDsWaves; ++w) {
            const v4f v = s_part[w][b][lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[r] += v[r];
        }
        const int n = col0 + 16 * (b % NT) + c16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = row0 + 16 * (b / NT) + 4 * q + r;
            if (m < p.M && n < p.N)
                p.out[(int64_t)m * p.N + n] = __float2half(as_f32(sum[r] * p.asc[m]));
        }
    }
}

template <int MT>
int launch_split_t(const SplitParams& p, hipStream_t s) {
    const dim3 grid((unsigned)((p.N + 16 * NT - 1) / (16 * NT)), (unsigned)((p.M + 16 * MT - 1) / (16 * MT)));
    if (p.z) dense_split_kernel<MT, true><<<grid, dim3(64 * kDsWaves), 0, s>>>(p);
    else dense_split_kernel<MT, false><<<grid, dim3(64 * kDsWaves), 0, s>>>(p);
    return check_launch("dense_split_kernel");
}

}  // namespace

// While its 64-row x 16-column work-groups fit the CUs in one round and either the rows are few
// or K is long: the wide tiles then have too few work-groups, each walking all of K (us, this /
// 32 x 64 tiles: (N, K) = (4096, 12288) M = 17 23 / 52, M = 64 40 / 53; (2048, 6144) M = 17
// 14 / 27, M = 128 25 / 29).
bool dense_split_leads(int64_t M, int64_t N, int64_t K) {
    const int64_t wgs = (N + 15) / 16 * ((M + 63) / 64);
    return wgs <= device_cu_count() && (M <= 48 || K > 32 * kGroup);
}

int launch_dense_split(const GroupedArgs& a, hipStream_t s) {
    if (a.P == 0) return W4A8_OK;
    SplitParams p;
    p.xq = a.x_fp8;
    p.asc = a.act_scales;
    p.w = a.w;
    p.s = reinterpret_cast<const __half*>(a.scales);
    p.z = a.zeros;
    p.out = static_cast<__half*>(a.out);
    p.M = (int)a.P;
    p.N = (int)a.N;
    p.K = (int)a.K;
    p.G = (int)(a.K / kGroup);
    if (p.M <= 16) return launch_split_t<1>(p, s);
    if (p.M <= 32) return launch_split_t<2>(p, s);
    if (p.M <= 48) return launch_split_t<3>(p, s);
    return launch_split_t<4>(p, s);
}

}  // namespace w4a8
