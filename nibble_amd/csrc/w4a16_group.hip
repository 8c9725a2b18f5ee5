// Group sizes 32 and 64 at M = 1..8 on gfx950: the GEMV / small-batch kernel
// of layers whose scales are finer than 128 weights.
//
// Bound: the weight stream (HBM), as the ring kernel (w4a16_pair_ring.h). The
// scalar kernel these layers ran on before reads one byte a lane and decodes
// every weight with ten integer and conversion instructions.
//
// Operands (v_mfma_f32_16x16x32_f16, lane l = 16 q + c). Weights come as in
// the ring kernel: B column c is weight row c & 7 of an 8-row block, 128-weight
// run 2 p + (c >> 3) of run pair p, and lane q loads bytes 16 q .. of the run:
// 8 rows x 128 contiguous bytes an instruction. Those 16 bytes are the 32
// weights of ONE 32-weight chunk, and a matrix instruction adds over q, so as
// loaded it would add weights of different scales. Four swaps of 16 or 32
// lanes (v_permlane16_swap / v_permlane32_swap) transpose the 4 x 4 words of
// (q, word): register t of lane q is then word q of chunk t, step t covers
// chunk t alone (k = 32 t + 8 q .. + 7 of the run), and its fp32 sum takes
// the chunk's scale: one FMA per chunk and accumulator (G = 64 chains two
// steps before it). Codes are exact fp16 integers, so a product differs from
// the fp32 code * scale * x of the scalar kernel only in the order of its
// fp32 sums; outputs with an infinite scale are put right at the end.
//
// A row c holds activation row c & 7 of run 2 p + (c >> 3): D rows 0..7 x
// columns 0..7 and rows 8..15 x columns 8..15 are the wanted products, added
// across the halves at the end (lanes l and l + 40).
//
// Workgroup = SK wavefronts splitting the run pairs x SN on 8-row blocks; a
// wavefront keeps D loads of 1 KiB in flight. The activation rows are staged
// in LDS in unpack8's pair order; runs past K are staged as zeros and their
// scales taken as 0.
#include "w4a16_hip.h"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "w4a16_device.h"

namespace w4a16 {

constexpr int kGroupRun = 272;   // bytes of one staged run: 256 + 16, so that two runs fall on distinct bank slots

// bytes between staged activation rows: 32 mod 256, so the 16 units that one
// fragment read touches (8 rows, 2 runs) fall on distinct bank slots
__host__ __device__ constexpr int group_row_stride(int runs) { return (runs * kGroupRun + 255) / 256 * 256 + 32; }

__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {   // upper half of a <-> lower half of b
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {   // odd rows of 16 lanes of a <-> even rows of b
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// GS = group size (32 or 64), MS = accumulator rows a lane keeps (1 for M = 1, else 4)
template <int GS, int MS, int SK, int D>
__global__ void __launch_bounds__(512)
gemv_group(const f16* __restrict__ x, const uint8_t* __restrict__ w, const f16* __restrict__ scales,
           f16* __restrict__ out, int M, int N, int K, int SN) {
    static_assert(GS == 32 || GS == 64, "group sizes 32 and 64");
    constexpr int SC = 64 / GS;   // 32-bit words of scales per run
    extern __shared__ __align__(16) uint8_t smem[];
    const int runs = K >> 7;
    const int pairs = (runs + 1) >> 1;
    const int rs = group_row_stride(2 * pairs);
    const int threads = 64 * SK * SN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int c = lane & 15, q = lane >> 4;
    const int kw = wave % SK, nb = wave / SK;
    const int n0 = (blockIdx.x * SN + nb) * 8;
    const int per = (pairs + SK - 1) / SK;   // run pairs per wavefront
    const int p0 = kw * per;
    const int mine = n0 < N ? max(0, min(per, pairs - p0)) : 0;

    // the wavefront's loads: 32-bit byte offsets (the host checks the buffers)
    const uint32_t row = (uint32_t)min(n0 + (c & 7), N - 1);
    const uint32_t wbase = row * (uint32_t)(K >> 1) + 16u * q;
    const uint32_t sbase = row * (uint32_t)runs * (4u * SC);   // bytes of scales per run: 4 SC
    struct Pair {
        u32x4 w;
        uint32_t s[SC];
    };
    auto load = [&](Pair& b, int j) {
        const uint32_t run = (uint32_t)min(2 * (p0 + j) + (c >> 3), runs - 1);
        const uint32_t* sp =
            reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint8_t*>(scales) + (sbase + run * (4u * SC)));
#pragma unroll
        for (int i = 0; i < SC; ++i) b.s[i] = sp[i];
        b.w = load_stream(reinterpret_cast<const u32x4*>(w + (wbase + run * 64u)));
    };

    // 1. the first activation units, then the first D weight loads: all in flight before the first wait
    constexpr int A = 4;
    const int units = 2 * pairs * 16;   // 16-byte units staged per row, the padding run included
    const int total = M * units;
    u32x4 a[A];
    auto unit_load = [&](int i) {
        const int m = MS == 1 ? 0 : i / units, u = i - m * units;
        return *reinterpret_cast<const u32x4*>(x + (size_t)m * K + 8 * min(u, runs * 16 - 1));
    };
    auto unit_put = [&](int i, const u32x4& v) {
        const int m = MS == 1 ? 0 : i / units, u = i - m * units;
        if (i < total)
            *reinterpret_cast<u32x4*>(smem + m * rs + (u >> 4) * kGroupRun + (u & 15) * 16) =
                u < runs * 16 ? permute8(v) : (u32x4){0u, 0u, 0u, 0u};
    };
#pragma unroll
    for (int i = 0; i < A; ++i) a[i] = unit_load(min((int)threadIdx.x + i * threads, total - 1));
    Pair ring[D];
#pragma unroll
    for (int d = 0; d < D; ++d) load(ring[d], min(d, max(mine - 1, 0)));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < A; ++i) unit_put(threadIdx.x + i * threads, a[i]);
    for (int i0 = threadIdx.x + A * threads; i0 < total; i0 += A * threads) {
#pragma unroll
        for (int i = 0; i < A; ++i) a[i] = unit_load(min(i0 + i * threads, total - 1));
#pragma unroll
        for (int i = 0; i < A; ++i) unit_put(i0 + i * threads, a[i]);
    }
    __syncthreads();

    // 2. the run pairs of this wavefront
    const uint8_t* arow = smem + min(c & 7, M - 1) * rs + (c >> 3) * kGroupRun + 16 * q;
    float acc[MS];
#pragma unroll
    for (int i = 0; i < MS; ++i) acc[i] = 0.0f;
    // The chunk sums of a pair take their scales while the next pair's matrix
    // instructions run: a pair's sums are ready some 30 cycles after it issued.
    constexpr int SUMS = 128 / GS;   // per run
    f32x4 sums[SUMS];
    uint32_t pend[SC];
#pragma unroll
    for (int i = 0; i < SUMS; ++i) sums[i] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < SC; ++i) pend[i] = 0;
    auto scale_sums = [&]() {
#pragma unroll
        for (int g = 0; g < SUMS; ++g) {
            const float s = (float)__builtin_bit_cast(f16, (uint16_t)(pend[g >> 1] >> (16 * (g & 1))));
#pragma unroll
            for (int i = 0; i < MS; ++i) acc[i] = __builtin_fmaf(sums[g][i], s, acc[i]);
        }
    };
    auto compute = [&](const Pair& b, int j) {
        const int p = p0 + j;
        f16x8 av[4], bv[4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
            av[t] = __builtin_bit_cast(f16x8, *reinterpret_cast<const u32x4*>(arow + 2 * p * kGroupRun + 64 * t));
        uint32_t t0 = b.w[0], t1 = b.w[1], t2 = b.w[2], t3 = b.w[3];
        swap32(t0, t2);
        swap32(t1, t3);
        swap16(t0, t1);
        swap16(t2, t3);
        const uint32_t word[4] = {t0, t1, t2, t3};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const Codes8 cw = unpack8(word[t]);
            bv[t] = __builtin_bit_cast(
                f16x8, (u32x4){as_u32(cw.p[0]), as_u32(cw.p[1]), as_u32(cw.p[2]), as_u32(cw.p[3])});
        }
        f32x4 now[SUMS];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int g = t * SUMS / 4;
            const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
            now[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[t], bv[t], t % (4 / SUMS) == 0 ? zero : now[g], 0, 0, 0);
        }
        scale_sums();
        const bool live = 2 * p + (c >> 3) < runs;
#pragma unroll
        for (int i = 0; i < SC; ++i) pend[i] = live ? b.s[i] : 0u;
#pragma unroll
        for (int g = 0; g < SUMS; ++g) sums[g] = now[g];
    };
    int j = 0;
    for (; j + 2 * D <= mine; j += D) {   // full rounds: every slot is refilled with a pair that exists
#pragma unroll
        for (int d = 0; d < D; ++d) {
            compute(ring[d], j + d);
            load(ring[d], j + D + d);
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {   // the last D .. 2 D - 1 pairs (fewer where the wavefront has fewer than D)
        if (j + d < mine) compute(ring[d], j + d);
        if (j + D + d < mine) load(ring[d], j + D + d);
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (j + D + d < mine) compute(ring[d], j + D + d);
    scale_sums();

    // 3. the two run halves of an output, then the SK partial sums in order
    float sum[MS];
#pragma unroll
    for (int i = 0; i < MS; ++i) sum[i] = acc[i] + __shfl(acc[i], (lane + 40) & 63);
    const bool holds = q < 2 && c < 8 && 4 * q < M;   // rows 4 q .. of column c (MS = 1: row 0)
    if (SK > 1) {
        float* red = reinterpret_cast<float*>(smem + M * rs);   // [waves][MS][16]
        const int slot = q * 8 + c;   // the 16 lanes that hold outputs
        if (holds)
#pragma unroll
            for (int i = 0; i < MS; ++i) red[(wave * MS + i) * 16 + slot] = sum[i];
        __syncthreads();
        if (kw != 0) return;
        if (holds)
            for (int k = 1; k < SK; ++k)
#pragma unroll
                for (int i = 0; i < MS; ++i) sum[i] += red[((wave + k) * MS + i) * 16 + slot];
    }
    const int n = n0 + c;
    bool infinite = false;
    if (holds && n < N)
#pragma unroll
        for (int i = 0; i < MS; ++i)
            if (4 * q + i < M) {
                store_through(out + (size_t)(4 * q + i) * N + n, (f16)sum[i]);
                infinite |= __builtin_isinf(sum[i]);
            }

    // 4. An infinite scale (after the stores, so that no other output waits for
    // this): a code or activation of 0 makes the output NaN, and so do products
    // of both signs, where the exact sum of the group times the scale is an
    // infinity. Such groups are added once more, weight by weight as the scalar
    // kernel does: their infinity stays or becomes NaN. The test costs 0.4% of a
    // call in the mean over K x N 128 x 8 .. 8192 x 28672 (4096 x 4096, G = 64,
    // M = 1: 4.85 us against 4.83).
    if (__ballot(infinite) == 0) return;
    const int groups = K / GS;
    uint32_t rows = 0;   // of the block, those with an infinite scale
#pragma unroll 1
    for (int r = 0; r < min(8, N - n0); ++r) {
        bool found = false;
        for (int g = lane; g < groups; g += 64) found |= __builtin_isinf((float)scales[(size_t)(n0 + r) * groups + g]);
        if (__ballot(found) != 0) rows |= 1u << r;
    }
    if (!infinite || !(rows >> c & 1)) return;
#pragma unroll
    for (int i = 0; i < MS; ++i) {
        if (4 * q + i >= M || !__builtin_isinf(sum[i])) continue;
        const f16* xr = x + (size_t)(4 * q + i) * K;
#pragma unroll 1
        for (int k = 0; k < K; ++k) {
            const float s = (float)scales[(size_t)n * groups + k / GS];
            const int byte = w[((size_t)n * K + k) >> 1];
            const int code = (((k & 1 ? byte >> 4 : byte) & 15) ^ 8) - 8;
            if (__builtin_isinf(s)) sum[i] = __builtin_fmaf((float)xr[k], (float)code * s, sum[i]);
        }
        store_through(out + (size_t)(4 * q + i) * N + n, (f16)sum[i]);
    }
}

using GroupKern = void (*)(const f16*, const uint8_t*, const f16*, f16*, int, int, int, int);

template <int GS, int MS, int SK>
GroupKern pick_depth(int depth) {
    switch (depth) {
        case 1: return gemv_group<GS, MS, SK, 1>;
        case 2: return gemv_group<GS, MS, SK, 2>;
        case 4: return gemv_group<GS, MS, SK, 4>;
    }
    return nullptr;
}

template <int GS, int MS>
GroupKern pick_group(int sk, int depth) {
    switch (sk) {
        case 1: return pick_depth<GS, MS, 1>(depth);
        case 2: return pick_depth<GS, MS, 2>(depth);
        case 4: return pick_depth<GS, MS, 4>(depth);
        case 8: return pick_depth<GS, MS, 8>(depth);
    }
    return nullptr;
}

}  // namespace w4a16

namespace w4a16_internal {

int ensure_lds(const void* kernel, int bytes);             // w4a16_hip.hip
void set_last_error(const std::string& message);           // w4a16_hip.hip

namespace {
constexpr int64_t kLds = 160 * 1024;
int64_t group_red_bytes(int64_t rows, int waves) { return (int64_t)waves * (rows == 1 ? 1 : 4) * 64; }
int64_t group_lds_bytes(int64_t rows, int64_t K, int waves) {
    return rows * w4a16::group_row_stride((int)(2 * ((K / 128 + 1) / 2))) + group_red_bytes(rows, waves);
}
}  // namespace

// Whether gemv_group takes a layer: group size 32 or 64, whole 128-weight
// runs, one staged activation row within LDS, 32-bit offsets, and scales of a
// run aligned to their 8 or 4 bytes.
bool group_fits(int64_t M, int64_t N, int64_t K, int64_t G, const void* scales) {
    if ((G != 32 && G != 64) || M < 1 || M > 8 || N < 1 || K < 128 || K % 128 != 0 || K > 65536) return false;
    if (reinterpret_cast<uintptr_t>(scales) % (G == 32 ? 8 : 4) != 0) return false;
    return N * (K / 2) < ((int64_t)1 << 32) && group_lds_bytes(1, K, 8) <= kLds;
}

// Whether (wavefronts on K, wavefronts on blocks, loads in flight) is a shape gemv_group is built for.
bool group_shape(int sk, int sn, int depth) {
    const auto of = [](int v, int top) { return v >= 1 && v <= top && (v & (v - 1)) == 0; };
    return of(sk, 8) && of(depth, 4) && sn >= 1 && sn <= 8 && sk * sn <= 8;
}

// Launch shape, from a sweep of (SK, SN, D) over 16 layers (graph timing,
// rotated weights; us of the shape taken against the next kind). M = 1: the
// staged row is small, so one 8-row block a workgroup, 8 wavefronts on K (4096
// x 4096 4.64 against 4.76 with 4; 14336 x 4096 9.7 against 11.1), 4 from N =
// 5120 on (4096 x 14336 8.3 against 9.3). M >= 2: wider workgroups share the
// staging: 4 wavefronts on K x 2 blocks from N = 4096 (4096 x 4096 at M = 8
// 6.8 against 7.9 for 8 x 1), 2 x 4 on wide layers of short rows (4096 x 14336
// at M = 4 10.9 against 12.7), 8 x 1 on narrow ones (5632 x 2048 7.6 against
// 8.5). One load in flight a wavefront is enough while other workgroups share
// the CU; 2 where a wavefront has more than five pairs or stages many rows. 4
// runs through the tuned entry point only: it loses on rows of up to 4096
// weights (4096 x 4096, G = 64, M = 1: 6.7 against 5.1) and on most of 14336,
// and would win on rows of 28672 (x 8192: 30.4 against 37.2).
void group_plan(int64_t M, int64_t N, int64_t K, int* sk, int* sn, int* depth) {
    const int64_t pairs = (K / 128 + 1) / 2;
    int k = M == 1 ? (N >= 5120 ? 4 : 8) : N >= 8192 && K <= 4096 ? 2 : N >= 4096 ? 4 : 8;
    *sn = M == 1 || N < 4096 ? 1 : 8 / k;
    while (k > pairs) k /= 2;
    const int64_t per = (pairs + k - 1) / k;
    *sk = k;
    *depth = per >= (M == 1 || k == 8 ? 6 : 2) ? 2 : 1;
}

int launch_group(int G, int sk, int sn, int depth, int M, const void* x, const uint8_t* w, const void* s, void* o,
                 int N, int K, hipStream_t stream) {
    using namespace w4a16;
    if (!group_fits(M, N, K, G, s) || !group_shape(sk, sn, depth)) {
        set_last_error("group kernel: group size 32 or 64, M <= 8, K a multiple of 128, splits 1, 2, 4 or 8, unroll 1, 2 "
                       "or 4, at most 8 wavefronts");
        return W4A16_ERR_CONFIG;
    }
    // rows past what LDS holds go in further launches of about equal size (the weights are read again)
    int per = M;
    while (per > 1 && group_lds_bytes(per, K, sk * sn) > kLds) --per;
    const int parts = (M + per - 1) / per;
    for (int i = 0, m0 = 0; i < parts; ++i) {
        const int rows = (M - m0 + parts - i - 1) / (parts - i);
        const GroupKern kern = G == 32 ? (rows == 1 ? pick_group<32, 1>(sk, depth) : pick_group<32, 4>(sk, depth))
                                       : (rows == 1 ? pick_group<64, 1>(sk, depth) : pick_group<64, 4>(sk, depth));
        const int lds = (int)group_lds_bytes(rows, K, sk * sn);
        const int rc = ensure_lds(reinterpret_cast<const void*>(kern), lds);
        if (rc != W4A16_OK) return rc;
        const int64_t blocks = (N + 7) / 8;
        hipLaunchKernelGGL(kern, dim3((unsigned)((blocks + sn - 1) / sn)), dim3(64 * sk * sn), lds, stream,
                           static_cast<const f16*>(x) + (size_t)m0 * K, w, static_cast<const f16*>(s),
                           static_cast<f16*>(o) + (size_t)m0 * N, rows, N, K, sn);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            set_last_error(std::string("kernel launch failed: ") + hipGetErrorString(e));
            return W4A16_ERR_LAUNCH;
        }
        m0 += rows;
    }
    return W4A16_OK;
}

}  // namespace w4a16_internal
