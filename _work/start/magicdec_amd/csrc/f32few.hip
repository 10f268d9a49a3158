// 32-bit linear of a step's few rows (gfx950):  out[M][N] = x[M][K] . W[N][K]^T, all float32, row-major, M <= 16, and
// N <= 4096 (f32_few_kernel) or a shallow K (f32_wide_kernel)
//
// replaces: the library products of 32-bit steps of the layered designs (and of recorded traces) over narrow weights.
//
// What bounds it: the weight's bytes, and what a CU keeps in flight of them.  A workgroup of eight wavefronts takes 16 or 8 rows of W and all
// of K, an eighth a wavefront: independent pipelines with eight KB of W in flight each, straight from memory into the order of
// v_mfma_f32_16x16x4, no barrier, no K split over workgroups to combine.  x goes through LDS: as fragments from memory it would be as many
// bytes in flight as W.  The wavefronts' partial tiles are added in their order, so that a row's bits do not depend on the rows beside it.
// Six rows, us, library / here: 3 072 x 2 048 12.6 / 9.9, 2 048 x 2 048 12.1 / 8.0, 2 048 x 8 192 23.5 / 19.4 (one row 16.9: 4.0 TB/s),
// 2 048 x 5 632 17.9 / 15.6, 1 536 x 1 536 9.6 / 6.9; error against 64 bits half of the library's.  Wider weights are level that
// way (8 192 x 2 048 17.9 / 18.2, 32 000 x 2 048 61.4 / 61.6: each workgroup's x).
#include "md_common.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int kNW = 8;                             // wavefronts, K slices

struct FewParams {
    const float* x;
    const float* w;
    float* out;
    int64_t ldx, ldo;
    int M, N, K;
};

// COLS: 16, or 8: rows of W a workgroup (twice the workgroups where 16 leave CUs idle; a fragment then holds eight rows twice, with other k,
// and the product with the other half's x is thrown away).  ROWS: staged rows of x, 4, 8 or 16.
// The eight loads of W in flight are one chunk of x: a wait for x is one for all that was asked for before it, and behind it stand the
// loads of a whole chunk (two chunks in the ring: 2 048 x 8 192 24.2 us).
template <int COLS, int ROWS>
__global__ __launch_bounds__(64 * kNW, COLS == 8 ? 2 : 4) void f32_few_kernel(const FewParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    constexpr int L = COLS / 8, S = 8 / L;                      // loads a step of 32 k, steps a chunk
    constexpr int kPitch = S * 128 + 16, kWave = 16 * kPitch, LPR = S * 8, RPI = 64 / LPR, AI = ROWS / RPI;     // lanes a row, rows an instruction
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, q = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * COLS, steps = p.K / (32 * kNW), k0 = wave * steps * 32;
    unsigned char* image = lds + wave * kWave;
    // A load: 8 rows of 128 bytes, whole lines.  Lane (j, q) has row j & 7 of it, k 8 q + 4 (j >> 3) .. + 3
    const float* wrow[L];
#pragma unroll
    for (int h = 0; h < L; ++h) wrow[h] = p.w + (int64_t)min(n0 + h * 8 + (j & 7), p.N - 1) * p.K + k0 + q * 8 + (j >> 3) * 4;
    // Workgroups begin their slices at different steps, and go round: rows are as far apart as slices, often a power of two, and in step
    // they would all ask the same few channels of the memory
    const int turn = (int)(blockIdx.x * 5u % (unsigned)steps);
    auto w_load = [&](int s, int h) {
        s = min(s, steps - 1) + turn;
        return *reinterpret_cast<const f32x4*>(wrow[h] + (s < steps ? s : s - steps) * 32);
    };
    // lanes 8 .. 15 of `keep` (above) or 0 .. 7 (below) from the other half of `other`'s row of lanes
    auto above = [](float keep, float other) {
        return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(keep), __float_as_int(other), 0x128, 0xf, 0xc, false));
    };
    auto below = [](float keep, float other) {
        return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(keep), __float_as_int(other), 0x128, 0xf, 0x3, false));
    };
    // x: rows behind the last are the last
    const int ar = lane / LPR, ac = lane % LPR;
    f32x4 xa[AI];
    auto x_load = [&](int c) {
        int s = min(c * S + ac / 8, steps - 1) + turn;
        s = s < steps ? s : s - steps;
        const int k = k0 + s * 32 + ac % 8 * 4;
#pragma unroll
        for (int i = 0; i < AI; ++i) xa[i] = *reinterpret_cast<const f32x4*>(p.x + (int64_t)min(RPI * i + ar, p.M - 1) * p.ldx + k);
    };
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, wr[S][L];
    x_load(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int h = 0; h < L; ++h) wr[s][h] = w_load(s, h);
    const int chunks = (steps + S - 1) / S;
#pragma unroll 1
    for (int c = 0; c < chunks; ++c) {
#pragma unroll
        for (int i = 0; i < AI; ++i) *reinterpret_cast<f32x4*>(image + (RPI * i + ar) * kPitch + ac * 16) = xa[i];
        asm volatile("" ::: "memory");
        if (c + 1 < chunks) x_load(c + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int st = 0; st < S; ++st) {
            if (c * S + st >= steps) break;         // wave-uniform
            f32x4 b[2], a[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) a[h] = *reinterpret_cast<const f32x4*>(image + j * kPitch + st * 128 + q * 32 + h * 16);
            if constexpr (COLS == 16) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    b[0][e] = above(wr[st][0][e], wr[st][1][e]);      // row j, k 8 q + e
                    b[1][e] = below(wr[st][1][e], wr[st][0][e]);      // and 8 q + 4 + e
                }
            } else {
                b[0] = b[1] = wr[st][0];            // row j & 7: k 8 q + e of the first eight, 8 q + 4 + e of the others
            }
#pragma unroll
            for (int h = 0; h < L; ++h) wr[st][h] = w_load(c * S + st + S, h);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int h = 0; h < 2; ++h) acc[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[h][e], a[h][e], acc[h], 0, 0, 0);
        }
        asm volatile("" ::: "memory");
    }
    // acc[.][r] = row j, column 4 q + r: the wavefronts' tiles to LDS (each over its own, consumed image), added in their order
    const f32x4 part = COLS == 16 ? acc[0] + acc[1] : q < 2 ? acc[0] : acc[1];
    *reinterpret_cast<f32x4*>(image + (j * 16 + q * 4) * 4) = part;
    __syncthreads();
    if (tid >= 16 * COLS / 4) return;
    const int row = tid / (COLS / 4), at = tid % (COLS / 4) * 4, col = n0 + at;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kNW; ++w)
#pragma unroll
        for (int h = 0; h < 2 / L; ++h) s += *reinterpret_cast<const f32x4*>(lds + w * kWave + (row * 16 + h * 8 + at) * 4);
    if (row < p.M && col < p.N) *reinterpret_cast<f32x4*>(p.out + (int64_t)row * p.ldo + col) = s;
}

// Wide weights, K = 256 STEPS at most 2 048: a workgroup a CU takes every 256th tile of 16 columns.  x stays in registers, as fragments of
// the wavefront's slice of K; the loads of a tile are on their way while the one before it is multiplied, across the barrier at which the
// slices' sums meet, which a wavefront after the other adds up.  Workgroups' wavefronts start at different slices: rows are a power of two apart.
template <int STEPS>
__global__ __launch_bounds__(64 * kNW, 2) void f32_wide_kernel(const FewParams p, int tiles) {
    __shared__ f32x4 parts[2][kNW][64];
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, q = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slice = (wave + blockIdx.x) % kNW, k0 = slice * STEPS * 32;
    f32x4 a[STEPS][2], wr[STEPS][2];
    const float* xr = p.x + (int64_t)min(j, p.M - 1) * p.ldx + k0 + q * 8;
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) a[s][h] = *reinterpret_cast<const f32x4*>(xr + s * 32 + h * 4);
    auto row_of = [&](int t, int h) { return p.w + (int64_t)min(t * 16 + h * 8 + (j & 7), p.N - 1) * p.K + k0 + q * 8 + (j >> 3) * 4; };
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) wr[s][h] = *reinterpret_cast<const f32x4*>(row_of(blockIdx.x, h) + s * 32);
    auto above = [](float keep, float other) {
        return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(keep), __float_as_int(other), 0x128, 0xf, 0xc, false));
    };
    auto below = [](float keep, float other) {
        return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(keep), __float_as_int(other), 0x128, 0xf, 0x3, false));
    };
    int turn = 0;
#pragma unroll 1
    for (int t = blockIdx.x; t < tiles; t += gridDim.x, ++turn) {
        const int next = t + (int)gridDim.x;
        const float* from[2];                       // (behind the last tile: one line that is at hand)
#pragma unroll
        for (int h = 0; h < 2; ++h) from[h] = next < tiles ? row_of(next, h) : p.w;
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            f32x4 b[2];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                b[0][e] = above(wr[s][0][e], wr[s][1][e]);                // row j, k 8 q + e
                b[1][e] = below(wr[s][1][e], wr[s][0][e]);                // and 8 q + 4 + e
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) wr[s][h] = *reinterpret_cast<const f32x4*>(from[h] + s * 32);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int h = 0; h < 2; ++h) acc[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[h][e], a[s][h][e], acc[h], 0, 0, 0);
        }
        parts[turn & 1][slice][lane] = acc[0] + acc[1];                   // row j, columns 4 q .. + 3
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                // (the loads stay on their way)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (wave != turn % kNW) continue;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kNW; ++i) sum += parts[turn & 1][i][lane];
        const int col = t * 16 + q * 4;
        if (j < p.M && col < p.N) *reinterpret_cast<f32x4*>(p.out + (int64_t)j * p.ldo + col) = sum;
    }
}

template <int STEPS>
void launch_wide(const FewParams& p, hipStream_t st) {
    const int tiles = (p.N + 15) / 16;
    hipLaunchKernelGGL((f32_wide_kernel<STEPS>), dim3(tiles < 256 ? tiles : 256), dim3(64 * kNW), 0, st, p, tiles);
}

template <int COLS, int ROWS>
int launch_rows(const FewParams& p, hipStream_t st) {
    constexpr int bytes = kNW * 16 * (64 / COLS * 128 + 16);
    static MdPerDeviceOnce once;
    if (once.first() &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(&f32_few_kernel<COLS, ROWS>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
        once.undo();
        md_set_error("md_linear_f32_few: hipFuncSetAttribute(%d B LDS) failed", bytes);
        return MD_ERR_LAUNCH;
    }
    hipLaunchKernelGGL((f32_few_kernel<COLS, ROWS>), dim3((p.N + COLS - 1) / COLS), dim3(64 * kNW), bytes, st, p);
    return MD_OK;
}
template <int COLS>
int launch(const FewParams& p, hipStream_t st) {
    if (p.M <= 4) return launch_rows<COLS, 4>(p, st);
    return p.M <= 8 ? launch_rows<COLS, 8>(p, st) : launch_rows<COLS, 16>(p, st);
}

}  // namespace

namespace {
bool shape_ok(int M, int N, int K) {
    // wide: 6 rows, us, library / here 32 000 x 2 048 61.8 / 53.8, x 1 024 34.7 / 29.3, 8 192 x 1 024 14.6 / 10.9; level at 11 264 x 2 048 (22.6 / 22.1)
    // and below (6 144 16.0 / 16.5), 16 rows of 128 256 199 / 205
    const bool wide = K <= 1024 || (K <= 2048 && N >= 16384 && (M <= 8 || N <= 65536));
    return M > 0 && M <= 16 && N > 0 && K > 0 && (N <= 4096 || wide) && N < (1 << 26) && N % 4 == 0 && K % (32 * kNW) == 0 && K < (1 << 22);
}
}  // namespace

// Against the library over 1 800 products of 1 to 16 rows (16 to 140 000 columns, K = 256 to 16 384; operands from memory), which is the faster
// one, us, library / here:
//   * above 2 048 columns behind a K of 2 048: 4 096 x 4 096 17.1 / 18.6, 2 304 x 8 192 23.8 / 27.1 (its workgroups have 16 columns and all of K);
//   * with nine rows and more, whose x is staged twice as often, over up to 1 024 columns behind that K (1 024 x 3 072 9.0 / 10.6, 64 x 8 192
//     16.3 / 17.7), over more of them up to a K of 4 096 (2 048 x 3 072 11.7 / 12.7), and of few columns in front of it (128 x 1 536 6.1 / 6.9;
//     from 512 on and at 256 x 2 048 level or ahead).  Deeper ones of more than 1 024 columns are level alone (2 048 x 8 192 22.3 / 23.1), a
//     hundredth of a step faster in one, and less far off 64 bits (0.7 of the library's error);
//   * where either is little more than a launch: 4 096 x 256 5.0 / 5.1, 1 024 x 256 4.1 / 4.6, 16 x 256 3.9 / 4.3, 512 x 512 4.6 / 5.0,
//     384 x 768 1.03 times, but 128 x 256 9.9 / 4.5, 256 x 512 11.4 / 4.9, 768 x 512 5.7 / 5.0, 512 x 768 6.4 / 5.3;
//   * of a very wide weight, 65 536 x 256 18.0 / 22.3 (40 000 0.97 on average).
// What is left is 0.8 of the library's time on average, 1.09 at the worst (16 384 x 2 048, which the library likes).
extern "C" int md_linear_f32_few_supported(int M, int N, int K) {
    MD_CHECK_ARG(M > 0 && N > 0 && K > 0, "md_linear_f32_few_supported: M=%d N=%d K=%d", M, N, K);
    if (!shape_ok(M, N, K)) return 0;
    if (N > 4096) return K > 256 || N <= 49152;
    if (K == 256) return N > 32 && N <= 256;
    if (K <= 768) return (N > 32 && N <= 256) || N >= (K == 512 ? 768 : 512);
    if (N > 2048) return K <= 2048;
    if (M <= 8) return 1;
    return K <= 2048 ? N >= 512 || (N >= 256 && K > 1536) : N > 1024 && K > 4096;
}

extern "C" int md_linear_f32_few(const float* x, int64_t ldx, const float* w, float* out, int64_t ldo, int M, int N, int K, int tile, md_stream_t stream) {
    MD_CHECK_ARG(x && w && out, "md_linear_f32_few: null pointer argument");
    MD_CHECK_ARG(shape_ok(M, N, K) && ldx >= K && ldx % 4 == 0 && ldo >= N && ldo % 4 == 0 &&
                     (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0,
                 "md_linear_f32_few: M=%d N=%d K=%d ldx=%lld ldo=%lld unsupported", M, N, K, (long long)ldx, (long long)ldo);
    MD_CHECK_ARG(tile == 0 || tile == 8 || tile == 16, "md_linear_f32_few: tile of %d columns", tile);
    const FewParams p = {x, w, out, ldx, ldo, M, N, K};
    if (N > 4096) {
        hipStream_t st = (hipStream_t)stream;
        switch (K / 256) {
        case 1: launch_wide<1>(p, st); break;
        case 2: launch_wide<2>(p, st); break;
        case 3: launch_wide<3>(p, st); break;
        case 4: launch_wide<4>(p, st); break;
        case 5: launch_wide<5>(p, st); break;
        case 6: launch_wide<6>(p, st); break;
        case 7: launch_wide<7>(p, st); break;
        default: launch_wide<8>(p, st);
        }
        MD_CHECK_LAUNCH("md_linear_f32_few");
        return MD_OK;
    }
    // eight rows a workgroup: where 16 leave half the CUs idle (2 048 x 2 048 9.2 us, 8.0; but 768 x 512 5.0 and 5.4: few steps a wavefront)
    const int rc = (tile ? tile == 8 : N <= 2048 && K >= 1024) ? launch<8>(p, (hipStream_t)stream) : launch<16>(p, (hipStream_t)stream);
    if (rc != MD_OK) return rc;
    MD_CHECK_LAUNCH("md_linear_f32_few");
    return MD_OK;
}
