// 32-bit linear of a prompt's rows (gfx950):  out[M][N] = x[M][K] . W[N][K]^T, all float32, row-major
//
// replaces: the library products of the layered designs in 32-bit (prompts and the recorded traces that check a design).
//
// What bounds it: v_mfma_f32_16x16x4_f32, 64 flop per clock and SIMD (157 TFLOP/s; an 8192^3 library product reaches 152).  A step of 32 k
// of a 64 x 128 tile is 2 048 clocks of it for 24 KB (64 x 64: 1 024 for 16, 32 x 64: 512 for 12): both operands come by DMA in whole
// lines, three buffers, one barrier a step, two and more workgroups of four wavefronts on a CU that cover each other's barriers.  (Straight from memory into the instruction's order -- 64 bytes of
// 16 rows a load -- the address unit takes 42 clocks a load, and 64 x 64 wavefront tiles reach 124 TFLOP/s, 64 x 32 ones 83.)  A lane reads
// four k of a row at once; product e takes the e-th of each, the same four k of either operand.  What is left to choose is the tile, whose
// count should divide evenly among 256 CUs.
#include "md_common.h"

#include <algorithm>

namespace {

constexpr int kGroup = 16;    // row tiles whose column tiles are walked together

struct F32Params {
    const float* x;
    const float* w;
    float* out;
    int64_t ldx, ldo;
    int M, N, K;
    int mt, nt, total, per, group;
};

// four wavefronts, 2 x 2, of 16 TM rows x 16 TN columns each
template <int TM, int TN>
__global__ __launch_bounds__(256, 2) void f32_gemm_kernel(const F32Params p) {
    constexpr int kA = 32 * TM * 128, kBuf = kA + 32 * TN * 128, P = 4 * TM * TN;       // P: products of half a step
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];      // 3 x ([32 TM rows of x], [32 TN rows of W]) x 8 pieces of 16 B
    const int v = (blockIdx.x & 7) * p.per + (blockIdx.x >> 3);              // an XCD's workgroups lie side by side
    if (v >= p.total) return;
    const int g = v / (p.group * p.nt), r = v - g * p.group * p.nt, rows = min(p.group, p.mt - g * p.group);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, j = lane & 15, q = lane >> 4;
    const int tm = (g * p.group + r % rows) * 32 * TM, tn = r / rows * 32 * TN;
    // the descriptors end with the rows: those behind them read as zeros
    auto descriptor = [&](const float* base, int64_t first, int64_t pitch, int have) {
        const uint64_t at = (uint64_t)(base + first * pitch);
        return u32x4{(unsigned)at, (unsigned)(at >> 32) & 0xffffu, (unsigned)(have * pitch * 4), 0x00020000u};
    };
    const u32x4 rx = descriptor(p.x, tm, p.ldx, min(p.M - tm, 32 * TM)), rw = descriptor(p.w, tn, p.K, min(p.N - tn, 32 * TN));
    // piece c of row r stands at c ^ (r >> 1 & 7); the DMA writes lane after lane, so a lane fetches the piece that belongs at its place
    const unsigned piece = (unsigned)((tid & 7) ^ ((tid >> 4) & 7)) * 16;
    const unsigned xo = (unsigned)(tid >> 3) * (unsigned)p.ldx * 4 + piece, wo = (unsigned)(tid >> 3) * (unsigned)p.K * 4 + piece;
    auto load = [&](int buf, int k) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         : : "s"(buf * kBuf + i * 4096 + wave * 1024), "v"(xo + (unsigned)i * 128u * (unsigned)p.ldx), "s"(rx), "s"(k * 4) : "memory", "m0");
#pragma unroll
        for (int i = 0; i < TN; ++i)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         : : "s"(buf * kBuf + kA + i * 4096 + wave * 1024), "v"(wo + (unsigned)i * 128u * (unsigned)p.K), "s"(rw), "s"(k * 4) : "memory", "m0");
    };
    unsigned ar[2], br[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const unsigned at = (unsigned)(j * 128 + (((4 * h + q) ^ ((j >> 1) & 7)) * 16));
        ar[h] = at + (wave & 1) * 16 * TM * 128;
        br[h] = at + kA + (wave >> 1) * 16 * TN * 128;
    }
    f32x4 acc[TM][TN], a[2][TM], b[2][TN];
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int u = 0; u < TN; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto read = [&](int buf, int h, int i) {
        if (i < TM) a[h][i] = *reinterpret_cast<const f32x4*>(lds + ar[h] + (buf * kBuf + i * 2048));
        else b[h][i - TM] = *reinterpret_cast<const f32x4*>(lds + br[h] + (buf * kBuf + (i - TM) * 2048));
    };
    auto half = [&](int h, auto beside) {
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const int e = i / (TM * TN), t = i / TN % TM, u = i % TN;
            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[h][u][e], a[h][t][e], acc[t][u], 0, 0, 0);
            beside(i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // what a step needs was asked for two steps ago; behind the barrier nobody reads the third buffer any more
    auto step = [&](int buf, int k) {
        if (k + 32 < p.K) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(TM + TN) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (k + 64 < p.K) load((buf + 2) % 3, k + 64);
#pragma unroll
        for (int i = 0; i < TM + TN; ++i) read(buf, 0, i);
        __builtin_amdgcn_sched_barrier(0);
        half(0, [&](int i) {
#pragma unroll
            for (int l = 0; l < TM + TN; ++l)
                if (l * P / 2 / (TM + TN) == i) read(buf, 1, l);
        });
        half(1, [&](int) {});
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    load(0, 0);
    if (32 < p.K) load(1, 32);
    for (int k = 0; k < p.K; k += 96) {
        step(0, k);
        if (k + 32 < p.K) step(1, k + 32);
        if (k + 64 < p.K) step(2, k + 64);
    }
    const int m0 = tm + (wave & 1) * 16 * TM, n0 = tn + (wave >> 1) * 16 * TN;
    // lane (j, q) has row j of a tile and its columns 4 q .. + 3
#pragma unroll
    for (int t = 0; t < TM; ++t) {
        const int row = m0 + t * 16 + j;
        if (row >= p.M) continue;
#pragma unroll
        for (int u = 0; u < TN; ++u) {
            const int col = n0 + u * 16 + q * 4;
            if (col < p.N) *reinterpret_cast<f32x4*>(p.out + (int64_t)row * p.ldo + col) = acc[t][u];
        }
    }
}

template <int TM, int TN>
int launch(F32Params& p, hipStream_t st) {
    p.mt = (p.M + 32 * TM - 1) / (32 * TM);
    p.nt = (p.N + 32 * TN - 1) / (32 * TN);
    p.total = p.mt * p.nt;
    p.per = (p.total + 7) / 8;
    const int groups = (p.mt + kGroup - 1) / kGroup;
    p.group = (p.mt + groups - 1) / groups;
    static MdPerDeviceOnce once;
    if (3 * 32 * (TM + TN) * 128 > 64 * 1024 && once.first() &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(&f32_gemm_kernel<TM, TN>), hipFuncAttributeMaxDynamicSharedMemorySize,
                            3 * 32 * (TM + TN) * 128) != hipSuccess) {
        once.undo();
        md_set_error("md_linear_f32: hipFuncSetAttribute(%d B LDS) failed", 3 * 32 * (TM + TN) * 128);
        return MD_ERR_LAUNCH;
    }
    hipLaunchKernelGGL((f32_gemm_kernel<TM, TN>), dim3(8 * p.per), dim3(256), 3 * 32 * (TM + TN) * 128, st, p);
    return MD_OK;
}

// Tiles: rows x columns, and what one takes for 2 048 k: us by itself on a CU, and as one of several there; before its first step, us.  Measured from 32 to 8 192 rows;
// us, library / here: 4 803 x 3 072 x 2 048 539 / 444, x 2 048 x 2 048 367 / 307, x 8 192 x 2 048 1 187 / 1 098, 2 500 x 4 096 x 512 94 / 82,
// 700 x 3 072 x 2 048 107 / 84, 8192^3 7 358 / 7 234.  (128 x 128: 125 TFLOP/s there, 64 x 128 152.)
struct Tile {
    int rows, cols;
    double alone, among, first;
};
constexpr Tile kTiles[] = {{64, 128, 71.0, 56.5, 4.0}, {64, 64, 41.0, 29.0, 1.5}, {32, 64, 27.0, 15.6, 0.5}};

double tile_us(const Tile& t, int M, int N, int K) {
    const int64_t on_cu = ((int64_t)((M + t.rows - 1) / t.rows) * ((N + t.cols - 1) / t.cols) + 255) / 256;
    return 3.0 + (double)on_cu * t.first + K / 2048.0 * std::max(t.alone, (double)on_cu * t.among);
}

const Tile& best_tile(int M, int N, int K, double* us) {
    const Tile* best = nullptr;
    for (const Tile& t : kTiles) {
        const double c = tile_us(t, M, N, K);
        if (!best || c < *us) {
            best = &t;
            *us = c;
        }
    }
    return *best;
}

bool shape_ok(int M, int N, int K) { return M > 0 && N > 0 && K > 0 && N % 4 == 0 && K % 32 == 0 && K < (1 << 22); }

}  // namespace

// (Behind other launches, operands not in the caches, us, library / here: 4 803 x 3 072 x 2 048 521 / 441, x 2 048 x 8 192 1 233 / 1 206,
// 1 400 x 8 192 x 2 048 372 / 336, but 999 x 2 048 x 8 192 244 / 259, 560 x 2 048 x 8 192 157 / 203, 130 x 8 192 x 2 048 47 / 54: few rows,
// above all of deep products, leave CUs idle at the end, and the library splits K: 1 582 x 1 024 x 4 096 112 / 132.  Over 260 products of 1 200 to
// 6 000 rows 0.95 of the library's time, 1.09 at the worst; from 5 632 k on 0.85 to 1.09, level on average.)
extern "C" int md_linear_f32_supported(int M, int N, int K) {
    MD_CHECK_ARG(M > 0 && N > 0 && K > 0, "md_linear_f32_supported: M=%d N=%d K=%d", M, N, K);
    if (!shape_ok(M, N, K) || M < (K < 8192 ? 1200 : 2000)) return 0;
    double us = 0;
    best_tile(M, N, K, &us);
    return us <= 1.05 * (2e-6 * M * N / 130 * K + 8) ? 1 : 0;
}

extern "C" int md_linear_f32(const float* x, int64_t ldx, const float* w, float* out, int64_t ldo, int M, int N, int K, int tile,
                             md_stream_t stream) {
    MD_CHECK_ARG(x && w && out, "md_linear_f32: null pointer argument");
    MD_CHECK_ARG(shape_ok(M, N, K) && ldx >= K && ldx % 4 == 0 && ldx < (1 << 22) && ldo >= N && ldo % 4 == 0 &&
                     (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0,
                 "md_linear_f32: M=%d N=%d K=%d ldx=%lld ldo=%lld unsupported", M, N, K, (long long)ldx, (long long)ldo);
    F32Params p;
    p.x = x;
    p.w = w;
    p.out = out;
    p.ldx = ldx;
    p.ldo = ldo;
    p.M = M;
    p.N = N;
    p.K = K;
    double us = 0;
    const Tile& t = best_tile(M, N, K, &us);
    const int rows = tile ? tile / 1000 : t.rows, cols = tile ? tile % 1000 : t.cols;
    hipStream_t st = (hipStream_t)stream;
    int rc;
    if (rows == 64 && cols == 128) rc = launch<2, 4>(p, st);
    else if (rows == 64 && cols == 64) rc = launch<2, 2>(p, st);
    else if (rows == 32 && cols == 64) rc = launch<1, 2>(p, st);
    else {
        md_set_error("md_linear_f32: no tile of %d x %d", rows, cols);
        return MD_ERR_UNSUPPORTED;
    }
    if (rc != MD_OK) return rc;
    MD_CHECK_LAUNCH("md_linear_f32");
    return MD_OK;
}
