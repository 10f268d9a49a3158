// 32-bit linear of a prompt's rows on the bf16 matrix cores (gfx950):  out[M][N] = x[M][K] . W[N][K]^T, all float32, row-major
//
// replaces: md_linear_f32 (fp32 matrix instructions, 157 TFLOP/s) for prompts of the layered designs in 32-bit.
//
// A float32 number is the sum of three bf16 numbers: a = a1 + a2 + a3, each the rounded rest of those before it (8 + 8 + 8 bits of mantissa).
// Of the nine products of two such sums six are taken, smallest first: a3 b1, a2 b2 + a2 b1, a1 b3 + a1 b2 + a1 b1.  The others are 2^-27.5 of
// a b as a root mean square, a fifth of what rounding that product to 32 bits costs, and at most 2^-24, as much as that, where the rests are
// as large as they can be (1 + 2^-8 - 2^-17 + 2^-23 squared).  bf16 products are exact in the instruction, whose sums are 32-bit as those of
// the fp32 instruction are, and of 32 products instead of 4; they round towards smaller sums a little.
// Error against 64 bits as a 2-norm, over md_linear_f32's (K = 256 / 2 048 / 8 192): normal numbers 0.80 / 0.86 / 0.88, uniform positive ones 0.79 / 0.64 /
// 0.63, activations of xIELU 0.82 / 0.85 / 0.84, outliers 0.73 / 0.71 / 0.69, but rows of which half are zeros, which cost the fp32 sums nothing, 1.09 /
// 1.15 / 1.17 (both operands 1.32 / 1.24 / 1.18), a single term a sum 1.25; sums of equal terms, which 32 bits may hold exactly, up to 2^-17.
// Parts are multiples of 2^-133: numbers below 2^-110 have fewer bits than 24, and are off by up to 2^-134 (md_linear_f32 keeps them).
//
// What bounds it: the matrix cores, at 16 times the fp32 instruction's rate for six products instead of one.  8192^3: 4 113 us here, 7 462
// md_linear_f32, matrix cores busy for 84 % of the cycles at the 1.78 GHz that so many of them leave; error against 64 bits 0.86 of it
// (2 000 x 2 048 x 2 048: 6.98e-7, 8.09e-7 there and in the library).
//   * x is split by a pass of its own (6.6 TB/s), into the order in which the instruction takes it: a 16-row, 32-k piece is 3 KB in a row;
//   * W comes as it stands, by DMA into the wavefront's own part of LDS, and is split in registers beside the products (176 vector
//     instructions, in twos, beside 384 products a step of 32 k of 256 x 256; in fives the matrix cores wait: 79 % busy): no copy of a
//     weight that could grow old, no second pass over it;
//   * four wavefronts of BM rows x 16 NT columns each; all read every row's piece from LDS, 12 products for each KB at NT = 4;
//   * two to four buffers, one barrier per 32 k, where the last products' pieces are in registers already: the loads of a later step begin
//     there, one beside every fifth or sixth product (all beside the last 48: 4 658 us; with half lines of W as well).
#include "md_common.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace {

constexpr int kGroup = 8;     // most row tiles whose column tiles are walked together

struct ThirdsParams {
    const float* x;
    const float* w;
    const unsigned char* xs;   // [16-row pieces][K / 32][3][64 lanes][8] bf16
    float* out;
    int64_t ldx, ldo;
    int M, N, K;
    int mt, nt, total, per, group;
};

__device__ __forceinline__ unsigned int pack2(float a, float b) {
    const bf16x2 v = {f32_to_bf16(a), f32_to_bf16(b)};
    return *reinterpret_cast<const unsigned int*>(&v);
}
// two numbers' next parts; what is left of them stays
__device__ __forceinline__ unsigned int part2(float& a, float& b) {
    const unsigned int q = pack2(a, b);
    a -= __uint_as_float(q << 16);
    b -= __uint_as_float(q & 0xffff0000u);
    return q;
}
template <int... I, class F>
__device__ __forceinline__ void unrolled(std::integer_sequence<int, I...>, F f) {
    (f(std::integral_constant<int, I>()), ...);
}
// f(k) for those of n things that lie behind place i of p, spread evenly
template <class F>
__device__ __forceinline__ void spread(int i, int p, int n, F f) {
#pragma unroll
    for (int k = 0; k < n; ++k)
        if (k * p / n == i) f(k);
}

// ---------------------------------------------------------------------------------------------------------- x in three parts
// A wavefront: 16 rows x 32 k.  Lane (j, q) has row j and k 4 q .. + 3 and 16 + 4 q .. + 3: whole lines of x in two loads, and W's lanes
// read theirs in the same order.  Rows behind the last are zeros.
__global__ __launch_bounds__(256) void thirds_kernel(const float* __restrict__ x, int64_t ldx, int M, int units, unsigned char* __restrict__ xs) {
    const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4, row = blockIdx.y * 16 + j;
    const int u = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= units) return;
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
    if (row < M) {
        const float* at = x + (int64_t)row * ldx + u * 32 + q * 4;
        lo = *reinterpret_cast<const f32x4*>(at);
        hi = *reinterpret_cast<const f32x4*>(at + 16);
    }
    float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    unsigned char* to = xs + ((int64_t)blockIdx.y * units + u) * 3072 + lane * 16;
#pragma unroll
    for (int i = 0; i < 3; ++i)
        *reinterpret_cast<u32x4*>(to + i * 1024) = u32x4{part2(v[0], v[1]), part2(v[2], v[3]), part2(v[4], v[5]), part2(v[6], v[7])};
}

// ---------------------------------------------------------------------------------------------------------- the product
template <int MT, int NT>
constexpr int buffers() {
    return std::min(4, 163840 / (MT * 3072 + NT * 8192));
}

template <int MT, int NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void f32_thirds_kernel(const ThirdsParams p) {
    constexpr int BM = 16 * MT, kA = MT * 3072, kW = NT * 2048, kBuf = kA + 4 * kW;     // a buffer: x's pieces, four wavefronts' columns of W
    constexpr int NB = buffers<MT, NT>();
    // pieces of x a step; how far they are read ahead (LDS answers after 130 cycles and more); registers for them
    constexpr int F = 3 * MT, R = NT == 4 || MT < 8 ? 4 : 8, RING = NT == 4 ? 6 : 12;
    static_assert(F % RING == 0, "the ring goes on where the step before ended");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int v = (blockIdx.x & 7) * p.per + (blockIdx.x >> 3);  // an XCD's workgroups lie side by side
    if (v >= p.total) return;
    const int g = v / (p.group * p.nt), r0 = v - g * p.group * p.nt, rows = min(p.group, p.mt - g * p.group);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, j = lane & 15, q = lane >> 4;
    const int tm = (g * p.group + r0 % rows) * BM, tn = r0 / rows * 64 * NT + wave * 16 * NT;
    const int units = p.K / 32, pieces = (p.M + 15) / 16;
    // the descriptors end with the rows: those behind them read as zeros
    auto descriptor = [&](const void* base, uint64_t bytes) {
        const uint64_t at = (uint64_t)base;
        return u32x4{(unsigned)__builtin_amdgcn_readfirstlane((int)at), (unsigned)__builtin_amdgcn_readfirstlane((int)(at >> 32) & 0xffff),
                     (unsigned)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
    };
    const u32x4 rx = descriptor(p.xs + (int64_t)(tm / 16) * units * 3072, (uint64_t)min(pieces - tm / 16, MT) * units * 3072);
    const int have = max(0, min(p.N - tn, 16 * NT));
    const u32x4 rw = descriptor(p.w + (have ? (int64_t)tn * p.K : 0), (uint64_t)have * p.K * 4);
    // W: 8 rows x 128 bytes a load, whole lines.  Piece c of row r stands at c ^ (r >> 1); the DMA writes lane after lane, so a lane
    // fetches the piece that belongs at its place
    unsigned wo[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) wo[h] = ((unsigned)(h * 8 + (lane >> 3)) * p.K + ((lane & 7) ^ (h * 4 + (lane >> 4))) * 4) * 4u;
    const unsigned wr = (unsigned)(j * 128 + ((q ^ (j >> 1)) * 16));         // (piece 4 + q: 64 bytes on or back)
    // DMA of one step: piece i of this wavefront (its share of x, then its own columns of W) into the buffer at `to`
    constexpr int DA = (F + 3) / 4, DW = 2 * NT, D = DA + DW;
    unsigned from[D];
#pragma unroll
    for (int i = 0; i < D; ++i) {
        const int f = i * 4 + wave, n = (i - DA) / 2;
        from[i] = i < DA ? (unsigned)(f / 3 * units) * 3072u + (unsigned)(f % 3) * 1024u + lane * 16u : wo[(i - DA) & 1] + (unsigned)n * 64u * (unsigned)p.K;
    }
    auto load = [&](unsigned to, int u, auto ic) {
        constexpr int i = decltype(ic)::value;
        if (i < DA && F % 4 != 0 && i * 4 + wave >= F) return;
        unsigned at = i < DA ? (unsigned)u * 3072u : (unsigned)u * 128u, lds_at = to + (i < DA ? wave * 1024u : kA + wave * kW);
        const unsigned off = from[i];
        const u32x4 rsrc = i < DA ? rx : rw;
        asm volatile("" : "+s"(at), "+s"(lds_at));               // (in registers, constant or not)
        asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     : : "s"(lds_at), "v"(off), "s"(rsrc), "s"(at), "n"(i < DA ? i * 4096 : (i - DA) * 1024) : "memory", "m0", "scc");
    };
    bf16x8 a[RING];
    unsigned b1[NT][4], b2[NT][4], b3[NT][4], next1[NT][4];      // W's parts; its first part of the step to come
    float raw[NT][8];                                            // what is left of it
    // piece f of a step: the third parts of all rows, then the second, then the first
    auto read_a = [&](unsigned from, auto fc) {
        constexpr int f = decltype(fc)::value;
        a[f % RING] = *reinterpret_cast<const bf16x8*>(lds + from + lane * 16 + ((f % MT) * 3 + 2 - f / MT) * 1024);
    };
    auto read_w = [&](unsigned from, int i) {
        const f32x4 z = *reinterpret_cast<const f32x4*>(lds + from + kA + wave * kW + (i / 2) * 2048 + (wr ^ (i & 1) * 64));
#pragma unroll
        for (int e = 0; e < 4; ++e) raw[i / 2][(i & 1) * 4 + e] = z[e];
    };
    f32x4 acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[n][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto product = [&](const unsigned (&b)[4], const bf16x8& x, f32x4& c) {
        // (in assembly: left to the compiler, accumulators of four registers wander)
        asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(u32x4{b[0], b[1], b[2], b[3]}), "v"(x));
    };

    // ---- before the first step
    constexpr int L = (3 * R + MT) * NT;                         // products beside which a step's loads are issued
#pragma unroll
    for (int k = 0; k < NB; ++k)
        unrolled(std::make_integer_sequence<int, D>(), [&](auto i) {
            if (k < NB - 1 || i * L / D < 3 * R * NT) load(k * kBuf, min(k, units - 1), i);     // (the last ones: those that stand behind a barrier)
        });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < DW; ++i) read_w(0, i);
    unrolled(std::make_integer_sequence<int, R>(), [&](auto f) { read_a(0, f); });
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) b1[n][e] = pack2(raw[n][2 * e], raw[n][2 * e + 1]);

    unsigned place[NB];                                          // of this step and of those that follow
#pragma unroll
    for (int k = 0; k < NB; ++k) place[k] = k * kBuf;
    for (int u = 0; u < units; ++u) {
        const unsigned now = place[0], other = place[1];
        const int before = min(u + NB - 1, units - 1), after = min(u + NB, units - 1);          // (behind the last step: loads that nobody reads)
        unrolled(std::make_integer_sequence<int, F>(), [&](auto fc) {
            constexpr int f = decltype(fc)::value, t = f % MT, part = f / MT, parts = part + 1;
            if constexpr (f == F - R) {
                // Every piece of this step is read, and the next step's loads are there: behind the barrier this step's buffer is free and
                // the next one whole.  (In flight may be the loads of the steps behind that one)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NB - 2) * (DW + F / 4)) : "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
            // W's parts are written by vector instructions, which the compiler does not see a product behind
            if constexpr (t == 0) asm volatile("s_nop 1" ::: "memory");
            unrolled(std::make_integer_sequence<int, parts * NT>(), [&](auto ic) {
                constexpr int i = decltype(ic)::value, n = i % NT, k = i / NT;      // k: W's part, the last one first
                product(part - k == 2 ? b3[n] : part - k == 1 ? b2[n] : b1[n], a[f % RING], acc[n][t]);
                if constexpr (i == 0) {
                    if constexpr (f + R < F) read_a(now, std::integral_constant<int, (f + R < F ? f + R : 0)>());
                    else read_a(other, std::integral_constant<int, (f + R < F ? 0 : f + R - F)>());
                }
                constexpr int at = t * parts * NT + i, P = MT * parts * NT, behind = (f - (F - R)) * 3 * NT + i;
                // What is left of W behind its first part, then the second; behind that, then the third: two or three instructions beside
                // a product hide behind it, five do not
                if constexpr (part < 2)
                    spread(at, P, 12 * NT, [&](int y) {
                        const int x = y / 3, n = x / 4, e = x % 4;
                        const unsigned before = part == 0 ? b1[n][e] : b2[n][e];
                        if (y % 3 == 0) raw[n][2 * e] -= __uint_as_float(before << 16);
                        else if (y % 3 == 1) raw[n][2 * e + 1] -= __uint_as_float(before & 0xffff0000u);
                        else (part == 0 ? b2 : b3)[n][e] = pack2(raw[n][2 * e], raw[n][2 * e + 1]);
                    });
                if constexpr (behind >= 0) {
                    spread(behind, 3 * NT, DW, [&](int x) { read_w(other, x); });
                    spread(behind - 6 * NT, 6 * NT, 4 * NT, [&](int x) { next1[x / 4][x % 4] = pack2(raw[x / 4][2 * (x % 4)], raw[x / 4][2 * (x % 4) + 1]); });
                }
                // the loads of the step that takes this one's buffer: from the barrier on, to the end of the next step's third parts
                constexpr int since = behind >= 0 ? behind : part == 0 ? 3 * R * NT + t * NT + i : -1;
                if constexpr (since >= 0)
                    unrolled(std::make_integer_sequence<int, D>(), [&](auto x) {
                        if constexpr (x * L / D == since) load(behind >= 0 ? now : place[NB - 1], behind >= 0 ? after : before, x);
                    });
                __builtin_amdgcn_sched_barrier(0);
            });
        });
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) b1[n][e] = next1[n][e];
#pragma unroll
        for (int k = 0; k < NB - 1; ++k) place[k] = place[k + 1];
        place[NB - 1] = now;
        asm volatile("" ::: "memory");
    }
    // (the products are assembly: what the compiler would wait between the last of them and reading its accumulator; and no DMA into another
    // workgroup's LDS)
    asm volatile("s_nop 15\n\ts_nop 15\n\ts_waitcnt vmcnt(0)" ::: "memory");
    // lane (j, q) has row j of a tile and its columns 4 q .. + 3
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int row = tm + t * 16 + j;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int col = tn + n * 16 + q * 4;
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float z;
                asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(z) : "a"(acc[n][t][e]));
                o[e] = z;
            }
            if (row >= p.M || col >= p.N) continue;
            // infinities (and numbers that round to them) fall into parts that cancel: such sums once more, in 32 bits
            const float size = fmaxf(fmaxf(fabsf(o[0]), fabsf(o[1])), fmaxf(fabsf(o[2]), fabsf(o[3])));
            if (__builtin_expect(!(size < INFINITY) || o[0] != o[0] || o[1] != o[1] || o[2] != o[2] || o[3] != o[3], 0)) {
                const float* xr = p.x + (int64_t)row * p.ldx;
                for (int e = 0; e < 4; ++e) {
                    if (fabsf(o[e]) < INFINITY) continue;
                    const float* wr = p.w + (int64_t)(col + e) * p.K;
                    float s = 0.f;
                    for (int k = 0; k < p.K && s == s; ++k) s = fmaf(xr[k], wr[k], s);
                    o[e] = s;
                }
            }
            *reinterpret_cast<f32x4*>(p.out + (int64_t)row * p.ldo + col) = o;
        }
    }
}

template <int MT, int NT>
int launch(ThirdsParams& p, hipStream_t st) {
    constexpr int bm = 16 * MT, bn = 64 * NT, bytes = buffers<MT, NT>() * (MT * 3072 + NT * 8192);
    p.mt = (p.M + bm - 1) / bm;
    p.nt = (p.N + bn - 1) / bn;
    p.total = p.mt * p.nt;
    p.per = (p.total + 7) / 8;
    const int groups = (p.mt + kGroup - 1) / kGroup;
    p.group = (p.mt + groups - 1) / groups;
    static MdPerDeviceOnce once;
    if (once.first() && hipFuncSetAttribute(reinterpret_cast<const void*>(&f32_thirds_kernel<MT, NT>),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
        once.undo();
        md_set_error("md_linear_f32_thirds: hipFuncSetAttribute(%d B LDS) failed", bytes);
        return MD_ERR_LAUNCH;
    }
    hipLaunchKernelGGL((f32_thirds_kernel<MT, NT>), dim3(8 * p.per), dim3(256), bytes, st, p);
    return MD_OK;
}

// Tiles: rows x columns, and what one takes: us before the first step of 32 and behind the last, us a step while most CUs idle, and how much
// slower that is with all of them busy (the clock).  Drawn from 170 random products (91 to 6 920 rows, 13 weights of 768 x 3 072 to
// 11 264 x 2 048, operands not in the caches); the tile that this picks is within 0.5 % of the best at the worst.
struct Tile {
    int rows, cols;
    double fixed, step, busy;
};
constexpr Tile kTiles[] = {{256, 256, 18.5, 2.80, 1.27}, {192, 256, 15.2, 2.20, 1.24}, {160, 256, 13.8, 1.99, 1.19}, {128, 256, 12.3, 1.63, 1.20},
                           {256, 128, 12.0, 1.53, 1.24}, {192, 128, 11.0, 1.23, 1.21}, {128, 128, 9.9, 0.92, 1.16}, {64, 128, 6.5, 0.66, 1.00}};

double tile_us(const Tile& t, int M, int N, int K) {
    const int64_t total = (int64_t)((M + t.rows - 1) / t.rows) * ((N + t.cols - 1) / t.cols), rounds = total / 256, rest = total % 256;
    const double body = (double)(K / 32) * t.step;
    double us = (double)rounds * (t.fixed + body * t.busy);
    if (rest) us += t.fixed + body * (1.0 + (t.busy - 1.0) * (double)rest / 256);
    return us;
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

bool shape_ok(int M, int N, int K) { return M > 0 && N > 0 && K > 0 && N % 4 == 0 && K % 32 == 0 && K < (1 << 20); }

}  // namespace

// Against the library and md_linear_f32, the faster of them, which take 2 M N K / 130 TFLOP/s and some us at best: over the 170 products
// above 0.82 of their time (4 803 x 8 192 x 2 048 1 129 / 708, x 2 048 x 8 192 1 197 / 736, 994 x 8 192 x 2 048 245 / 144, 348 x 4 096 x 4 096
// 109 / 103), 1.02 at the worst, and five products left to them that were 3 % faster here and more.  Few rows of a narrow weight leave CUs idle,
// and the library splits K: 460 x 2 048 x 8 192 130 / 185.
extern "C" int md_linear_f32_thirds_supported(int M, int N, int K) {
    MD_CHECK_ARG(M > 0 && N > 0 && K > 0, "md_linear_f32_thirds_supported: M=%d N=%d K=%d", M, N, K);
    if (!shape_ok(M, N, K)) return 0;
    double us = 0;
    best_tile(M, N, K, &us);
    us += 2.5 + 10.0 * M * K / 6e6;                            // (x's parts: 4 bytes read, 6 written)
    return us <= 2e-6 * M * N / 130 * K + 4 ? 1 : 0;
}

extern "C" size_t md_linear_f32_thirds_workspace(int M, int K) { return M > 0 && K > 0 ? (size_t)((M + 15) / 16) * 16 * K * 6 : 0; }

extern "C" int md_linear_f32_thirds(const float* x, int64_t ldx, const float* w, float* out, int64_t ldo, int M, int N, int K, int tile,
                                    void* ws, size_t ws_bytes, md_stream_t stream) {
    MD_CHECK_ARG(x && w && out && ws, "md_linear_f32_thirds: null pointer argument");
    MD_CHECK_ARG(shape_ok(M, N, K) && ldx >= K && ldx % 4 == 0 && ldo >= N && ldo % 4 == 0 &&
                     (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)ws) & 15) == 0,
                 "md_linear_f32_thirds: M=%d N=%d K=%d ldx=%lld ldo=%lld unsupported", M, N, K, (long long)ldx, (long long)ldo);
    MD_CHECK_ARG(M <= 16 * 65535, "md_linear_f32_thirds: M=%d: the parts' grid has a row of workgroups for 16 rows, at most 65 535", M);
    MD_CHECK_ARG(ws_bytes >= md_linear_f32_thirds_workspace(M, K), "md_linear_f32_thirds: workspace of %zu bytes, %zu needed", ws_bytes,
                 md_linear_f32_thirds_workspace(M, K));
    ThirdsParams p;
    p.x = x;
    p.w = w;
    p.xs = (const unsigned char*)ws;
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
    const int units = K / 32;
    hipLaunchKernelGGL(thirds_kernel, dim3((units + 3) / 4, (M + 15) / 16), dim3(256), 0, st, x, ldx, M, units, (unsigned char*)ws);
    MD_CHECK_LAUNCH("md_linear_f32_thirds (split)");
    int rc;
    if (rows == 256 && cols == 256) rc = launch<16, 4>(p, st);
    else if (rows == 192 && cols == 256) rc = launch<12, 4>(p, st);
    else if (rows == 160 && cols == 256) rc = launch<10, 4>(p, st);
    else if (rows == 128 && cols == 256) rc = launch<8, 4>(p, st);
    else if (rows == 256 && cols == 128) rc = launch<16, 2>(p, st);
    else if (rows == 192 && cols == 128) rc = launch<12, 2>(p, st);
    else if (rows == 128 && cols == 128) rc = launch<8, 2>(p, st);
    else if (rows == 64 && cols == 128) rc = launch<4, 2>(p, st);
    else {
        md_set_error("md_linear_f32_thirds: no tile of %d x %d", rows, cols);
        return MD_ERR_UNSUPPORTED;
    }
    if (rc != MD_OK) return rc;
    MD_CHECK_LAUNCH("md_linear_f32_thirds");
    return MD_OK;
}
