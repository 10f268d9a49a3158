// GEMM of a prompt's rows (gfx950):  out = epilogue(x[M][K] . W[N][K]^T + bias), W in the streaming layout of md_linear
//
// replaces: the nn.Linear calls of a prompt (Engine/SnapKV/model.py:288-289 wqkv / wo, :446-455 w1 / w3 / w2), M of several hundred to
//           16 384 rows, which ran on the library: over row-major weights that every prompt had to bring back from the streaming layout
//           first (unpack_weight: 320 of 6 500 us of a two-layer 8B prompt), and with the gated activation as a pass of its own (260 us).
//
// Also a step's 129 to 256 rows where the block kernel needs a second round of the chip for its 128 columns a workgroup.
//
// What bounds it.  The matrix cores, busy for 78 to 85 % of the cycles of the large products, at the clock that so many of them leave: 1.8 to
// 1.9 of 2.4 GHz, as the library's (profiles/prompt_kernels.txt).  v_mfma_f32_16x16x32 moves half the accumulator bytes per flop of
// 32x32x16, and an 8192^3 product took no longer with it, although its 16 cycles hide less behind each.  Measured, us:
// (8192, 4096, 4096) 180, library 184; (8192, 4096, 14336) 612 / 604; (8192, 28672, 4096) with SiLU * mul 1 299 / 1 391;
// (8196, 4096, 18432) 972 / 1 311; (6144, 2048, 8192) 135 / 152; (2081, 37888, 3584) 433 / 552.
//   * four wavefronts of 256 rows x 64 columns, one per SIMD with 256 accumulators: each reads all of A from LDS and its own columns of W
//     straight from memory, already in the instruction's order (W through LDS as well would need 2 048 of the 2 048 cycles that a step of
//     64 takes there; 128 x 128 tiles per wavefront load W twice, which the address unit does not keep up with);
//   * A by DMA through three buffers: by way of registers its LDS writes alone cost 12 % of the cycles;
//   * W four steps of 64 ahead in registers (two: 1 024 x 4 096 x 4 096 in 37.6 us instead of 31.6, 6 144 x 3 072 x 2 048 in 70.2 instead of
//     64.2, the large ones 1 % slower), A two to three in LDS and half a step in registers; one barrier a step, where the last LDS
//     instruction lies some products back;
//   * one instruction beside each product, in an order that the compiler has to keep (spread): in bunches the four wavefronts queue at the
//     address unit and at LDS, and the matrix cores wait (8192 x 28 672 x 4 096: 1 610 us so, 1 384 spread);
//   * workgroups stay and take tile after tile; the loads of the next tile are in flight behind the last steps of one;
//   * an XCD's 32 workgroups take 8 row tiles x 4 column tiles, whose operands its L2 holds (4 or 16 row tiles: 1.5 / 4 % slower).
#include "md_common.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace {

enum { PE_NONE = 0, PE_SWIGLU = 1, PE_XIELU = 2, PE_GEGLU = 3, PE_BIAS = 4 };

struct PromptParams {
    const bf16_t* x;
    const bf16_t* w;        // [tiles of 32 columns][K/16][64 lanes][8]
    const bf16_t* bias;     // [N] or null (PE_NONE)
    const float* act;       // PE_XIELU
    bf16_t* out;
    int64_t ldx, ldo;
    int M, K, Nout;         // output columns
    unsigned w_bytes;
    int wtiles;             // 32-column tiles of the weight
    int mt, nt, total, per; // tiles of the launch, workgroups per XCD
    int group;              // row tiles whose column tiles are walked together
};

constexpr int kBK = 64;
constexpr int kGroup = 8;   // most row tiles in a group

__device__ __forceinline__ unsigned int pack2(float a, float b) {
    const bf16x2 v = {f32_to_bf16(a), f32_to_bf16(b)};
    return *reinterpret_cast<const unsigned int*>(&v);
}
__device__ __forceinline__ float round_bf16(float a) { return bf16_to_f32(f32_to_bf16(a)); }
// Activations of a tile's values, without a branch and in few instructions, since no product runs beside them.  Against 64-bit arithmetic
// they are as exact as what the other kernels call (expf and a division, expm1f): largest relative errors 1.3e-7 of SiLU (the same over
// all bf16 numbers), 1.6e-7 of GELU around 0, where those have 1.6e-7, 1.0e-7 of xIELU (alpha 0.85 and 1.1) for 1.6e-7.
// 8192 x 28 672 x 4096 with SiLU * mul 1 327 us, 1 351 with the calls; 8192 x 16 384 x 2048 388 and 406; 16 384 x 14 336 x 4096 with
// xIELU 1 363 and 1 388.  (The hardware's exponential and reciprocal alone: 1 303, 372 and 1 310, but up to 3e-6, and 0 where a sigmoid is
// no normal number; 2^x - 1 - n of a small negative n: 5e-5.)
// z / (1 + e), as exact as a division: of a 16th of both, since the reciprocal of 1 + e (up to 2^128) may be no normal number
__device__ __forceinline__ float over_one_plus(float z, float e) {
    const float d = fmaf(e, 0.0625f, 0.0625f), n = z * 0.0625f, r = __builtin_amdgcn_rcpf(d), q = n * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, d, n), r, q), d, n);        // (infinities, NaN)
}
// z / (1 + e^-z) of a bf16 number, whose product with 15 bits of log2(e) is exact
__device__ __forceinline__ float silu_flat(float z) {
    const float x = __builtin_amdgcn_fmed3f(z, -100.f, 100.f), t = x * -0x1.7154p+0f, k = rintf(t);
    return over_one_plus(z, __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(fmaf(x, -7.05260771340736e-06f, t - k)), (int)k));
}
// gelu_tanh: e^(-2 sqrt(2/pi) u) = 2^(-K u), K in two parts, the product's rounding added behind
__device__ __forceinline__ float gelu_flat(float z) {
    constexpr float kHi = -0x1.26aec2p+1f, kLo = -1.2948402037571394e-08f;
    const float u = __builtin_amdgcn_fmed3f(fmaf(0.044715f * z * z, z, z), -120.f, 120.f);
    const float t = u * kHi, rest = fmaf(u, kLo, fmaf(u, kHi, -t)), e = __builtin_amdgcn_exp2f(t);
    return over_one_plus(z, fmaf(fminf(e, 0x1.fffffep+127f), rest * 0.693147181f, e));
}
// Xielu.  e^n - 1 = 2^k (e^f - 1) + (2^k - 1) with n = k ln 2 + f, |f| < 0.35 (Cody and Waite), e^f - 1 from its series
__device__ __forceinline__ float xielu_flat(float ap, float an, float z) {
    const float n = fmaxf(fminf(z, 0.f), -104.f), k = rintf(n * 1.44269504f), f = fmaf(k, -1.42860682e-06f, fmaf(k, -0x1.62e4p-1f, n));
    float s = fmaf(f, 1.f / 5040, 1.f / 720);
    s = fmaf(s, f, 1.f / 120);
    s = fmaf(s, f, 1.f / 24);
    s = fmaf(s, f, 1.f / 6);
    s = fmaf(s, f, 0.5f);
    const float scale = __builtin_amdgcn_ldexpf(1.0f, (int)k), em1 = fmaf(scale, fmaf(f * f, s, f), scale - 1.0f);
    const float half = 0.5f * z;
    return z > 0.f ? fmaf(ap * z, z, half) : fmaf(an, em1 - z, half);
}
// f(0), f(1), ...: what a loop of this length is not always unrolled to
template <int... I, class F>
__device__ __forceinline__ void unrolled(std::integer_sequence<int, I...>, F f) {
    (f(I), ...);
}
// f(k) for those of n things that lie behind place i of p, spread evenly; shift: 0 even places first, else odd ones
template <class F>
__device__ __forceinline__ void spread(int i, int p, int n, int shift, F f) {
#pragma unroll
    for (int k = 0; k < n; ++k)
        if (min(k * p / n | shift, p - 1) == i) f(k);
}
__device__ __forceinline__ void wait_lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int MT, int NT, int EPI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void prompt_gemm_kernel(const PromptParams p) {
    constexpr int BM = 16 * MT, AL = BM / 32, AH = AL / 2;       // AL: 16-byte pieces of A per thread and step
    constexpr int kBuf = BM * kBK * 2;
    constexpr bool GATED = EPI == PE_SWIGLU || EPI == PE_GEGLU;
    constexpr int CW = NT * (GATED ? 8 : 16), CH = CW / 8;       // columns of a wavefront's output, in 16-byte pieces
    constexpr int AR = MT > 8 ? MT / 2 : MT;                      // tiles of A in registers
    constexpr int P = MT * NT;                                   // products of half a step
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];      // 3 x [BM rows][8 chunks of 16 B], chunk ^ (row >> 1 & 7)
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, j = lane & 15, kq = lane >> 4;
    const int grid = gridDim.x, first = (blockIdx.x & 7) * p.per + (blockIdx.x >> 3);
    if (first >= p.total) return;
    const int steps = p.K / kBK;
    unsigned char* image = lds + 3 * kBuf + wave * (2 * 32 * CW * 2);

    auto place = [&](int v, int& m, int& n) {
        const int g = v / (p.group * p.nt), r = v - g * p.group * p.nt, rows = min(p.group, p.mt - g * p.group);
        m = g * p.group + r % rows;
        n = r / rows;
    };

    // ---- the two load streams.  A's descriptor ends with the rows (those behind them read as zeros), W's tiles behind the last are the last
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.w), (short)0, (int)p.w_bytes, 0x00020000);
    u32x4 ra;                                                    // A's descriptor: base, bytes, flags
    unsigned ka, bbase[NT / 2], bnext[NT / 2];
    const unsigned boff = (unsigned)((kq >> 1) * 1024 + (kq & 1) * 512 + j * 16);
    unsigned aoff[AL];
#pragma unroll
    for (int i = 0; i < AL; ++i) aoff[i] = (unsigned)(((tid >> 3) + i * 32) * (int)p.ldx * 2 + (((tid & 7) ^ ((tid >> 4) & 7)) * 16));
    auto seek_a = [&](int v) {
        int m, n;
        place(v, m, n);
        const uint64_t base = (uint64_t)(p.x + (int64_t)m * BM * p.ldx);
        ra = u32x4{(unsigned)base, (unsigned)(base >> 32) & 0xffffu, (unsigned)(min(p.M - m * BM, BM) * (int)p.ldx * 2), 0x00020000u};
        ka = 0;
    };
    auto seek_b = [&](int v) {
        int m, n;
        place(v, m, n);
#pragma unroll
        for (int t = 0; t < NT / 2; ++t) bnext[t] = (unsigned)min((n * 4 + wave) * (NT / 2) + t, p.wtiles - 1) * (unsigned)(p.K * 64);
    };
    bf16x8 b[4][2][NT], a[AR];
    // rows tid / 8 + 32 i to LDS, without a register between.  The DMA writes lane after lane: a lane fetches the piece that belongs at
    // its place.  In assembly, since the compiler would have every LDS read wait for it; the waits are counted by hand (wait_a)
    auto load_a = [&](unsigned buf, int i) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     : : "s"(buf + (unsigned)(i * 4096 + wave * 1024)), "v"(aoff[i]), "s"(ra), "s"(ka) : "memory", "m0");
    };
    auto load_b = [&](int e, int h, const unsigned (&base)[NT / 2], int n) {
        const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(rw, boff + h * 2048 + (n & 1) * 256, base[n >> 1], 0);
        b[e][h][n] = *reinterpret_cast<const bf16x8*>(&q);
    };
    // ---- LDS addresses
    unsigned raddr[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) raddr[h] = (unsigned)(j * 128 + (((4 * h + kq) ^ ((j >> 1) & 7)) * 16));
    auto read_a = [&](unsigned buf, int h, int t) { a[t % AR] = *reinterpret_cast<const bf16x8*>(lds + (raddr[h] + buf) + t * 2048); };
    f32x4 acc[NT][MT];
    // the products of half h of step e of four, each followed by what `beside` issues there: an order that the compiler keeps
    auto half = [&](int e, int h, auto beside) {
        unrolled(std::make_integer_sequence<int, P>(), [&](int i) __attribute__((always_inline)) {
            const int t = i / NT, n = t & 1 ? NT - 1 - i % NT : i % NT;
            // (in assembly: left to the compiler, accumulators of four registers wander, by 200 moves a step)
            asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[n][t]) : "v"(b[e][h][n]), "v"(a[t % AR]));
            beside(i);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // A of this step, of the next and of the one after it: places in LDS
    unsigned buf0 = 0, buf1 = kBuf, buf2 = 2 * kBuf;
    // step e of four: its products, A of the second and third step ahead, W of the third and fourth
    auto step = [&](auto place_of_four, auto turn) {
        constexpr int e = decltype(place_of_four)::value, o = (e + 3) % 4;
        constexpr int G = MT - AR + 2;                            // groups of products in front of the barrier
        half(e, 0, [&](int i) {
            const int t = i / NT + AR;
            if (i % NT == NT - 1) read_a(buf0, t / MT, t % MT);
            spread(i, P, AL - AH + NT, 1, [&](int x) { if (x < NT) load_b(o, 1, bbase, x); else load_a(buf2, AH + x - NT); });
        });
        turn();
        half(e, 1, [&](int i) {
            const int t = i / NT + AR;
            if (t < MT && i % NT == NT - 1) read_a(buf0, 1, t);
            // Behind the barrier no wavefront reads A of this step any more, and A of the next is there: of the loads in flight at most
            // those of two halves are younger.  It stands where the last LDS instruction lies a few products back
            if (i == G * NT - 1) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NT + AL) : "memory");
                wait_lds_barrier();
            }
            if (i == G * NT || i == G * NT + 1) read_a(buf1, 0, i - G * NT);
            if (i >= G * NT && i % NT == NT - 1) read_a(buf1, 0, t - MT);
            spread(i, G * NT, NT, 1, [&](int x) { load_b(e, 0, bnext, x); });
            spread(i - G * NT, P - G * NT, AH, 1, [&](int x) { load_a(buf0, x); });
        });
        const unsigned done = buf0;
        buf0 = buf1;
        buf1 = buf2;
        buf2 = done;
        asm volatile("" ::: "memory");
    };
    auto advance_b = [&]() {
#pragma unroll
        for (int t = 0; t < NT / 2; ++t) {
            bbase[t] = bnext[t];
            bnext[t] += 4096;
        }
    };
    // ---- what is in flight when the first step begins, in the loop's order: the waits there count the loads behind what they wait for
    auto ask = [&](auto f, int from, int to) {
#pragma unroll
        for (int i = from; i < to; ++i) {
            f(i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    seek_a(first);
    seek_b(first);
    ask([&](int i) { load_a(buf0, i); }, 0, AL);
    ka += kBK * 2;
    ask([&](int i) { load_a(buf1, i); }, 0, AL);
    ask([&](int i) { load_b(0, 0, bnext, i); }, 0, NT);
    ask([&](int i) { load_b(0, 1, bnext, i); }, 0, NT);
    ka += kBK * 2;
#pragma unroll
    for (int e = 1; e < 4; ++e) {
#pragma unroll
        for (int t = 0; t < NT / 2; ++t) bnext[t] += 4096;
        if (e == 3) ask([&](int i) { load_a(buf2, i); }, 0, AH);
        ask([&](int i) { load_b(e, 0, bnext, i); }, 0, NT);
        if (e < 3) ask([&](int i) { load_b(e, 1, bnext, i); }, 0, NT);
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AL + AH + 7 * NT) : "memory");
    wait_lds_barrier();
    ask([&](int i) { read_a(buf0, 0, i); }, 0, AR);

    float act_p = 0.f, act_n = 0.f;
    if constexpr (EPI == PE_XIELU) {
        const Xielu f(p.act);
        act_p = f.ap;
        act_n = f.an;
    }
    for (int v = first; v < p.total; v += grid) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[n][t][r] = 0.f;
        asm volatile("s_nop 7" ::: "memory");
        const int next = v + grid < p.total ? v + grid : first;       // (behind the last tile: rows that exist, and are not used)
        for (int k = 0; k < steps; k += 4) {
            auto turn = [&]() { ka += kBK * 2; };
            advance_b();
            if (__builtin_expect(k == steps - 4, 0)) seek_b(next);
            __builtin_amdgcn_sched_barrier(0);
            step(std::integral_constant<int, 0>(), turn);
            advance_b();
            __builtin_amdgcn_sched_barrier(0);
            step(std::integral_constant<int, 1>(), [&]() {
                ka += kBK * 2;
                if (__builtin_expect(k == steps - 4, 0)) seek_a(next);
                __builtin_amdgcn_sched_barrier(0);
            });
            advance_b();
            __builtin_amdgcn_sched_barrier(0);
            step(std::integral_constant<int, 2>(), turn);
            advance_b();
            __builtin_amdgcn_sched_barrier(0);
            step(std::integral_constant<int, 3>(), turn);
        }
        // (the products are assembly: what the compiler would wait between the last of them and reading its accumulator)
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        // ---- out.  Lane (j, kq) has row j of a row tile and columns 4 kq .. + 3 of each column tile.  The wavefront's columns of 32 rows
        // go through LDS, so that a store writes whole lines (16 bytes of 32 rows each took 9 us a tile)
        int m, n0;
        place(v, m, n0);
        const int rows_left = min(p.M - m * BM, BM);
        const __amdgpu_buffer_rsrc_t rsrc =
            __builtin_amdgcn_make_buffer_rsrc((void*)(p.out + (int64_t)m * BM * p.ldo), (short)0, rows_left * (int)p.ldo * 2, 0x00020000);
        const int col = (n0 * 4 + wave) * CW + (lane % CH) * 8;
        const unsigned at = col < p.Nout ? (unsigned)((lane / CH) * (int)p.ldo + col) * 2 : 0xc0000000u;     // (past the end: not stored)
        auto put = [&](int t) {
            unsigned char* slot = image + (t >> 1 & 1) * (32 * CW * 2);
            const int row = (t & 1) * 16 + j;
            constexpr int OT = GATED ? NT / 2 : NT;
#pragma unroll
            for (int n = 0; n < OT; ++n) {
                float z[4], g[4], o[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(z[r]) : "a"(acc[GATED ? 2 * n : n][t][r]));
                    if constexpr (GATED) asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(g[r]) : "a"(acc[2 * n + 1][t][r]));
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if constexpr (EPI == PE_SWIGLU) {
                        const float h1 = round_bf16(z[r]), h3 = round_bf16(g[r]);
                        o[r] = round_bf16(silu_flat(h1)) * h3;
                    } else if constexpr (EPI == PE_GEGLU) {
                        o[r] = gelu_flat(z[r]) * g[r];
                    } else if constexpr (EPI == PE_XIELU) {
                        o[r] = xielu_flat(act_p, act_n, z[r]);
                    } else if constexpr (EPI == PE_BIAS) {
                        o[r] = z[r] + bf16_to_f32(p.bias[min((n0 * 4 + wave) * CW + n * 16 + kq * 4 + r, p.Nout - 1)]);
                    } else {
                        o[r] = z[r];
                    }
                }
                const int chunk = 2 * n + (kq >> 1);
                *reinterpret_cast<u32x2*>(slot + row * (CW * 2) + ((chunk ^ (row / (16 / CH) & (CH - 1))) * 16) + (kq & 1) * 8) =
                    u32x2{pack2(o[0], o[1]), pack2(o[2], o[3])};
            }
        };
        auto take = [&](int t) {
            const unsigned char* slot = image + (t & 1) * (32 * CW * 2);
#pragma unroll
            for (int i = 0; i < CH / 2; ++i) {
                const int r = lane / CH + i * (64 / CH), c = lane % CH;
                const u32x4 q = *reinterpret_cast<const u32x4*>(slot + r * (CW * 2) + ((c ^ (r / (16 / CH) & (CH - 1))) * 16));
                __builtin_amdgcn_raw_buffer_store_b128(q, rsrc, at + (unsigned)((t * 32 + i * (64 / CH)) * (int)p.ldo * 2), 0, 0);
            }
        };
#pragma unroll
        for (int t = 0; t < MT / 2; ++t) {
            put(2 * t);
            put(2 * t + 1);
            if (t > 0) take(t - 1);
        }
        take(MT / 2 - 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // (the DMA of steps that do not come: not into another workgroup's LDS)
}

// Tiles: rows x columns, and what one takes: us before the first step of 64 and behind the last, us a step while most CUs idle, and how much
// slower that is with all of them busy (the clock).  Drawn from 435 random products (257 to 16 384 rows, 33 weights of 768 x 768 to
// 128 256 x 2 048); the tile that this picks is within 0.5 % of the best on average, 18 % at the worst.
struct Tile {
    int rows, cols;
    double fixed, step, busy;
};
constexpr Tile kTiles[] = {{256, 256, 9.5, 0.906, 1.41}, {192, 256, 8.0, 0.692, 1.41}, {128, 256, 6.4, 0.507, 1.38},
                           {256, 128, 6.2, 0.540, 1.30}, {192, 128, 5.0, 0.434, 1.27}, {128, 128, 3.3, 0.368, 1.10}};

double tile_us(const Tile& t, int M, int64_t cols, int K) {
    const int64_t total = (int64_t)((M + t.rows - 1) / t.rows) * ((cols + t.cols - 1) / t.cols), rounds = total / 256, rest = total % 256;
    const double body = (double)(K / kBK) * t.step;
    double us = (double)rounds * (t.fixed + body * t.busy);
    if (rest) us += t.fixed + body * (1.0 + (t.busy - 1.0) * (double)rest / 256);
    return us;
}

const Tile& best_tile(int M, int64_t cols, int K, double* us) {
    const Tile* best = nullptr;
    for (const Tile& t : kTiles) {
        const double c = tile_us(t, M, cols, K);
        if (!best || c < *us) {
            best = &t;
            *us = c;
        }
    }
    return *best;
}

bool shape_ok(int M, int N, int K, bool gated) {
    const int nout = gated ? N / 2 : N;
    const size_t tiles = gated ? (nout + 15) / 16 : (nout + 31) / 32;
    return M > 0 && N > 0 && (!gated || N % 2 == 0) && nout % 8 == 0 && K >= 4 * kBK && K % (4 * kBK) == 0 && K < (1 << 20) &&
           nout < (1 << 20) && tiles * K * 64 < ((size_t)1 << 32);
}

template <int MT, int NT, int EPI>
int launch_tile(PromptParams& p, hipStream_t st) {
    constexpr int bm = 16 * MT, bn = 64 * NT;
    constexpr bool gated = EPI == PE_SWIGLU || EPI == PE_GEGLU;
    p.mt = (p.M + bm - 1) / bm;
    p.nt = (p.wtiles * 32 + bn - 1) / bn;
    const int groups = (p.mt + kGroup - 1) / kGroup;
    p.group = (p.mt + groups - 1) / groups;                    // (9 row tiles: 5 and 4, not 8 and one that has W to itself)
    p.total = p.mt * p.nt;
    p.per = (std::min(p.total, 256) + 7) / 8;
    constexpr int bytes = 3 * bm * kBK * 2 + 2 * 32 * (gated ? bn / 2 : bn) * 2;      // A's buffers; two images of 32 rows of each wavefront
    static MdPerDeviceOnce once;
    if (once.first() && hipFuncSetAttribute(reinterpret_cast<const void*>(&prompt_gemm_kernel<MT, NT, EPI>),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
        once.undo();
        md_set_error("md_linear_prompt: hipFuncSetAttribute(%d B LDS) failed", bytes);
        return MD_ERR_LAUNCH;
    }
    hipLaunchKernelGGL((prompt_gemm_kernel<MT, NT, EPI>), dim3(8 * p.per), dim3(256), bytes, st, p);
    return MD_OK;
}

template <int EPI>
int launch(PromptParams& p, int rows, int cols, hipStream_t st) {
    if (rows == 256 && cols == 256) return launch_tile<16, 4, EPI>(p, st);
    if (rows == 192 && cols == 256) return launch_tile<12, 4, EPI>(p, st);
    if (rows == 128 && cols == 256) return launch_tile<8, 4, EPI>(p, st);
    if (rows == 256 && cols == 128) return launch_tile<16, 2, EPI>(p, st);
    if (rows == 192 && cols == 128) return launch_tile<12, 2, EPI>(p, st);
    if (rows == 128 && cols == 128) return launch_tile<8, 2, EPI>(p, st);
    md_set_error("md_linear_prompt: no tile of %d x %d", rows, cols);
    return MD_ERR_UNSUPPORTED;
}

}  // namespace

extern "C" double md_linear_prompt_us(int M, int N, int K, int epilogue) {
    if (!shape_ok(M, N, K, epilogue == PE_SWIGLU || epilogue == PE_GEGLU)) {
        md_set_error("md_linear_prompt_us: M=%d N=%d K=%d unsupported", M, N, K);
        return -1.0;
    }
    double us = 0;
    best_tile(M, N, K, &us);
    return us;
}

extern "C" int md_linear_prompt(const void* x, int64_t ldx, const void* w_packed, const void* bias, const float* act, void* out, int64_t ldo,
                                int M, int N, int K, int epilogue, int tile, md_stream_t stream) {
    MD_CHECK_ARG(x && w_packed && out, "md_linear_prompt: null pointer argument");
    const bool gated = epilogue == PE_SWIGLU || epilogue == PE_GEGLU;
    MD_CHECK_ARG(shape_ok(M, N, K, gated), "md_linear_prompt: M=%d N=%d K=%d unsupported", M, N, K);
    PromptParams p;
    p.x = (const bf16_t*)x;
    p.w = (const bf16_t*)w_packed;
    p.bias = (const bf16_t*)bias;
    p.act = act;
    p.out = (bf16_t*)out;
    p.ldx = ldx;
    p.ldo = ldo;
    p.M = M;
    p.K = K;
    p.Nout = gated ? N / 2 : N;
    p.wtiles = gated ? (p.Nout + 15) / 16 : (N + 31) / 32;
    p.w_bytes = (unsigned)((size_t)p.wtiles * K * 64);
    // (32-bit offsets within a row tile: rows of less than 2^20 elements)
    MD_CHECK_ARG(ldx >= K && ldx % 8 == 0 && ldx < (1 << 20) && ldo >= p.Nout && ldo % 8 == 0 && ldo < (1 << 20) &&
                     (((uintptr_t)x | (uintptr_t)out | (uintptr_t)w_packed) & 15) == 0,
                 "md_linear_prompt: x, out and w_packed must be 16-byte aligned, their rows a multiple of 8 and of less than 2^20 elements");
    MD_CHECK_ARG(epilogue == PE_NONE || !bias, "md_linear_prompt: a bias goes with no epilogue only");
    MD_CHECK_ARG((epilogue == PE_XIELU) == (act != nullptr), "md_linear_prompt: act goes with the xIELU epilogue");
    double us = 0;
    const Tile& t = best_tile(M, (int64_t)p.wtiles * 32, K, &us);
    const int rows = tile ? tile / 1000 : t.rows, cols = tile ? tile % 1000 : t.cols;
    hipStream_t st = (hipStream_t)stream;
    int rc;
    switch (epilogue) {
        case PE_NONE: rc = bias ? launch<PE_BIAS>(p, rows, cols, st) : launch<PE_NONE>(p, rows, cols, st); break;
        case PE_SWIGLU: rc = launch<PE_SWIGLU>(p, rows, cols, st); break;
        case PE_XIELU: rc = launch<PE_XIELU>(p, rows, cols, st); break;
        case PE_GEGLU: rc = launch<PE_GEGLU>(p, rows, cols, st); break;
        default: md_set_error("md_linear_prompt: unknown epilogue %d", epilogue); return MD_ERR_INVALID_ARG;
    }
    if (rc != MD_OK) return rc;
    MD_CHECK_LAUNCH("md_linear_prompt");
    return MD_OK;
}
