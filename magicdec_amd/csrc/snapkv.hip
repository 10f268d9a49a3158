// SnapKV select for gfx950.
//
// reference: Attention.gen_draft_kv  Engine/SnapKV/model.py:389-439
// restated (bit-exact vs the reference on CPU) in oracle/magicdec_ref.py:snapkv_scores.
//
// Rounding sequence reproduced (g = H/KH, W = window, S = ctx_len, L = g*W rows
// per kv head ordered (r,l)):
//   for each chunk of 8g rows:  s = bf16(q.k)  (UNSCALED);  the last W rows x last
//   W columns of the chunk get the WxW causal mask;  p = bf16(softmax_fp32(s));
//   rows regrouped (r'=g, l'=8): gs = bf16(sum_l' p[..., :S-W]);  acc[r'] = bf16(acc[r'] + gs)
//   pooled = bf16(avg_pool1d(acc, k, pad k/2, /k));  score = bf16(sum_r' pooled)
//   indices = top-(budget-W) of score, descending score, ties -> lowest index
//   draft rows = K,V[indices] ++ K,V[S-W:S]
//
// Five small launches, none on the timed decode path (once per prefill per layer):
//   stats   : the table of exponentials (below); row max / sum-exp partials per column chunk   (MFMA scores; float64 sums)
//   finalize: per-row (max, 1 / sum) of the whole context from the chunk partials, where those are many
//   accum   : recompute scores, p, 8-row group sums, bf16 chunk accumulation
//   pool    : pool + group sum
//   select  : exact radix select, ranked by counting (one WG per b,kvh)
//   gather  : copy the selected rows into the draft pages
#include "md_common.h"

#include <type_traits>
#include <utility>

namespace {

template <int... I, class F>
__device__ __forceinline__ void unrolled(std::integer_sequence<int, I...>, F f) {
    (f(std::integral_constant<int, I>()), ...);
}

struct SnapParams {
    const bf16_t* q;      // [B*W, H, D]
    const void* cache;    // paged full KV (bf16, or e4m3fn bytes with per-head scales)
    const float* k_scale;
    const int32_t* page_indices;
    const int32_t* page_indptr;
    double* partials;       // [B*KH][L][nch][2] = (row max, sum of exp) per `cols` columns, float64
    unsigned short* aws;    // [B][H][S-W] bf16 bits
    int B, H, KH, g, W, S, L, nch, page_size;
    int cols;             // columns per workgroup of the two score kernels
    int64_t page_stride;
    int slot_stride;      // elements between rows of a page: KH*D (NHD) or D (HND)
    int head_stride;      // elements between kv heads: D (NHD) or page_size*D (HND)
};

// K fragment (A operand) of 16 consecutive columns (kv positions) col0..col0+15 for head kvh:
// lane (lq,lc) holds K[col0+lq][ks*32 + lc*8 .. +8]
template <int D, bool FP8>
__device__ __forceinline__ void load_kfrag(const SnapParams& p, int b, int kvh, int col0, int lq, int lc,
                                           bf16x8 (&kf)[D / 32]) {
    const int col = col0 + lq;
    const bf16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
    if (col < p.S) {
        const int page = col / p.page_size, slot = col - page * p.page_size;
        const int64_t pid = p.page_indices[p.page_indptr[b] + page];
        const int64_t off = pid * p.page_stride + (int64_t)slot * p.slot_stride + (int64_t)kvh * p.head_stride + lc * 8;   // elements
        if constexpr (FP8) {
            const unsigned char* kp = reinterpret_cast<const unsigned char*>(p.cache) + off;
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) {
                const u32x2 w = *reinterpret_cast<const u32x2*>(kp + ks * 32);   // 8 e4m3fn bytes -> 8 bf16 (exact)
                bf16x8 r;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[h], 1.0f, false);
                    const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[h], 1.0f, true);
                    r[4 * h] = a[0];
                    r[4 * h + 1] = a[1];
                    r[4 * h + 2] = c[0];
                    r[4 * h + 3] = c[1];
                }
                kf[ks] = r;
            }
        } else {
            const bf16_t* kp = reinterpret_cast<const bf16_t*>(p.cache) + off;
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) kf[ks] = *reinterpret_cast<const bf16x8*>(kp + ks * 32);
        }
    } else {
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) kf[ks] = z;
    }
}

// The fragments of 32 or 64 consecutive columns (NC 16-column groups).  Pages of a multiple of 32 rows hold all of them in one page, which is
// then looked up once per wavefront; rows past the context are not read from beyond it (zeros).
template <int D, bool FP8, int NC>
__device__ __forceinline__ void load_kfrags(const SnapParams& p, int b, int kvh, int col0, bool whole, int lq, int lc,
                                            bf16x8 (&kf)[NC][D / 32]) {
#pragma unroll
    for (int g = 0; g < NC; g += 2) {
        const int at = col0 + g * 16;
        if (!FP8 && whole && at + 32 <= p.S) {
            const int page = at / p.page_size;
            const int64_t pid = p.page_indices[p.page_indptr[b] + page];
            const bf16_t* kp = reinterpret_cast<const bf16_t*>(p.cache) + pid * p.page_stride +
                               (int64_t)(at - page * p.page_size) * p.slot_stride + (int64_t)kvh * p.head_stride;
            const unsigned off = (unsigned)(lq * p.slot_stride + lc * 8);
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int ks = 0; ks < D / 32; ++ks)
                    kf[g + c][ks] = *reinterpret_cast<const bf16x8*>(kp + (int64_t)c * 16 * p.slot_stride + off + ks * 32);
        } else {
            load_kfrag<D, FP8>(p, b, kvh, at, lq, lc, kf[g]);
            load_kfrag<D, FP8>(p, b, kvh, at + 16, lq, lc, kf[g + 1]);
        }
    }
}

// exp(x) for x <= 0 in float64, ~1 ulp: k = rint(x log2 e), r = x - k ln2 (two-part constant), degree-13 Taylor polynomial
// (|r| <= 0.347: remainder 4e-18), scaled by 2^k -- 17 dependent f64 instructions instead of OCML's exp().
__device__ __forceinline__ double exp_neg(double x) {
    if (!(x > -700.0)) return 0.0;                       // -inf (masked) and anything that underflows anyway
    const double k = rint(x * 1.4426950408889634074);
    double r = fma(-k, 6.93147180369123816490e-01, x);
    r = fma(-k, 1.90821492927058770002e-10, r);
    double q = 1.0 / 6227020800.0;
    q = fma(q, r, 1.0 / 479001600.0);
    q = fma(q, r, 1.0 / 39916800.0);
    q = fma(q, r, 1.0 / 3628800.0);
    q = fma(q, r, 1.0 / 362880.0);
    q = fma(q, r, 1.0 / 40320.0);
    q = fma(q, r, 1.0 / 5040.0);
    q = fma(q, r, 1.0 / 720.0);
    q = fma(q, r, 1.0 / 120.0);
    q = fma(q, r, 1.0 / 24.0);
    q = fma(q, r, 1.0 / 6.0);
    q = fma(q, r, 0.5);
    q = fma(q, r, 1.0);
    q = fma(q, r, 1.0);
    return ldexp(q, (int)k);
}

// ---- the softmax of the select without a float64 exponential per element.
// The reference's scores are bf16 VALUES (model.py:411: a bf16 einsum), i.e. one of 65 536 numbers, and the
// probabilities must be correctly rounded bf16(exp(s - M) / Z) (see "Rounding sequence" above: an fp32 evaluation with
// another summation order flips ~1e-4 of those roundings).  exp() in float64 per element is a billion OCML calls per
// layer for 64 requests of 16 000 tokens, 0.21 TB/s of K bytes = 2.6 % of the HBM peak.  So exp(v) of every bf16 value with 2^-23 <= |v| < 2^9 sits in a float64 table in LDS (filled with OCML's exp once
// per call): the row sum is  sum_i T[s_i]  (reference 0: e^512 * 65 536 columns is far below the float64 range) and a
// probability is  T[s] * (exp(-M) / Z)  -- one LDS gather and one f64 multiply.  Of the few scores outside the table, tiny
// ones are a short polynomial, the others (|s| >= 512, masked) take the lean exp_neg() above against a running maximum, so
// nothing overflows whatever the raw (unscaled) scores are.
// The UNSCALED q.k of a seeded-random 1B layer is ~N(0, 6.5^2) and a trained checkpoint's reaches the hundreds: the table covers 32
// binades x 128 mantissas x 2 signs = 8 192 entries = 64 KB, laid out [magnitude][sign] so that the byte offset of a score is
// (magnitude index << 4) | (sign << 3) and still fits 16 bits.  One score in 10^8 of N(0, 6.5^2) is smaller than that; with 2^-14 as the
// smallest it was one in 10^5, and one batch of 1 024 in 130 left the hot path.  Kernels whose query image leaves no room take the
// upper 23 binades.
constexpr int kTabE0 = 104;                 // biased bf16 exponent of 2^-23
constexpr int kTabBinades = 32;             // 2^-23 .. 2^9
constexpr int kTabMag = kTabBinades * 128;  // magnitude indices: (exponent - E0) * 128 + mantissa
constexpr int kTabN = 2 * kTabMag;          // [magnitude][sign]
constexpr int kTabSmall = 23;               // binades of the small table
__device__ __attribute__((aligned(16))) double g_exp_tab[kTabN];
template <int BIN> struct Tab {             // BIN binades up to 2^9
    static constexpr int E0 = kTabE0 + kTabBinades - BIN, N = BIN * 256;
};

// Filled by every workgroup of the first pass for itself (8 exponentials a thread: 2 us, where a launch in front took 4.5) and left by
// its first one for the second pass: the same bytes in every call.
template <int BIN>
__device__ __forceinline__ void fill_table(double* tab, int tid, int nthr, bool leave) {
    for (int i = tid; i < kTabN; i += nthr) {
        const int at = i - (kTabN - Tab<BIN>::N);
        if (at < 0 && !leave) continue;
        const unsigned int bits = ((unsigned int)(i & 1) << 15) | (unsigned int)((i >> 1) + (kTabE0 << 7));
        const double e = exp((double)bf16_bits_to_f32((unsigned short)bits));
        if (at >= 0) tab[at] = e;
        if (leave) g_exp_tab[i] = e;
    }
}
template <int BIN>
__device__ __forceinline__ void load_table(double* tab, int tid, int nthr) {
    const u32x4* from = reinterpret_cast<const u32x4*>(g_exp_tab + (kTabN - Tab<BIN>::N));
#pragma unroll 4
    for (int i = tid; i < Tab<BIN>::N / 2; i += nthr) reinterpret_cast<u32x4*>(tab)[i] = from[i];
}

// exp(v) for |v| < 2^-14: the next term is below 2^-60
__device__ __forceinline__ double exp_tiny(float v) {
    const double x = (double)v;
    return fma(x, fma(x, fma(x, 1.0 / 6.0, 0.5), 1.0), 1.0);
}
__device__ __forceinline__ bool is_tiny(float v) { return fabsf(v) < 6.103515625e-05f; }

// table index of a bf16 value held in a float, or -1 (outside the table: tiny, large, zero, inf)
template <int BIN>
__device__ __forceinline__ int tab_index(float s) {
    const unsigned int bits = __float_as_uint(s) >> 16;
    const unsigned int a = (bits & 0x7fffu) - ((unsigned int)Tab<BIN>::E0 << 7);
    return a < (unsigned int)(BIN * 128) ? (int)((a << 1) | (bits >> 15)) : -1;
}

// Two scores at a time: `w` = two bf16 values in one dword (v_cvt_pk_bf16_f32).  With d = bits - (E0 << 7) a score in the table has
// magnitude index d & 0x7fff < 4096, so that rotating d left by four gives its byte offset (magnitude x 16 + sign x 8); any
// other d leaves one of the low three bits set, or (small table) an offset past the last entry.  `top` (maximum) and `low` (or) collect
// both over a batch of scores: tab_outside says whether all of them lie inside.
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned int pack_bf16(float a, float b) {
    return __builtin_bit_cast(unsigned int, __builtin_convertvector((f32x2{a, b}), bf16x2));
}
// The same where the halves are taken apart again, which the compiler would convert one by one.  (Not for a matrix product's result: the
// compiler does not see the wait that assembly behind one needs)
__device__ __forceinline__ unsigned int round_pair(float a, float b) {
    unsigned int pk;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(pk) : "v"(a), "v"(b));
    return pk;
}
// both to bf16 and back (they may be one and the same)
__device__ __forceinline__ void round2(float& a, float& b) {
    const unsigned int pk = round_pair(a, b);
    a = __uint_as_float(pk << 16);
    if (&a != &b) b = __uint_as_float(pk & 0xffff0000u);
}
template <int BIN>
__device__ __forceinline__ unsigned int tab_offsets2(unsigned int w, u16x2& top, unsigned int& low) {
    const u16x2 d = *reinterpret_cast<const u16x2*>(&w) - (unsigned short)(Tab<BIN>::E0 << 7);
    const u16x2 turned = d >> (unsigned short)12;
    u16x2 r;
    asm("v_pk_mad_u16 %0, %1, %2, %3" : "=v"(r) : "v"(d), "s"(0x00100010u), "v"(turned));      // (left alone: a shift and an or)
    if constexpr (BIN < kTabBinades) top = __builtin_elementwise_max(top, r);
    const unsigned int o = *reinterpret_cast<const unsigned int*>(&r);
    low |= o;
    return o;
}
template <int BIN>
__device__ __forceinline__ bool tab_outside(u16x2 top, unsigned int low) {
    return (low & 0x00070007u) != 0 || (BIN < kTabBinades && (top[0] >= Tab<BIN>::N * 8 || top[1] >= Tab<BIN>::N * 8));
}
__device__ __forceinline__ double tab_at(const double* tab, unsigned int offset) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const unsigned char*>(tab) + offset);
}

// (m, Z) <- merge of two partial softmax sums  sum exp(s - m)
__device__ __forceinline__ void merge_mz(double& m, double& Z, double m2, double Z2) {
    if (m2 == m) {                                       // the common case: both sums with reference 0
        Z += Z2;
        return;
    }
    const double mn = fmax(m, m2);
    if (!(mn > -INFINITY)) return;
    Z = (m > -INFINITY ? Z * exp_neg(m - mn) : 0.0) + (m2 > -INFINITY ? Z2 * exp_neg(m2 - mn) : 0.0);
    m = mn;
}

constexpr int kQPad = 16;                   // bytes of padding per row of the Q image in LDS
constexpr int kMaxRT = 16;                  // 16-row tiles per kv head: L = g * W <= 256

// Q rows of one (request, kv head), ordered (r, l), into LDS: row rg at rg * (2 D + 16) bytes.  An odd number of 16-row tiles: the last one
// twice, so that tiles come in twos
__host__ __device__ constexpr int image_rows(int L) { return (L + 31) / 32 * 32; }
template <int D>
__device__ __forceinline__ void load_q_image(const SnapParams& p, int b, int kvh, unsigned char* qimg, int tid, int nthr) {
    constexpr int CH = D * 2 / 16;
    for (int c = tid; c < image_rows(p.L) * CH; c += nthr) {
        const int at = c / CH, ch = c - at * CH, rg = at < p.L ? at : at - 16;
        const int r = rg / p.W, l = rg - r * p.W;
        const u32x4 v = *reinterpret_cast<const u32x4*>(p.q + ((int64_t)(b * p.W + l) * p.H + kvh * p.g + r) * D + ch * 8);
        *reinterpret_cast<u32x4*>(qimg + at * (D * 2 + kQPad) + ch * 16) = v;
    }
}

// is (row rg, column col) masked?  The last W rows of every 8g-row chunk x the last W columns carry the W x W causal mask
// of the reference (model.py:412-415, mis-aligned on purpose: bug-for-bug)
__device__ __forceinline__ bool masked(int S, int W, int chunk_rows, int rg, int col) {
    const int mrow = rg % chunk_rows - (chunk_rows - W);
    return col >= S || (mrow >= 0 && col - (S - W) > mrow);
}

// Wavefronts of a workgroup of the two score kernels, which share the table and the Q image: what a CU can hold.
constexpr int score_waves(int D, int rt) { return D == 64 && rt <= 8 ? 16 : 8; }

constexpr int stats_binades(int D, int rt) { return D == 128 && rt > 8 ? kTabSmall : kTabBinades; }

// One row's scores of a batch where some lie outside the table or may be masked: w = columns col .. + 3 and col + 16 .. + 19.  Returns the sum
// of exponentials against 0; those outside go to the wavefront's (m, Z) pair of the row, the four lanes of a row in turns.
// (A call: in line it costs the hot path ten registers that it spills.)
typedef __attribute__((address_space(3))) double lds_double;
template <int BIN>
__device__ __noinline__ double stats_slow(const lds_double* tab, lds_double* pair, unsigned int w0, unsigned int w1, unsigned int w2, unsigned int w3, int S, int W,
                                          int chunk_rows, int rg, int col, int lc, bool tail) {
    double m2 = -INFINITY, z2 = 0.0, t = 0.0;
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {
        const unsigned int w = i < 4 ? (i < 2 ? w0 : w1) : (i < 6 ? w2 : w3);
        const float v = bf16_bits_to_f32((unsigned short)(i & 1 ? w >> 16 : w & 0xffffu));
        if (tail && masked(S, W, chunk_rows, rg, col + (i >> 2) * 16 + (i & 3))) continue;      // (an integer modulo: off the hot path)
        const int ti = tab_index<BIN>(v);
        if (ti >= 0)
            t += tab[ti];
        else if (is_tiny(v))
            t += exp_tiny(v);
        else if (v > -INFINITY)
            merge_mz(m2, z2, (double)v, 1.0);
    }
#pragma unroll 1
    for (int q = 0; q < 4; ++q) {
        if (lc == q && m2 > -INFINITY) {
            double m = pair[0], Z = pair[1];
            merge_mz(m, Z, m2, z2);
            pair[0] = m;
            pair[1] = Z;
        }
        __builtin_amdgcn_wave_barrier();
    }
    return t;
}
// Two rows' probabilities of one column likewise, as two bf16
template <int BIN>
__device__ __noinline__ unsigned int accum_slow(const lds_double* tab, const lds_double* rowc, const lds_double* rowm, unsigned int w, int S, int W, int chunk_rows,
                                                int row, int col, bool tail) {
    float pr[2] = {0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const float v = bf16_bits_to_f32((unsigned short)(e ? w >> 16 : w & 0xffffu));
        if (!(tail && masked(S, W, chunk_rows, row + e, col))) {
            const int ti = tab_index<BIN>(v);
            const double c2 = rowc[row + e];
            if ((ti >= 0 || is_tiny(v)) && c2 > 0.0)
                pr[e] = (float)((ti >= 0 ? tab[ti] : exp_tiny(v)) * c2);
            else
                pr[e] = (float)(exp_neg((double)v - rowm[(row + e) * 2]) * rowm[(row + e) * 2 + 1]);
        }
    }
    return pack_bf16(pr[0], pr[1]);
}

// Pass 1: per (row, column chunk) the pair (m, Z), Z = sum over the chunk's columns of exp(s - m).  A lane owns ONE row
// of every 16-row tile (rows <-> lanes lq) and 4 of a tile's 16 columns, and keeps the table sum of each of its rows
// (reference 0) in registers: no cross-lane traffic until the end.  Out-of-table scores (rare) go to a per-wave (m, Z)
// pair per row in LDS.  A wavefront takes 2 x 2 tiles at a time: two column groups share the query fragments, and the 16 table
// gathers of a lane are in flight together.  16 requests of 16 000 keys (8 kv heads of 64, 128 rows each): 92 us; 120 in two workgroups of
// eight wavefronts a CU, each with its own table and image (12 us to fill), with the rare scores in line (spills) and 23 binades (0.8 % of
// the batches are rare then); 150 tile by tile.  Bound by LDS, active for 68 % of the cycles: 4 gathers of 8 random bytes per lane and
// tile, about 7 cycles each, beside 8 for the fragments; vector instructions 47 %.
template <int D, bool FP8, int RTM>     // RTM: register-resident 16-row tiles (8 for g * W <= 128 rows, else kMaxRT)
__global__ __launch_bounds__(64 * score_waves(D, RTM), score_waves(D, RTM) / 4) void snapkv_stats_kernel(const SnapParams p) {
    constexpr int kSnapWaves = score_waves(D, RTM), BIN = stats_binades(D, RTM);
    __shared__ __attribute__((aligned(16))) double tab[Tab<BIN>::N];
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn[];   // Q image, then [waves][L][2] doubles
    const int chunk = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 15, lc = lane >> 4;
    unsigned char* qimg = dyn;
    double* ms = reinterpret_cast<double*>(dyn + (size_t)image_rows(p.L) * (D * 2 + kQPad));
    double* sw = ms + (size_t)wave * p.L * 2;                 // this wave's (m, Z) of the out-of-table scores, per row
    fill_table<BIN>(tab, tid, 64 * kSnapWaves, (chunk | kvh | b) == 0);
    load_q_image<D>(p, b, kvh, qimg, tid, 64 * kSnapWaves);
    for (int i = lane; i < p.L; i += 64) {
        sw[i * 2] = -INFINITY;
        sw[i * 2 + 1] = 0.0;
    }
    __syncthreads();
    const int RT = p.L / 16;
    const bool whole = p.page_size % 32 == 0;
    const float kscale = FP8 ? p.k_scale[kvh] : 1.0f;
    double zt[RTM];
#pragma unroll
    for (int rt = 0; rt < RTM; ++rt) zt[rt] = 0.0;
    const int ncg = (min(p.cols, p.S - chunk * p.cols) + 31) / 32;                   // 32-column groups of this chunk
    bf16x8 kf[2][D / 32], kn[2][D / 32];
    if (wave < ncg) load_kfrags<D, FP8>(p, b, kvh, chunk * p.cols + wave * 32, whole, lq, lc, kf);
    for (int cg = wave; cg < ncg; cg += kSnapWaves) {
        const int col0 = chunk * p.cols + cg * 32;
        if (cg + kSnapWaves < ncg) load_kfrags<D, FP8>(p, b, kvh, col0 + kSnapWaves * 32, whole, lq, lc, kn);
        const bool tail = col0 + 32 > p.S - p.W;                     // wave-uniform: only these columns can be masked
#pragma unroll
        for (int r0 = 0; r0 < RTM; r0 += 2) {
            if (r0 < RT) {                                           // wave-uniform
                const bool two = r0 + 1 < RT;
                unsigned int w[2][2][2];                             // scores rounded to bf16, two per dword: [row tile][column group]
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const unsigned char* qp = qimg + lq * (D * 2 + kQPad) + lc * 16 + (r0 + u) * 16 * (D * 2 + kQPad);
                    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
                    for (int ks = 0; ks < D / 32; ++ks) {
                        const bf16x8 qf = *reinterpret_cast<const bf16x8*>(qp + ks * 64);
#pragma unroll
                        for (int c = 0; c < 2; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[c][ks], qf, acc[c], 0, 0, 0);
                    }
                    // lane (lq, lc): row rt*16 + lq, columns col0 + c*16 + lc*4 + j
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        if (FP8) acc[c] *= kscale;
                        w[u][c][0] = pack_bf16(acc[c][0], acc[c][1]);
                        w[u][c][1] = pack_bf16(acc[c][2], acc[c][3]);
                    }
                }
                u16x2 top = {0, 0};
                unsigned int low = 0, o[2][2][2];
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int c = 0; c < 2; ++c)
#pragma unroll
                        for (int h = 0; h < 2; ++h) o[u][c][h] = tab_offsets2<BIN>(w[u][c][h], top, low);
                // hot path, no divergence: every score of the batch is in the table and no column can be masked
                if (!tail && __builtin_amdgcn_ballot_w64(tab_outside<BIN>(top, low)) == 0) {
                    double e[2][2][4];
#pragma unroll
                    for (int u = 0; u < 2; ++u)
#pragma unroll
                        for (int c = 0; c < 2; ++c)
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                e[u][c][j] = tab_at(tab, j & 1 ? o[u][c][j >> 1] >> 16 : o[u][c][j >> 1] & 0xffffu);
#pragma unroll
                    for (int u = 0; u < 2; ++u)
#pragma unroll
                        for (int c = 0; c < 2; ++c) {
                            const double t = (e[u][c][0] + e[u][c][1]) + (e[u][c][2] + e[u][c][3]);
                            if (u == 0 || two) zt[r0 + u] += t;
                        }
                } else {
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        if (u == 1 && !two) continue;
                        const int rg = (r0 + u) * 16 + lq;
                        zt[r0 + u] += stats_slow<BIN>((lds_double*)tab, (lds_double*)(sw + rg * 2), w[u][0][0], w[u][0][1], w[u][1][0], w[u][1][1], p.S, p.W, 8 * p.g, rg,
                                                      col0 + lc * 4, lc, tail);
                    }
                }
            }
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) kf[c][ks] = kn[c][ks];
    }
    // per-lane -> per-row of this wave (the 4 lanes lq + 16 lc of a row), then over the waves, then out
#pragma unroll
    for (int rt = 0; rt < RTM; ++rt) {
        if (rt < RT) {
            double Z = zt[rt];
            Z += __shfl_xor(Z, 16);
            Z += __shfl_xor(Z, 32);
            if (lc == 0) {
                const int rg = rt * 16 + lq;
                double m = Z > 0.0 ? 0.0 : -INFINITY;
                if (sw[rg * 2] > -INFINITY) merge_mz(m, Z, sw[rg * 2], sw[rg * 2 + 1]);
                sw[rg * 2] = m;
                sw[rg * 2 + 1] = Z;
            }
        }
    }
    __syncthreads();
    for (int row = tid; row < p.L; row += 64 * kSnapWaves) {
        double M = -INFINITY, Z = 0.0;
        for (int w = 0; w < kSnapWaves; ++w) merge_mz(M, Z, ms[(w * p.L + row) * 2], ms[(w * p.L + row) * 2 + 1]);
        double* out = p.partials + (((int64_t)(b * p.KH + kvh) * p.L + row) * p.nch + chunk) * 2;
        out[0] = M;
        out[1] = Z;
    }
}

// Row statistics of the whole context from the per-chunk partials, once per row: (M, 1 / Z) overwrite chunk 0's slot.  Of a few chunks
// every workgroup of the second pass makes them for itself (a launch is 4.8 us).
constexpr int kFewChunks = 8;
__global__ __launch_bounds__(256) void snapkv_finalize_kernel(const SnapParams p) {
    const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (row >= (int64_t)p.B * p.KH * p.L) return;
    double* pp = p.partials + row * p.nch * 2;
    double M = -INFINITY, Z = 0.0;
    for (int c = 0; c < p.nch; ++c) merge_mz(M, Z, pp[c * 2], pp[c * 2 + 1]);
    pp[0] = M;
    pp[1] = 1.0 / Z;
}

// Pass 2: p = bf16(exp(s - M) / Z), 8-row group sums in fp32 -> bf16, bf16 accumulation over the row chunks in order.
// Rows <-> REGISTERS here (A = Q fragment, B = K fragment: lane (lq, lc) holds rows 16 rt + 4 lc + j of column lq), so an
// 8-row group sum is three adds in a lane and one exchange between neighbouring groups of 16 lanes, in the reference's pairwise order.
// Group G = 2 rt + half (lanes lc = 2 half) belongs to chunk G / g and pseudo head r' = G % g.  For even g a lane meets the same half
// in every tile, so the accumulators r' = 2 i + half are its registers a[x][i] (template GH = g / 2, else 0: accumulators in LDS, updated
// by the two halves in turn).  After the exchange a lane keeps one of two column groups' sums, so that one rounding serves two sums.
// NC column groups share a row tile's fragments and factors: four where a wavefront's 64 columns come out even (`four` below), the next
// ones' keys then loaded behind the last row tile's products.  16 requests of 16 000 keys, as above: 109 us; 124 on the same card with two
// row tiles of two column groups, both of whose sums every lane kept.  Bound by vector issue and LDS in turn: vector
// instructions for 70 % of the cycles, LDS active for 58 % (37 of them bank conflicts of the random gathers).  (A table of floats, and the
// float64 product only where rounding is in doubt: 4 bytes at random cost what 8 do, 118 against 123; the scores a batch ahead of the
// gathers: 118 / 118.)
// BIN: the table's binades; all, but where the accumulators of 30 and 32 queries a kv head of 128 beside them would pass a CU's LDS.
template <int D, bool FP8, int GH, int RTM, int NC, int BIN = kTabBinades>
__global__ __launch_bounds__(64 * score_waves(D, RTM), score_waves(D, RTM) / 4) void snapkv_accum_kernel(const SnapParams p) {
    constexpr int kSnapWaves = score_waves(D, RTM);
    constexpr int BT = GH >= 2 && NC == 2 ? 2 : 1, NG = NC / 2, COLS = NC * 16;      // row tiles per batch; column groups of a lane
    __shared__ __attribute__((aligned(16))) double tab[Tab<BIN>::N];
    // Q image, [L] exp(-M) / Z, [L][2] (M, 1 / Z), GH == 0: [waves][g][32] floats
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn[];
    const int ctile = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 15, lc = lane >> 4;
    unsigned char* qimg = dyn;
    double* rowc = reinterpret_cast<double*>(dyn + (size_t)image_rows(p.L) * (D * 2 + kQPad));
    double* rowm = rowc + p.L;
    float* accs = reinterpret_cast<float*>(rowm + p.L * 2) + wave * p.g * 32;
    __shared__ int s_slow_rows;
    if (tid == 0) s_slow_rows = 0;
    load_table<BIN>(tab, tid, 64 * kSnapWaves);
    load_q_image<D>(p, b, kvh, qimg, tid, 64 * kSnapWaves);
    __syncthreads();
    for (int row = tid; row < p.L; row += 64 * kSnapWaves) {
        const double* pp = p.partials + ((int64_t)(b * p.KH + kvh) * p.L + row) * p.nch * 2;
        double M = pp[0], rZ = pp[1];                         // left by snapkv_finalize_kernel, or still one of a few chunks'
        if (p.nch <= kFewChunks) {
            for (int c = 1; c < p.nch; ++c) merge_mz(M, rZ, pp[c * 2], pp[c * 2 + 1]);
            rZ = 1.0 / rZ;
        }
        rowm[row * 2] = M;
        rowm[row * 2 + 1] = rZ;
        double c2 = 0.0;                                      // 0: exp(-M) is not representable -> the exp_neg path
        if (M >= 0.0) c2 = exp_neg(-M) * rZ;
        else if (M > -700.0) c2 = rZ / exp_neg(M);
        rowc[row] = c2;
        if (!(c2 > 0.0)) s_slow_rows = 1;
    }
    __syncthreads();
    const bool fast_rows = s_slow_rows == 0;                  // workgroup-uniform
    const int N = p.S - p.W;
    const bool whole = p.page_size % 32 == 0;
    const float kscale = FP8 ? p.k_scale[kvh] : 1.0f;
    const int ncg = (min(p.cols, N - ctile * p.cols) + COLS - 1) / COLS;             // column groups of this workgroup
    bf16x8 kf[NC][D / 32], kn[NC == 2 ? 2 : 1][D / 32];
    if (wave < ncg) load_kfrags<D, FP8>(p, b, kvh, ctile * p.cols + wave * COLS, whole, lq, lc, kf);
    for (int cg = wave; cg < ncg; cg += kSnapWaves) {
        const int col0 = ctile * p.cols + cg * COLS;
        const bool more = cg + kSnapWaves < ncg;
        if (NC == 2 && more) load_kfrags<D, FP8>(p, b, kvh, col0 + kSnapWaves * COLS, whole, lq, lc, kn);
        const bool tail = col0 + COLS > p.S - p.W;             // wave-uniform: only these columns can be masked
        float a[NG][GH > 0 ? GH : 1];                          // [column group 2 x + (lc & 1)][i], bf16 values
        if constexpr (GH > 0) {
#pragma unroll
            for (int x = 0; x < NG; ++x)
#pragma unroll
                for (int i = 0; i < GH; ++i) a[x][i] = 0.f;
        } else {
            for (int i = lane; i < p.g * 32; i += 64) accs[i] = 0.f;
            __builtin_amdgcn_wave_barrier();
        }
        // group sums of the BT row tiles from rt on: lanes lc < 2 have group 2 rt, the others 2 rt + 1, of column groups 2 x + (lc & 1)
        auto sums = [&](int rt, float (&gs)[BT][NG]) {
            unsigned int w[BT][NC][2];
#pragma unroll
            for (int u = 0; u < BT; ++u) {
                const unsigned char* qp = qimg + ((rt + u) * 16 + lq) * (D * 2 + kQPad) + lc * 16;
                f32x4 acc[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < D / 32; ++ks) {
                    const bf16x8 qf = *reinterpret_cast<const bf16x8*>(qp + ks * 64);
#pragma unroll
                    for (int c = 0; c < NC; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf, kf[c][ks], acc[c], 0, 0, 0);
                }
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    if (FP8) acc[c] *= kscale;
                    w[u][c][0] = pack_bf16(acc[c][0], acc[c][1]);
                    w[u][c][1] = pack_bf16(acc[c][2], acc[c][3]);
                }
            }
            // the next columns' fragments in the place of these, while the last row tiles' gathers and sums go on
            if (NC == 4 && more && rt + BT == p.L / 16) load_kfrags<D, FP8>(p, b, kvh, col0 + kSnapWaves * COLS, whole, lq, lc, kf);
            u16x2 top = {0, 0};
            unsigned int low = 0, o[BT][NC][2], pk[BT][NC][2];
#pragma unroll
            for (int u = 0; u < BT; ++u)
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int h = 0; h < 2; ++h) o[u][c][h] = tab_offsets2<BIN>(w[u][c][h], top, low);
            if (fast_rows && !tail && __builtin_amdgcn_ballot_w64(tab_outside<BIN>(top, low)) == 0) {
                // hot path, no divergence: table value x the row's exp(-M) / Z, softmax -> bf16 (model.py:416)
#pragma unroll
                for (int u = 0; u < BT; ++u) {
                    const double* rc = rowc + (rt + u) * 16 + lc * 4;
                    const double c2[4] = {rc[0], rc[1], rc[2], rc[3]};
#pragma unroll
                    for (int c = 0; c < NC; ++c)
#pragma unroll
                        for (int h = 0; h < 2; ++h)
                            pk[u][c][h] = round_pair((float)(tab_at(tab, o[u][c][h] & 0xffffu) * c2[2 * h]),
                                                    (float)(tab_at(tab, o[u][c][h] >> 16) * c2[2 * h + 1]));
                }
            } else {
#pragma unroll
                for (int u = 0; u < BT; ++u)
#pragma unroll
                    for (int c = 0; c < NC; ++c)
#pragma unroll
                        for (int h = 0; h < 2; ++h)
                            pk[u][c][h] = accum_slow<BIN>((lds_double*)tab, (lds_double*)rowc, (lds_double*)rowm, w[u][c][h], p.S, p.W, 8 * p.g, (rt + u) * 16 + lc * 4 + 2 * h,
                                                          col0 + c * 16 + lq, tail);
            }
            // 8-row group sum in fp32, pairwise as a butterfly over consecutive rows, -> bf16 (:418)
#pragma unroll
            for (int u = 0; u < BT; ++u)
#pragma unroll
                for (int x = 0; x < NG; ++x) {
                    float t[2];
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        const unsigned int v = pk[u][2 * x + c][0], y = pk[u][2 * x + c][1];
                        t[c] = (__uint_as_float(v << 16) + __uint_as_float(v & 0xffff0000u)) +
                               (__uint_as_float(y << 16) + __uint_as_float(y & 0xffff0000u));
                    }
                    // the one column group's odd 16 lanes against the other's even ones: a lane then has both halves of one group's sum
                    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(t[0]), __float_as_uint(t[1]), false, false);
                    gs[u][x] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
                }
            round2(gs[0][0], gs[BT - 1][NG - 1]);
        };
        if constexpr (GH > 0) {
            for (int rt = 0; rt < p.L / 16; rt += GH)          // one chunk of 8 g rows
                unrolled(std::make_integer_sequence<int, GH / BT>(), [&](auto ic) {      // (accumulators in registers: not a loop)
                    constexpr int i = decltype(ic)::value * BT;
                    float gs[BT][NG];
                    sums(rt + i, gs);
#pragma unroll
                    for (int u = 0; u < BT; ++u)
#pragma unroll
                        for (int x = 0; x < NG; ++x) a[x][i + u] += gs[u][x];
                    round2(a[0][i], a[NG - 1][i + BT - 1]);
                });
            // bf16 accumulators: aws[b][kvh*g + r'][col]; lane (lq, lc): half lc / 2
#pragma unroll
            for (int x = 0; x < NG; ++x) {
                const int col = col0 + (2 * x + (lc & 1)) * 16 + lq;
#pragma unroll
                for (int i = 0; i < GH; ++i)
                    if (col < N)
                        p.aws[((int64_t)b * p.H + kvh * p.g + 2 * i + (lc >> 1)) * N + col] = (unsigned short)(__float_as_uint(a[x][i]) >> 16);
            }
        } else {
            int rp0 = 0;                                       // (2 rt) % g, kept by increments: no modulo per tile
            for (int rt = 0; rt < p.L / 16; ++rt) {
                float gs[BT][NG];
                sums(rt, gs);
                // the two halves in group order (with g = 1 both land on the same accumulator)
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    if (lc >> 1 == half) {
                        float* x = accs + rp0 * 32 + (lc & 1) * 16 + lq;
                        *x = bf16_to_f32(f32_to_bf16(*x + gs[0][0]));
                    }
                    rp0 = rp0 + 1 == p.g ? 0 : rp0 + 1;
                    __builtin_amdgcn_wave_barrier();
                }
            }
            for (int i = lane; i < p.g * 32; i += 64) {
                const int rp = i / 32, c = i % 32;
                if (col0 + c < N) {
                    const bf16_t v = f32_to_bf16(accs[i]);
                    p.aws[((int64_t)b * p.H + kvh * p.g + rp) * N + col0 + c] = *reinterpret_cast<const unsigned short*>(&v);
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
        if constexpr (NC == 2) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int ks = 0; ks < D / 32; ++ks) kf[c][ks] = kn[c][ks];
        }
    }
}

__device__ __forceinline__ unsigned int ordered16(unsigned short bits) {
    return (bits & 0x8000u) ? (unsigned int)(~bits & 0xffffu) : (unsigned int)(bits | 0x8000u);
}

// Pooled + group-summed scores of 1024 columns of one (kv head, request), as bf16 bits: a thread owns four neighbouring columns, the
// rows' columns (and half a pool width on either side) come through LDS.  All CUs take part; inside the selection's one workgroup per
// (kv head, request) it was most of that kernel's 135 us.
// Bound by latency: the columns of four rows are asked for together (each row behind the last one's barrier: 14 us for 16 MB, now 10.2; two bytes a load 10.6).
constexpr int kPoolCols = 1024, kPoolHalf = 64;         // widest half pool that is staged
constexpr int kPoolRows = 4;                            // rows staged at a time

template <int KS, bool VEC>                             // the pool's width where it is known (taps in registers), else 0; rows of whole 8-byte pieces
__global__ __launch_bounds__(256) void snapkv_pool_kernel(const unsigned short* __restrict__ aws, int H, int KH, int g, int N, int ksz_any,
                                                          unsigned short* __restrict__ score_out) {
    constexpr int kImg = kPoolCols + 2 * kPoolHalf, kEdge = (2 * (KS ? KS / 2 : kPoolHalf) + 255) / 256;
    __shared__ __attribute__((aligned(16))) float img[kPoolRows][kImg];      // column c0 + i at kPoolHalf + i
    const int ksz = KS ? KS : ksz_any;
    const int c0 = blockIdx.x * kPoolCols, kvh = blockIdx.y, b = blockIdx.z, tid = threadIdx.x, half = ksz / 2;
    const bool staged = half <= kPoolHalf;
    const unsigned short* rows = aws + ((int64_t)b * H + kvh * g) * N;
    float tot[4] = {0.f, 0.f, 0.f, 0.f};
    for (int r0 = 0; r0 < g; r0 += kPoolRows) {
        if (staged) {
            // a thread's own four columns of each row, and the first threads' half widths on either side
            unsigned short v[kPoolRows][4], w[kPoolRows][kEdge > 0 ? kEdge : 1];
            const int own = c0 + tid * 4;
#pragma unroll
            for (int r = 0; r < kPoolRows; ++r) {
                const unsigned short* row = rows + (int64_t)min(r0 + r, g - 1) * N;
                if constexpr (VEC) {
                    const u32x2 x = *reinterpret_cast<const u32x2*>(row + min(own, N - 4));
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[r][j] = (unsigned short)(x[j >> 1] >> (16 * (j & 1)));
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[r][j] = row[min(own + j, N - 1)];
                }
#pragma unroll
                for (int k = 0; k < kEdge; ++k) {
                    const int i = tid + k * 256, at = i < half ? c0 - half + i : c0 + kPoolCols + i - half;
                    w[r][k] = row[min(max(at, 0), N - 1)];
                }
            }
            if (r0) __syncthreads();
#pragma unroll
            for (int r = 0; r < kPoolRows; ++r) {            // (adding 0 is what leaving a column out is)
                f32x4 x;
#pragma unroll
                for (int j = 0; j < 4; ++j) x[j] = own + j < N ? bf16_bits_to_f32(v[r][j]) : 0.f;
                *reinterpret_cast<f32x4*>(img[r] + kPoolHalf + tid * 4) = x;
#pragma unroll
                for (int k = 0; k < kEdge; ++k) {
                    const int i = tid + k * 256, at = i < half ? c0 - half + i : c0 + kPoolCols + i - half;
                    if (i < 2 * half) img[r][kPoolHalf + at - c0] = at >= 0 && at < N ? bf16_bits_to_f32(w[r][k]) : 0.f;
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int r = 0; r < kPoolRows; ++r) {
            if (r0 + r >= g) break;
            float tap[4 + (KS ? KS - 1 : 0)];
            if constexpr (KS > 0) {
#pragma unroll
                for (int k = 0; k < 4 + KS - 1; ++k) tap[k] = img[r][kPoolHalf - KS / 2 + tid * 4 + k];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int s = tid * 4 + j;
                float acc = 0.f;
                if constexpr (KS > 0) {
#pragma unroll
                    for (int k = 0; k < KS; ++k) acc += tap[j + k];
                } else if (staged) {
                    for (int k = 0; k < ksz; ++k) acc += img[r][kPoolHalf - half + s + k];
                } else {
                    for (int k = -half; k <= half; ++k) {
                        const int c = c0 + s + k;
                        if (c >= 0 && c < N) acc += bf16_bits_to_f32(rows[(int64_t)(r0 + r) * N + c]);
                    }
                }
                tot[j] += bf16_to_f32(f32_to_bf16(acc / (float)ksz));
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int s = c0 + tid * 4 + j;
        const bf16_t tb = f32_to_bf16(tot[j]);
        if (s < N) score_out[((int64_t)b * KH + kvh) * N + s] = *reinterpret_cast<const unsigned short*>(&tb);
    }
}

// inclusive sums over the 1024 threads of a workgroup; `waves` is LDS scratch of 16 entries
__device__ __forceinline__ unsigned int scan1024(unsigned int v, unsigned int* waves, int lane, int wave) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned int u = __shfl_up(v, o);
        if (lane >= o) v += u;
    }
    if (lane == 63) waves[wave] = v;
    __syncthreads();
    unsigned int before = 0;
    for (int w = 0; w < wave; ++w) before += waves[w];
    __syncthreads();
    return v + before;
}

// Exact top-k of N bf16 scores, one workgroup (1024 threads) per (kv head, request).  Histogram of the keys' upper 12 bits (scores of
// one context share a few exponents: 8 bits would put nearly all of them into two counters), a workgroup scan for the bin of the k-th
// largest, the same over its 16 low values; a thread's run of consecutive keys then knows by one scan which of the equal ones are
// the first; the selected keys are ranked by counting (they are distinct: each carries its index).  Bound by latency: a dozen barriers
// (the first version had 120, with single threads walking the histograms).  Scores come and keys go eight at a time where the rows are
// whole pieces of eight (VEC: contexts of a window and whole pages): 16 000 keys 16.7 -> 13.2 us.  (The copy of the rows by the same workgroup: 21 for 13.2 + 7.5
// here, but 7 us longer for rows of 128 or one request, where a workgroup's chain of loads is longer than the launch.)
template <bool VEC>
__global__ __launch_bounds__(1024) void snapkv_select_kernel(const unsigned short* __restrict__ scores, int KH, int N, int topk,
                                                             int32_t* idx_out) {
    constexpr int kBins = 4096;
    extern __shared__ __attribute__((aligned(16))) unsigned char smraw[];
    unsigned short* keys = reinterpret_cast<unsigned short*>(smraw);              // [N] ordered keys
    unsigned int* hist = reinterpret_cast<unsigned int*>(smraw + (N + 7) / 8 * 16);    // [4096]
    unsigned int* sel = hist + kBins;                                             // [1024]
    unsigned int* waves = sel + 1024;                                             // [16]
    unsigned int* misc = waves + 16;                                              // bin, rank in it, number above, [16] low counts
    const int kvh = blockIdx.x, b = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned short* src = scores + ((int64_t)b * KH + kvh) * N;
    constexpr int V = VEC ? 8 : 1;                            // keys at a time
    typedef std::conditional_t<VEC, u32x4, unsigned short> piece;
    const int np = N / V;                                     // pieces of the row
    auto key_of = [](piece x, int e) -> unsigned int {
        if constexpr (VEC) return e & 1 ? x[e >> 1] >> 16 : x[e >> 1] & 0xffffu;
        else return x;
    };
    auto held = [&](int i) -> piece { return reinterpret_cast<const piece*>(keys)[i]; };
    for (int i = tid; i < kBins; i += 1024) hist[i] = 0;
    sel[tid] = 0;
    if (tid < 32) misc[tid] = 0;
    __syncthreads();
    constexpr int U = VEC ? 2 : 8;                            // (loads on their way)
    for (int s0 = tid; s0 < np; s0 += U * 1024) {
        piece v[U];
#pragma unroll
        for (int j = 0; j < U; ++j) v[j] = reinterpret_cast<const piece*>(src)[min(s0 + j * 1024, np - 1)];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int s = s0 + j * 1024;
            if (s < np) {
                unsigned int k[V];
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    k[e] = ordered16((unsigned short)key_of(v[j], e));
                    atomicAdd(&hist[k[e] >> 4], 1u);
                }
                if constexpr (VEC)
                    reinterpret_cast<u32x4*>(keys)[s] = u32x4{k[0] | k[1] << 16, k[2] | k[3] << 16, k[4] | k[5] << 16, k[6] | k[7] << 16};
                else
                    keys[s] = (unsigned short)k[0];
            }
        }
    }
    __syncthreads();
    {   // thread t looks at the four bins 4 t .. 4 t + 3 counted from the top
        unsigned int n[4], sum = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            n[j] = hist[kBins - 1 - (tid * 4 + j)];
            sum += n[j];
        }
        const unsigned int upto = scan1024(sum, waves, lane, wave);
        unsigned int above = upto - sum;
        if (above < (unsigned int)topk && upto >= (unsigned int)topk) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (above < (unsigned int)topk && above + n[j] >= (unsigned int)topk) {
                    misc[0] = kBins - 1 - (tid * 4 + j);
                    misc[1] = topk - above;
                    break;
                }
                above += n[j];
            }
        }
    }
    __syncthreads();
    const unsigned int bin = misc[0];
    for (int s = tid; s < np; s += 1024) {
        const piece x = held(s);
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (key_of(x, e) >> 4 == bin) atomicAdd(&misc[16 + (key_of(x, e) & 15)], 1u);
    }
    __syncthreads();
    unsigned int need = misc[1], low = 15;                    // (every thread: 16 broadcast reads)
    for (; low > 0 && misc[16 + low] < need; --low) need -= misc[16 + low];
    const unsigned int T = bin << 4 | low;                    // the k-th largest key; `need` keys == T are selected, lowest indices first
    // thread t's run of consecutive keys
    const int run = (np + 1023) / 1024, first = min(tid * run, np), last = min(first + run, np);
    unsigned int eq = 0;
    for (int s = first; s < last; ++s) {
        const piece x = held(s);
#pragma unroll
        for (int e = 0; e < V; ++e) eq += key_of(x, e) == T;
    }
    unsigned int rank = scan1024(eq, waves, lane, wave) - eq;
    for (int s = first; s < last; ++s) {
        const piece x = held(s);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const unsigned int k = key_of(x, e), tag = k << 16 | (0xffffu - (unsigned int)(s * V + e));
            if (k > T) sel[atomicAdd(&misc[2], 1u)] = tag;
            if (k == T) {
                if (rank < need) sel[topk - need + rank] = tag;
                ++rank;
            }
        }
    }
    __syncthreads();
    if (tid < topk) {
        const unsigned int mine = sel[tid];
        unsigned int place = 0;
        for (int i = 0; i < topk; i += 4) {                   // (sel is 0 beyond topk: below every key that matters)
            const u32x4 o = *reinterpret_cast<const u32x4*>(sel + i);
            place += (o[0] > mine) + (o[1] > mine) + (o[2] > mine) + (o[3] > mine);
        }
        idx_out[((int64_t)b * KH + kvh) * topk + place] = (int32_t)(0xffffu - (mine & 0xffffu));
    }
}

struct GatherParams {
    const void* cache;
    const float* k_scale;
    const float* v_scale;
    const int32_t* page_indices;
    const int32_t* page_indptr;
    bf16_t* dcache;
    const int32_t* dindices;
    const int32_t* dindptr;
    const int32_t* dlast;
    const int32_t* idx;  // [B][KH][topk]
    int KH, D, page_size, S, W, budget, topk;
    int src_hnd;         // source pages are [2][KH][page_size][D] instead of [2][page_size][KH][D]
};

// a row's 16-byte pieces (k, then v) lie across 2 D / 8 lanes, several rows per wavefront
template <bool FP8>
__global__ __launch_bounds__(256) void snapkv_gather_kernel(const GatherParams p) {
    const int nv = p.D / 8, rows = 256 / (2 * nv), i = threadIdx.x % (2 * nv);
    const int j = blockIdx.x * rows + threadIdx.x / (2 * nv), kvh = blockIdx.y, b = blockIdx.z;
    if (j >= p.budget) return;
    const int src = j < p.topk ? p.idx[((int64_t)b * p.KH + kvh) * p.topk + j] : p.S - p.W + (j - p.topk);
    const int row_elems = p.KH * p.D;
    const int sp = src / p.page_size, ss = src - sp * p.page_size;
    const int64_t spid = p.page_indices[p.page_indptr[b] + sp];
    const int64_t soff = p.src_hnd ? spid * 2 * p.page_size * row_elems + ((int64_t)kvh * p.page_size + ss) * p.D
                                   : (spid * 2 * p.page_size + ss) * row_elems + kvh * p.D;
    const int dp0 = p.dindptr[b];
    const int dnp = p.dindptr[b + 1] - dp0;
    const int dlen = dnp > 0 ? (dnp - 1) * p.page_size + p.dlast[b] : 0;
    const int pos = dlen - p.budget + j;
    if (pos < 0 || pos >= dnp * p.page_size) return;
    const int dpg = pos / p.page_size, dsl = pos - dpg * p.page_size;
    const int64_t dpid = p.dindices[dp0 + dpg];
    const int64_t doff = (dpid * 2 * p.page_size + dsl) * row_elems + kvh * p.D;
    const int64_t half = (int64_t)p.page_size * row_elems;
    {
        const int64_t h = i < nv ? 0 : half;
        const int c = i < nv ? i : i - nv;
        if constexpr (FP8) {   // dequantise into the bf16 draft cache: bf16(byte * scale)
            const float sc = i < nv ? p.k_scale[kvh] : p.v_scale[kvh];
            const u32x2 w = *reinterpret_cast<const u32x2*>(reinterpret_cast<const unsigned char*>(p.cache) + soff + h + c * 8);
            bf16x8 r;
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const f32x2 a = __builtin_amdgcn_cvt_pk_f32_fp8(w[hh], false);
                const f32x2 cc = __builtin_amdgcn_cvt_pk_f32_fp8(w[hh], true);
                r[4 * hh] = f32_to_bf16(a[0] * sc);
                r[4 * hh + 1] = f32_to_bf16(a[1] * sc);
                r[4 * hh + 2] = f32_to_bf16(cc[0] * sc);
                r[4 * hh + 3] = f32_to_bf16(cc[1] * sc);
            }
            *reinterpret_cast<bf16x8*>(p.dcache + doff + h + c * 8) = r;
        } else {
            *reinterpret_cast<u32x4*>(p.dcache + doff + h + c * 8) =
                *reinterpret_cast<const u32x4*>(reinterpret_cast<const bf16_t*>(p.cache) + soff + h + c * 8);
        }
    }
}

// LDS that is left beside the table of BIN binades (and a few words)
template <int BIN>
constexpr int beside_table() {
    return 160 * 1024 - Tab<BIN>::N * 8 - 256;
}

// A score kernel, whose LDS, with the table of BIN binades, is more than 64 KB
template <auto Kernel, int BIN>
int score_launch(dim3 grid, int waves, size_t lds, const SnapParams& p, hipStream_t st) {
    static MdPerDeviceOnce once;
    constexpr int cap = beside_table<BIN>();
    if (once.first() && hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, cap) != hipSuccess) {
        once.undo();
        md_set_error("md_snapkv_select: hipFuncSetAttribute(%d B LDS) failed", cap);
        return MD_ERR_LAUNCH;
    }
    hipLaunchKernelGGL(Kernel, grid, dim3(64 * waves), lds, st, p);
    return MD_OK;
}

template <auto Kernel>
int select_launch(int KH, int B, size_t lds, const unsigned short* scores, int N, int topk, int32_t* idx_out, hipStream_t st) {
    static MdPerDeviceOnce once;
    if (once.first()) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) {
            once.undo();
            md_set_error("md_snapkv_select: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
            return MD_ERR_LAUNCH;
        }
    }
    hipLaunchKernelGGL(Kernel, dim3(KH, B), dim3(1024), lds, st, scores, KH, N, topk, idx_out);
    return MD_OK;
}

size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Columns per workgroup of the two score kernels, in rounds of the wavefronts' 32 columns each.  A CU holds one workgroup at a time, which
// costs its rounds and two more for the table, the query image and the merge; the launch ends with the CU that has the most.  (Drawn for
// workgroups of eight wavefronts over 320 sizes, within 0.6 % of the best number of chunks: 52 requests of 700 keys, 8 queries a kv head
// of 64, 162 us in one chunk, 188 in two; 25 requests of 2 100, 8 of 64, 121.)
int score_cols(int B, int KH, int L, int D, int ctx_len) {
    const int64_t pairs = (int64_t)B * KH;
    const int round = 32 * score_waves(D, (L + 15) / 16), all = std::max((ctx_len + round - 1) / round, 1);        // (a size may be asked for any length)
    double least = 1e300;
    int best = all;
    for (int r = 1; r <= all; ++r) {
        const double cost = (double)(2 + r) * (double)((pairs * ((all + r - 1) / r) + 255) / 256);
        if (cost < least) {
            least = cost;
            best = r;
        }
    }
    const int n = (all + best - 1) / best;                           // ... and as even as whole rounds go
    return (all + n - 1) / n * round;
}

// bytes of the partial sums: either head size (it is not among the sizes the workspace is asked for by)
size_t partial_bytes(int B, int KH, size_t L, int ctx_len) {
    size_t nch = 1;
    for (int D : {64, 128}) {
        const size_t cols = score_cols(B, KH, (int)L, D, ctx_len);
        nch = std::max(nch, (ctx_len + cols - 1) / cols);
    }
    return align_up((size_t)B * KH * L * nch * 2 * 8, 256);
}

}  // namespace

extern "C" size_t md_snapkv_workspace_bytes(int B, int H, int KH, int ctx_len, int window) {
    if (B <= 0 || H <= 0 || KH <= 0 || H % KH || ctx_len <= window) return 0;
    const int g = H / KH;
    const size_t L = (size_t)g * window;
    const size_t partials = partial_bytes(B, KH, L, ctx_len);
    const size_t aws = align_up((size_t)B * H * (ctx_len - window) * 2, 256);
    const size_t scores = align_up((size_t)B * KH * (ctx_len - window) * 2, 256);
    return partials + aws + scores + 256;
}

extern "C" size_t md_snapkv_scores_offset(int B, int H, int KH, int ctx_len, int window) {
    if (B <= 0 || H <= 0 || KH <= 0 || H % KH || ctx_len <= window) return 0;
    const int g = H / KH;
    const size_t L = (size_t)g * window;
    return partial_bytes(B, KH, L, ctx_len) + align_up((size_t)B * H * (ctx_len - window) * 2, 256);
}

extern "C" int md_snapkv_select(const void* q_win, const void* cache, const int32_t* page_indices,
                                const int32_t* page_indptr, int B, int H, int KH, int D, int page_size, int ctx_len,
                                int window, int budget, int pool_kernel, void* draft_cache,
                                const int32_t* draft_page_indices, const int32_t* draft_page_indptr,
                                const int32_t* draft_last_page_len, int32_t* idx_out, int kv_dtype,
                                const float* k_scale, const float* v_scale, void* workspace,
                                size_t workspace_bytes, md_stream_t stream) {
    MD_CHECK_ARG(q_win && cache && page_indices && page_indptr && draft_cache && draft_page_indices &&
                     draft_page_indptr && draft_last_page_len && idx_out && workspace,
                 "md_snapkv_select: null pointer argument");
    MD_CHECK_ARG(B > 0 && H > 0 && KH > 0 && H % KH == 0, "md_snapkv_select: bad heads H=%d KH=%d", H, KH);
    if (D != 64 && D != 128) {
        md_set_error("md_snapkv_select: head_dim %d unsupported (64 or 128)", D);
        return MD_ERR_UNSUPPORTED;
    }
    const int g = H / KH;
    const int L = g * window;
    const int topk = budget - window;
    const int N = ctx_len - window;
    // the reference itself raises for 8g < window (model.py:415: 8g-row chunk vs WxW mask)
    MD_CHECK_ARG(8 * g >= window, "md_snapkv_select: needs 8*(H/KH) >= window (reference raises for g=%d)", g);
    MD_CHECK_ARG(window > 0 && L % 16 == 0 && L % (8 * g) == 0, "md_snapkv_select: window %d unsupported", window);
    MD_CHECK_ARG(topk > 0 && topk <= N && topk <= 1024, "md_snapkv_select: budget-window=%d must be in [1, min(ctx-window,1024)]", topk);
    MD_CHECK_ARG(ctx_len <= 65536, "md_snapkv_select: ctx_len %d > 65536 unsupported", ctx_len);
    MD_CHECK_ARG(pool_kernel >= 1 && (pool_kernel & 1), "md_snapkv_select: pool kernel must be odd");
    MD_CHECK_ARG(workspace_bytes >= md_snapkv_workspace_bytes(B, H, KH, ctx_len, window) &&
                     (((uintptr_t)workspace) & 255) == 0,
                 "md_snapkv_select: workspace too small or not 256-byte aligned");
    MD_CHECK_ARG((kv_dtype & ~(MD_KV_DTYPE_MASK | MD_KV_LAYOUT_HND)) == 0, "md_snapkv_select: unknown kv_dtype flags");
    const bool hnd = (kv_dtype & MD_KV_LAYOUT_HND) != 0;
    kv_dtype &= MD_KV_DTYPE_MASK;
    MD_CHECK_ARG(kv_dtype == MD_KV_BF16 || (kv_dtype == MD_KV_FP8_E4M3 && k_scale && v_scale),
                 "md_snapkv_select: kv_dtype must be MD_KV_BF16 or MD_KV_FP8_E4M3 (with per-head scales)");
    const bool fp8 = kv_dtype == MD_KV_FP8_E4M3;
    hipStream_t st = (hipStream_t)stream;

    SnapParams p;
    p.q = (const bf16_t*)q_win;
    p.cache = cache;
    p.k_scale = k_scale;
    p.page_indices = page_indices;
    p.page_indptr = page_indptr;
    p.B = B;
    p.H = H;
    p.KH = KH;
    p.g = g;
    p.W = window;
    p.S = ctx_len;
    p.L = L;
    p.cols = score_cols(B, KH, L, D, ctx_len);
    p.nch = (ctx_len + p.cols - 1) / p.cols;
    p.page_size = page_size;
    p.slot_stride = hnd ? D : KH * D;
    p.head_stride = hnd ? page_size * D : D;
    p.page_stride = 2 * (int64_t)page_size * KH * D;
    unsigned char* ws = (unsigned char*)workspace;
    p.partials = (double*)ws;
    const size_t partials_b = partial_bytes(B, KH, L, ctx_len);
    p.aws = (unsigned short*)(ws + partials_b);
    const size_t aws_b = align_up((size_t)B * H * N * 2, 256);
    unsigned short* scores = (unsigned short*)(ws + partials_b + aws_b);

    MD_CHECK_ARG(L <= 16 * kMaxRT, "md_snapkv_select: g * window = %d rows per kv head, at most %d supported", L, 16 * kMaxRT);
    const size_t qimg_b = (size_t)image_rows(L) * (D * 2 + kQPad);
    const int waves = score_waves(D, L / 16);
    const size_t lds1 = qimg_b + (size_t)waves * L * 2 * 8;
    // accumulators in registers for g = 2, 4, 8 (a chunk of 8 g rows is then g / 2 whole tiles)
    const int gh = g == 2 || g == 4 || g == 8 ? g / 2 : 0;
    const size_t lds2 = qimg_b + (size_t)L * 3 * 8 + (gh ? 0 : (size_t)waves * g * 32 * 4);
    const dim3 sg(p.nch, KH, B), ag((N + p.cols - 1) / p.cols, KH, B);
    const bool small = L <= 128;
    const int rounds = p.cols / (32 * waves);                  // (wavefronts of 64 columns: half of the rounds, one too many of few odd ones)
    const bool four = rounds % 2 == 0 || rounds > 6;
    // (30 and 32 queries a kv head of 128: 171 648 and 174 080 bytes with the whole table, of 163 840)
    const bool tight = lds2 > (size_t)beside_table<kTabBinades>();
    MD_CHECK_ARG(lds1 <= (size_t)(D == 128 && !small ? beside_table<kTabSmall>() : beside_table<kTabBinades>()) &&
                     (!tight || (D == 128 && !small && gh == 0 && lds2 <= (size_t)beside_table<kTabSmall>())),
                 "md_snapkv_select: g=%d window=%d head_dim=%d need %zu / %zu bytes of LDS beside the table", g, window, D, lds1, lds2);
    int rc = MD_OK;
#define MD_SNAP_STATS(DD, FP)                                                                                                \
    rc = small ? score_launch<&snapkv_stats_kernel<DD, FP, 8>, stats_binades(DD, 8)>(sg, waves, lds1, p, st)                 \
               : score_launch<&snapkv_stats_kernel<DD, FP, kMaxRT>, stats_binades(DD, kMaxRT)>(sg, waves, lds1, p, st)
#define MD_SNAP_ACCUM(DD, FP, GG)                                                                                            \
    rc = !small          ? score_launch<&snapkv_accum_kernel<DD, FP, GG, kMaxRT, 2>, kTabBinades>(ag, waves, lds2, p, st)    \
         : four && GG > 0 ? score_launch<&snapkv_accum_kernel<DD, FP, GG, 8, GG ? 4 : 2>, kTabBinades>(ag, waves, lds2, p, st) \
                         : score_launch<&snapkv_accum_kernel<DD, FP, GG, 8, 2>, kTabBinades>(ag, waves, lds2, p, st)
#define MD_SNAP_LAUNCH(DD, FP)                                                                                               \
    do {                                                                                                                     \
        MD_SNAP_STATS(DD, FP);                                                                                               \
        if (rc != MD_OK) return rc;                                                                                          \
        if (p.nch > kFewChunks)                                                                                              \
            hipLaunchKernelGGL(snapkv_finalize_kernel, dim3((unsigned)(((int64_t)B * KH * L + 255) / 256)), dim3(256), 0, st, p); \
        if (gh == 4) MD_SNAP_ACCUM(DD, FP, 4);                                                                               \
        else if (gh == 2) MD_SNAP_ACCUM(DD, FP, 2);                                                                          \
        else if (gh == 1) MD_SNAP_ACCUM(DD, FP, 1);                                                                          \
        else if constexpr (DD == 128) {                                                                                      \
            if (tight) rc = score_launch<&snapkv_accum_kernel<DD, FP, 0, kMaxRT, 2, kTabSmall>, kTabSmall>(ag, waves, lds2, p, st); \
            else MD_SNAP_ACCUM(DD, FP, 0);                                                                                   \
        } else MD_SNAP_ACCUM(DD, FP, 0);                                                                                     \
        if (rc != MD_OK) return rc;                                                                                          \
    } while (0)
    if (D == 128) {
        if (fp8) MD_SNAP_LAUNCH(128, true); else MD_SNAP_LAUNCH(128, false);
    } else {
        if (fp8) MD_SNAP_LAUNCH(64, true); else MD_SNAP_LAUNCH(64, false);
    }
#undef MD_SNAP_LAUNCH
#undef MD_SNAP_STATS
#undef MD_SNAP_ACCUM
    MD_CHECK_LAUNCH("md_snapkv_select(scores)");

    const dim3 pgrid((N + kPoolCols - 1) / kPoolCols, KH, B);
    const auto pool = pool_kernel == 5 ? (N % 4 == 0 ? &snapkv_pool_kernel<5, true> : &snapkv_pool_kernel<5, false>)
                                       : (N % 4 == 0 ? &snapkv_pool_kernel<0, true> : &snapkv_pool_kernel<0, false>);
    hipLaunchKernelGGL(pool, pgrid, dim3(256), 0, st, p.aws, H, KH, g, N, pool_kernel, scores);
    const size_t lds3 = (size_t)((N + 7) / 8 * 8) * 2 + (4096 + 1024 + 16 + 32) * 4;
    rc = N % 8 == 0 ? select_launch<&snapkv_select_kernel<true>>(KH, B, lds3, scores, N, topk, idx_out, st)
                    : select_launch<&snapkv_select_kernel<false>>(KH, B, lds3, scores, N, topk, idx_out, st);
    if (rc != MD_OK) return rc;
    MD_CHECK_LAUNCH("md_snapkv_select(select)");

    GatherParams gp;
    gp.cache = cache;
    gp.k_scale = k_scale;
    gp.v_scale = v_scale;
    gp.page_indices = page_indices;
    gp.page_indptr = page_indptr;
    gp.dcache = (bf16_t*)draft_cache;
    gp.dindices = draft_page_indices;
    gp.dindptr = draft_page_indptr;
    gp.dlast = draft_last_page_len;
    gp.idx = idx_out;
    gp.KH = KH;
    gp.D = D;
    gp.page_size = page_size;
    gp.S = ctx_len;
    gp.W = window;
    gp.budget = budget;
    gp.topk = topk;
    gp.src_hnd = hnd ? 1 : 0;
    const int rows = 256 / (2 * D / 8);
    const dim3 ggrid((budget + rows - 1) / rows, KH, B);
    if (fp8)
        hipLaunchKernelGGL((snapkv_gather_kernel<true>), ggrid, dim3(256), 0, st, gp);
    else
        hipLaunchKernelGGL((snapkv_gather_kernel<false>), ggrid, dim3(256), 0, st, gp);
    MD_CHECK_LAUNCH("md_snapkv_select(gather)");
    return MD_OK;
}
