// Attention in 32-bit arithmetic on the fp32 matrix instructions (v_mfma_f32_16x16x4_f32): 32-bit models, and 16-bit pages where the
// bf16 matrix-core kernels of xattn_mfma.hip / latent_absorbed.hip do not apply (unbounded scores, unusual page sizes).  Queries, keys,
// values, scores, weights and sums are fp32 throughout, as in the plain kernel of xattn.hip, whose semantics these are.
//
// Two kernels, both on (token, head of the kv head) rows and KT-key tiles:
//   prompts, heads to 128   a wavefront owns 16 rows and all of a tile (xattn_f32_rows_kernel)
//   else                    a workgroup of four wavefronts owns R = 16 QT rows together (xattn_f32_kernel):
//   S^T = K.Q^T    a 16 x 16 score tile per wavefront and step; K and Q fragments are ds_read_b128 of padded LDS rows.  The four
//                  elements of a b128 are four k-steps (both operands permute the contraction the same way).
//   softmax        256 / R threads per row, scores through LDS; running maximum in log2 units, the distance penalty as one v_log_f32
//   O^T = V^T.P^T  each wavefront owns every fourth 16-wide slice of the value size, so its sums stay in registers for any head size
//                  and the weights are read back from LDS as B fragments.
// There three barriers per tile (four where values are a prefix of the key rows: one image serves both); the next tile is in registers
// while this one is computed.  Few rows (decode): 16-row tiles and the key range split over workgroups, merged by a second launch.
//
// Bound by the fp32 matrix rate (154 TFLOP/s in a large library product) for prompts, by latency for decode steps.  Six sequences of
// 100 to 1 500 tokens, 32 query and 8 kv heads of 64, one layer (22 GFLOP): 9 930 -> 445 -> 277 us; one token each behind them:
// 292 -> 17.4 + 5.8 us for the merge -> 15.0 + 5.3 with splits of three tiles (of the longest page table's keys) and their loads together in
// the merge (first figure: the plain kernel, one workgroup per row and head).
#include "xattn.h"

#include <algorithm>

namespace {

template <typename T>
struct Vec4;
template <>
struct Vec4<float> {
    typedef f32x4 type;
};
template <>
struct Vec4<bf16_t> {
    typedef bf16x4 type;
};

struct F32Launch {
    int nq, nsplit, R, dvw;      // row groups, kv splits, rows per group, elements per partial row
};

template <int DK, int DV, int QT, int KT, bool SHARED>
constexpr int f32_lds_bytes() {
    return (16 * QT * (DK + 4) + KT * (DK + 4) + (SHARED ? 0 : KT * (DV + 4)) + 16 * QT * (KT + 4) + 16 * QT) * 4 + 16;
}

template <int DK, int DV, int QT, int KT, bool SHARED>
constexpr int f32_waves_per_simd() {
    return f32_lds_bytes<DK, DV, QT, KT, SHARED>() <= 80 * 1024 ? 2 : 1;
}

template <typename T, int DK, int DV, int QT, int KT, bool SHARED>
__global__ __launch_bounds__(256, (f32_waves_per_simd<DK, DV, QT, KT, SHARED>())) void xattn_f32_kernel(const XattnParams p, const F32Launch L) {
    typedef typename Vec4<T>::type vec4;
    constexpr int R = 16 * QT, KP = DK + 4, VP = SHARED ? KP : DV + 4, PP = KT + 4;
    constexpr int KB = KT / 16, NS = (KB * QT + 3) / 4, NV = DV / 64;
    constexpr int TPR = 256 / R, KPT = KT / TPR;                 // softmax: threads per row, keys per thread
    constexpr int LK = KT * DK / 1024, LV = SHARED ? 1 : KT * DV / 1024;   // 4-element pieces of a tile per thread
    static_assert(KT * DK % 1024 == 0 && KT * DV % 1024 == 0 && DK % 16 == 0 && DV % 64 == 0 && KT % 32 == 0, "tile shapes");
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float* sq = lds;
    float* sk = sq + R * KP;
    float* sv = SHARED ? sk : sk + KT * KP;
    float* sp = (SHARED ? sk + KT * KP : sv + KT * VP);
    float* sa = sp + R * PP;                                     // per row: rescaling factor of a tile, final factor at the end
    int* sbad = reinterpret_cast<int*>(sa + R);                  // [2]: the tile's values hold an infinity or a NaN

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 15, lc = lane >> 4;
    const int b = blockIdx.z, kvh = blockIdx.y, g = p.g;
    const int qg = L.nq - 1 - (int)blockIdx.x / L.nsplit, split = (int)blockIdx.x % L.nsplit;    // longest key ranges first
    const int q0 = p.qo_indptr[b], nrows = (p.qo_indptr[b + 1] - q0) * g, R0 = qg * R;
    if (R0 >= nrows) return;
    const int pos0 = p.pos0[b], pg0 = p.page_indptr[b], cap = (p.page_indptr[b + 1] - pg0) * p.page_size;
    const int hi_wg = min(pos0 + (min(R0 + R, nrows) - 1) / g, cap - 1), lo_wg = ((pos0 + R0 / g) / p.chunk) * p.chunk;
    int t0 = 0, t1 = 0;
    if (hi_wg >= lo_wg) {
        const int first = lo_wg / KT, n = hi_wg / KT - first + 1, per = (n + L.nsplit - 1) / L.nsplit;
        t0 = first + min(split * per, n);
        t1 = first + min((split + 1) * per, n);
    }

    // queries: R rows, zeros beyond the rows and the head size
    for (int i = tid; i < R * (DK / 4); i += 256) {
        const int r = i / (DK / 4), d = (i % (DK / 4)) * 4, row = R0 + r;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (row < nrows && d < p.DKp)
            v = __builtin_convertvector(*reinterpret_cast<const vec4*>(reinterpret_cast<const T*>(p.q) +
                                        ((int64_t)(q0 + row / g) * p.H + kvh * g + row % g) * p.DKp + d), f32x4);
        *reinterpret_cast<f32x4*>(sq + r * KP + d) = v;
    }
    if (tid < 2) sbad[tid] = 0;

    // the row this thread does the softmax of
    const int r = tid / TPR, u = tid % TPR;
    int hi = -1, lo = 0;
    float r1 = 0.f, r2 = 0.f, m = -1e30f, l = 0.f;
    const int pos = pos0 + (R0 + r) / g;
    if (R0 + r < nrows) {
        hi = min(pos, cap - 1);
        lo = (pos / p.chunk) * p.chunk;
        if (p.r1) {
            r1 = p.r1[kvh * g + (R0 + r) % g];
            r2 = p.r2[kvh * g + (R0 + r) % g];
        }
    }
    const bool bias = p.r1 != nullptr;

    f32x4 o[QT][NV];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
        for (int v = 0; v < NV; ++v) o[qt][v] = f32x4{0.f, 0.f, 0.f, 0.f};

    vec4 kr[LK], vr[LV];
    // A tile's last keys may be past the workgroup's last one: their rows are not read, and beyond the 16-key group that holds it neither
    // staged nor multiplied (a sequence of a few keys costs what it has).
    auto request = [&](int t) {              // a tile's pieces into registers; its 32-key halves lie in one page each
        const T* kb[KT / 32];
        const T* vb[KT / 32];
#pragma unroll
        for (int h = 0; h < KT / 32; ++h) {
            const int at = min(t * KT + h * 32, cap - 32), page = at / p.page_size;
            const int64_t row = ((int64_t)p.page_indices[pg0 + page] * p.KH + kvh) * p.page_size + (at - page * p.page_size);
            kb[h] = reinterpret_cast<const T*>(p.k_cache) + row * p.ldk;
            vb[h] = reinterpret_cast<const T*>(p.v_cache) + row * p.ldv;
        }
#pragma unroll
        for (int i = 0; i < LK; ++i) {
            const int e = tid + 256 * i, row = e / (DK / 4), d = (e % (DK / 4)) * 4;
            const T* base = KT == 64 && row >= 32 ? kb[KT / 32 - 1] : kb[0];
            kr[i] = vec4{};
            if (d < p.DKp && t * KT + row <= hi_wg) kr[i] = *reinterpret_cast<const vec4*>(base + (int64_t)(row % 32) * p.ldk + d);
        }
        if constexpr (!SHARED) {
#pragma unroll
            for (int i = 0; i < LV; ++i) {
                const int e = tid + 256 * i, row = e / (DV / 4), d = (e % (DV / 4)) * 4;
                const T* base = KT == 64 && row >= 32 ? vb[KT / 32 - 1] : vb[0];
                vr[i] = vec4{};
                if (d < p.DVp && t * KT + row <= hi_wg) vr[i] = *reinterpret_cast<const vec4*>(base + (int64_t)(row % 32) * p.ldv + d);
            }
        }
    };
    auto odd = [](f32x4 v) {                 // an infinity or a NaN among the four
        return !(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))) <= 3.402823466e38f) || v[0] != v[0] ||
               v[1] != v[1] || v[2] != v[2] || v[3] != v[3];
    };
    auto stage_k = [&](int t) {              // rows past the workgroup's last key are zeros: they may hold anything
        bool bad = false;
#pragma unroll
        for (int i = 0; i < LK; ++i) {
            const int e = tid + 256 * i, row = e / (DK / 4), d = (e % (DK / 4)) * 4;
            f32x4 v = __builtin_convertvector(kr[i], f32x4);
            if (t * KT + row > hi_wg) v = f32x4{0.f, 0.f, 0.f, 0.f};
            if (SHARED) bad |= odd(v);
            if (t * KT + row <= (hi_wg | 15)) *reinterpret_cast<f32x4*>(sk + row * KP + d) = v;
        }
        if (SHARED && __builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0) sbad[t & 1] = 1;
    };
    auto stage_v = [&](int t) {
        bool bad = false;
#pragma unroll
        for (int i = 0; i < LV; ++i) {
            const int e = tid + 256 * i, row = e / (DV / 4), d = (e % (DV / 4)) * 4;
            f32x4 v = __builtin_convertvector(vr[i], f32x4);
            if (t * KT + row > hi_wg) v = f32x4{0.f, 0.f, 0.f, 0.f};
            bad |= odd(v);
            if (t * KT + row <= (hi_wg | 15)) *reinterpret_cast<f32x4*>(sv + row * VP + d) = v;
        }
        if (__builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0) sbad[t & 1] = 1;
    };

    __syncthreads();                         // sbad is clear, the queries are there
    if (t0 < t1) {
        request(t0);
        stage_k(t0);
        if constexpr (!SHARED) stage_v(t0);
        if (t0 + 1 < t1) request(t0 + 1);
    }
    __syncthreads();
    const int kt = wave % KB;                // this wavefront's 16 keys of a tile ...
    for (int t = t0; t < t1; ++t) {
        // ---- scores
        {
            f32x4 s[NS];
            const float* kp = sk + (kt * 16 + lq) * KP + lc * 4;
#pragma unroll
            for (int i = 0; i < NS; ++i) s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
            const int dk = t * KT + kt * 16 <= hi_wg ? DK : 0;
#pragma unroll 4
            for (int d = 0; d < dk; d += 16) {
                const f32x4 ka = *reinterpret_cast<const f32x4*>(kp + d);
#pragma unroll
                for (int i = 0; i < NS; ++i) {
                    const int qt = (wave + 4 * i) / KB;                   // ... against every (4 / KB)-th row tile
                    const f32x4 qb = *reinterpret_cast<const f32x4*>(sq + ((qt < QT ? qt : 0) * 16 + lq) * KP + lc * 4 + d);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[e], qb[e], s[i], 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                const int qt = (wave + 4 * i) / KB;
                if (qt < QT) *reinterpret_cast<f32x4*>(sp + (qt * 16 + lq) * PP + kt * 16 + lc * 4) = s[i];
            }
        }
        __syncthreads();
        // ---- softmax of row r over the tile's keys u * KPT ..
        {
            typedef float fvec __attribute__((ext_vector_type(KPT < 4 ? KPT : 4)));
            constexpr int W = KPT < 4 ? KPT : 4;
            float* row = sp + r * PP + u * KPT;
            float s[KPT];
            float mx = -INFINITY;
#pragma unroll
            for (int k = 0; k < KPT; k += W) {
                const fvec x = *reinterpret_cast<const fvec*>(row + k);
#pragma unroll
                for (int e = 0; e < W; ++e) s[k + e] = x[e];
            }
#pragma unroll
            for (int k = 0; k < KPT; ++k) {
                const int kp = t * KT + u * KPT + k;
                float v = s[k] * p.scale_log2;
                if (bias) v -= r1 * __builtin_amdgcn_logf(1.0f + r2 * (float)(pos - kp));
                s[k] = kp >= lo && kp <= hi ? v : -INFINITY;
                mx = fmaxf(mx, s[k]);
            }
#pragma unroll
            for (int x = 1; x < TPR; x <<= 1) mx = fmaxf(mx, __shfl_xor(mx, x));
            const float mnew = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - mnew);
            m = mnew;
            float ps = 0.f;
#pragma unroll
            for (int k = 0; k < KPT; k += W) {
                fvec x;
#pragma unroll
                for (int e = 0; e < W; ++e) {
                    x[e] = __builtin_amdgcn_exp2f(s[k + e] - mnew);
                    ps += x[e];
                }
                *reinterpret_cast<fvec*>(row + k) = x;
            }
#pragma unroll
            for (int x = 1; x < TPR; x <<= 1) ps += __shfl_xor(ps, x);
            l = l * alpha + ps;
            if (u == 0) sa[r] = alpha;
            if (tid == 0) sbad[(t + 1) & 1] = 0;
        }
        if constexpr (!SHARED) {
            if (t + 1 < t1) stage_k(t + 1);  // every wavefront has read this tile's keys
        }
        __syncthreads();
        // ---- values
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            const float a = sa[qt * 16 + lq];
#pragma unroll
            for (int v = 0; v < NV; ++v) o[qt][v] *= a;
        }
        if (sbad[t & 1] == 0) {
#pragma unroll
            for (int kk = 0; kk < KT; kk += 16) {
                if (t * KT + kk > hi_wg) break;
                f32x4 pb[QT];
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) pb[qt] = *reinterpret_cast<const f32x4*>(sp + (qt * 16 + lq) * PP + kk + lc * 4);
#pragma unroll
                for (int v = 0; v < NV; ++v)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float va = sv[(kk + lc * 4 + e) * VP + (wave + 4 * v) * 16 + lq];
#pragma unroll
                        for (int qt = 0; qt < QT; ++qt) o[qt][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(va, pb[qt][e], o[qt][v], 0, 0, 0);
                    }
            }
        } else {
            // a value that a row does not see must not reach it as 0 * infinity; one that it sees does, also with a weight that underflowed
            for (int k = 0; k < KT; ++k)
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    const float w = sp[(qt * 16 + lq) * PP + k];
                    const int at = pos0 + (R0 + qt * 16 + lq) / g, kp = t * KT + k;
                    if (kp >= (at / p.chunk) * p.chunk && kp <= min(at, cap - 1)) {
#pragma unroll
                        for (int v = 0; v < NV; ++v)
#pragma unroll
                            for (int e = 0; e < 4; ++e) o[qt][v][e] = fmaf(w, sv[k * VP + (wave + 4 * v) * 16 + lc * 4 + e], o[qt][v][e]);
                    }
                }
        }
        __syncthreads();
        if (t + 1 < t1) {
            if constexpr (SHARED) stage_k(t + 1);
            else stage_v(t + 1);
            if (t + 2 < t1) request(t + 2);
            if constexpr (SHARED) __syncthreads();
        }
    }
    // ---- out: lane (lq, lc) holds elements d .. d + 3 of row qt * 16 + lq
    const int64_t slot = (((int64_t)b * p.KH + kvh) * L.nq + qg) * L.nsplit + split;
    float* wo = p.ws + slot * R * L.dvw;
    if (u == 0) {
        if (L.nsplit == 1) {
            const float M = p.sink ? fmaxf(m, 0.f) : m, f = __builtin_amdgcn_exp2f(m - M);
            const float Z = l * f + (p.sink ? __builtin_amdgcn_exp2f(-M) : 0.f);
            sa[r] = Z > 0.f ? f / Z : Z != Z ? Z : 0.f;
        } else {
            float* ml = p.ws + (int64_t)p.B * p.KH * L.nq * L.nsplit * R * L.dvw + (slot * R + r) * 2;
            ml[0] = m;
            ml[1] = l;
        }
    }
    __syncthreads();
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int row = R0 + qt * 16 + lq;
        if (row >= nrows) continue;
        const float f = L.nsplit == 1 ? sa[qt * 16 + lq] : 1.f;
        T* out = reinterpret_cast<T*>(p.out) + ((int64_t)(q0 + row / g) * p.H + kvh * g + row % g) * p.DV;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int d = (wave + 4 * v) * 16 + lc * 4;
            if (L.nsplit > 1) {
                *reinterpret_cast<f32x4*>(wo + (qt * 16 + lq) * L.dvw + d) = o[qt][v];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (d + e < p.DV) out[d + e] = (T)(o[qt][v][e] * f);
            }
        }
    }
}

// Prompts, heads to 128: a wavefront has 16 query rows to itself, NW of them share a tile of KT keys and values in two buffers, one barrier a
// tile.  Scores come out of K.Q^T as V^T.P^T wants its weights -- lane (row, group) holds keys 16 k + 4 group + e -- and go from one product
// to the next without LDS; queries and sums stay in registers.
//
// What bounds it: fp32 products and vector instructions of a SIMD exclude each other (12 of 42 million vector instructions less took as many
// cycles off as they issue in), so everything beside the products counts: loads by descriptor, no address arithmetic; the reference of the
// softmax moves only where it must; four columns of V a read.  The shape above: four wavefronts on 64 rows together 445 us, this 310, with
// these 277 (80 TFLOP/s; products alone 250).  One prompt of 2 500 470 -> 268, 4 x 600 at 16 / 4 heads of 128 148 -> 97; tiles of 64 keys
// 10 % slower, eight wavefronts 2 to 20 %.
template <int DK, int DV, int KT>
constexpr int rows_lds_bytes() {
    return 2 * KT * (DK + DV + 8) * 4 + 16;
}

template <typename T, int DK, int DV, int KT, int NW, int OCC>
__global__ __launch_bounds__(64 * NW, OCC) void xattn_f32_rows_kernel(const XattnParams p, const F32Launch L) {
    typedef typename Vec4<T>::type vec4;
    constexpr int R = 16 * NW, NT = 64 * NW, KP = DK + 4, VP = DV + 4, KB = KT / 16, NV = DV / 16;
    constexpr int kTile = KT * (KP + VP);                        // floats of one buffer
    constexpr int LK = KT * DK / (4 * NT), LV = KT * DV / (4 * NT);
    static_assert(KT * DK % (4 * NT) == 0 && KT * DV % (4 * NT) == 0 && DK % 16 == 0 && DV % 64 == 0 && KT == 32, "tile shapes");
    extern __shared__ __attribute__((aligned(16))) float lds[];
    int* sbad = reinterpret_cast<int*>(lds + 2 * kTile);         // [3]: the tile's values hold an infinity, a NaN or 2^101 and more

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lq = lane & 15, lc = lane >> 4;
    const int pairs = p.KH * p.B, pair = blockIdx.x % pairs, part = blockIdx.x / pairs, kvh = pair % p.KH, b = pair / p.KH, g = p.g;
    const int qg = L.nq - 1 - part / L.nsplit, split = part % L.nsplit;                 // longest key ranges of all sequences first
    const int q0 = p.qo_indptr[b], nrows = (p.qo_indptr[b + 1] - q0) * g, R0 = qg * R;
    if (R0 >= nrows) return;
    const int pos0 = p.pos0[b], pg0 = p.page_indptr[b], cap = (p.page_indptr[b + 1] - pg0) * p.page_size;
    const int hi_wg = min(pos0 + (min(R0 + R, nrows) - 1) / g, cap - 1), lo_wg = ((pos0 + R0 / g) / p.chunk) * p.chunk;
    int t0 = 0, t1 = 0;
    if (hi_wg >= lo_wg) {
        const int first = lo_wg / KT, n = hi_wg / KT - first + 1, per = (n + L.nsplit - 1) / L.nsplit;
        t0 = first + min(split * per, n);
        t1 = first + min((split + 1) * per, n);
    }
    // this lane's row, and the keys that all and that any of the wavefront's rows see
    const int Rw = R0 + wave * 16, row = Rw + lq;
    const int first_pos = pos0 + Rw / g, last_pos = pos0 + (min(Rw + 16, nrows) - 1) / g;
    const int any_lo = first_pos / p.chunk * p.chunk, any_hi = Rw < nrows ? min(last_pos, cap - 1) : -1;
    const int all_lo = last_pos / p.chunk * p.chunk, all_hi = min(first_pos, cap - 1);
    int hi = -1, lo = 0;
    float r1 = 0.f, r2 = 0.f, m = 0.f, l = 0.f, top = -INFINITY;
    const int pos = pos0 + row / g;
    if (row < nrows) {
        hi = min(pos, cap - 1);
        lo = (pos / p.chunk) * p.chunk;
        if (p.r1) {
            r1 = p.r1[kvh * g + row % g];
            r2 = p.r2[kvh * g + row % g];
        }
    }
    const bool bias = p.r1 != nullptr;
    f32x4 q[DK / 16], o[NV];
#pragma unroll
    for (int i = 0; i < DK / 16; ++i) {
        const int d = i * 16 + lc * 4;
        q[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (row < nrows && d < p.DKp)
            q[i] = __builtin_convertvector(*reinterpret_cast<const vec4*>(reinterpret_cast<const T*>(p.q) +
                                           ((int64_t)(q0 + row / g) * p.H + kvh * g + row % g) * p.DKp + d), f32x4);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) o[v] = f32x4{0.f, 0.f, 0.f, 0.f};

    constexpr float kLag = 4.f;
    auto scaled = [&](float score) {
#pragma clang fp contract(off)
        return score * p.scale_log2;         // (rounded: no part of a fused operation)
    };
    // element x of o[v]: the values' column 4 j + v % 4 of 64 is row j of product v, so that a lane reads four columns at once
    auto at = [&](int v, int x) { return v / 4 * 64 + lc * 16 + x * 4 + v % 4; };

    // A tile's pieces into registers.  It lies in one page; the descriptor ends with the workgroup's last key, and what lies behind it or
    // beyond the head size reads as zeros
    vec4 kr[LK], vr[LV];
    unsigned kat[LK], vat[LV];
#pragma unroll
    for (int i = 0; i < LK; ++i) {
        const int e = tid + NT * i, key = e / (DK / 4), d = e % (DK / 4) * 4;
        kat[i] = d < p.DKp ? (unsigned)((key * p.ldk + d) * sizeof(T)) : 0xc0000000u;
    }
#pragma unroll
    for (int i = 0; i < LV; ++i) {
        const int e = tid + NT * i, key = e / (DV / 4), d = e % (DV / 4) * 4;
        vat[i] = d < p.DVp ? (unsigned)((key * p.ldv + d) * sizeof(T)) : 0xc0000000u;
    }
    auto fetch = [](__amdgpu_buffer_rsrc_t r, unsigned at) {
        if constexpr (sizeof(T) == 4) {
            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0);
            return *reinterpret_cast<const vec4*>(&v);
        } else {
            const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, 0);
            return *reinterpret_cast<const vec4*>(&v);
        }
    };
    auto request = [&](int t) {
        const int key = t * KT, page = key / p.page_size, keys = min(hi_wg - key + 1, KT);
        const int64_t line = ((int64_t)p.page_indices[pg0 + page] * p.KH + kvh) * p.page_size + (key - page * p.page_size);
        const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<T*>(reinterpret_cast<const T*>(p.k_cache) + line * p.ldk), (short)0, keys * p.ldk * (int)sizeof(T), 0x00020000);
#pragma unroll
        for (int i = 0; i < LK; ++i) kr[i] = fetch(rk, kat[i]);
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<T*>(reinterpret_cast<const T*>(p.v_cache) + line * p.ldv), (short)0, keys * p.ldv * (int)sizeof(T), 0x00020000);
#pragma unroll
        for (int i = 0; i < LV; ++i) vr[i] = fetch(rv, vat[i]);
    };
    auto stage = [&](int t) {                // (keys past the workgroup's last one are zeros: their memory may hold anything)
        float* sk = lds + ((t - t0) & 1) * kTile;
        float worst = 0.f;                   // (2^27 times the sum of the values' sizes: infinite or a NaN)
#pragma unroll
        for (int i = 0; i < LK; ++i) {
            const int e = tid + NT * i, key = e / (DK / 4), d = (e % (DK / 4)) * 4;
            *reinterpret_cast<f32x4*>(sk + key * KP + d) = __builtin_convertvector(kr[i], f32x4);
        }
#pragma unroll
        for (int i = 0; i < LV; ++i) {
            const int e = tid + NT * i, key = e / (DV / 4), d = (e % (DV / 4)) * 4;
            const f32x4 v = __builtin_convertvector(vr[i], f32x4);
            *reinterpret_cast<f32x4*>(sk + KT * KP + key * VP + d) = v;
            for (int x = 0; x < 4; ++x) worst = fmaf(fabsf(v[x]), 0x1p27f, worst);
        }
        if (__builtin_amdgcn_ballot_w64(!(worst < INFINITY)) != 0 && lane == 0) sbad[t % 3] = 1;
    };

    if (tid < 3) sbad[tid] = 0;
    if (t0 < t1) {
        request(t0);
        // (the queries have come: else the compiler waits in the loop for them, and for the tile requested behind)
#pragma unroll
        for (int i = 0; i < DK / 16; ++i) asm volatile("" : "+v"(q[i]));
        asm volatile("" : "+v"(r1), "+v"(r2));
        __syncthreads();
        stage(t0);
        if (t0 + 1 < t1) request(t0 + 1);
    }
    __syncthreads();
    for (int t = t0; t < t1; ++t) {
        // one barrier a tile: past it nobody reads the buffer of the tile before, nor its mark
        if (tid == 0) sbad[(t + 2) % 3] = 0;
        if (t + 1 < t1) stage(t + 1);
        if (t + 2 < t1) request(t + 2);
        const int base = t * KT;
        if (base <= any_hi && base + KT > any_lo) {
            const float* sk = lds + ((t - t0) & 1) * kTile;
            const float* sv = sk + KT * KP;
            // ---- scores: lane (lq, lc) gets keys 16 k + 4 lc + e of row lq
            f32x4 s[KB];
#pragma unroll
            for (int k = 0; k < KB; ++k) s[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < DK / 16; ++i) {
                f32x4 ka[KB];
#pragma unroll
                for (int k = 0; k < KB; ++k) ka[k] = *reinterpret_cast<const f32x4*>(sk + (k * 16 + lq) * KP + i * 16 + lc * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int k = 0; k < KB; ++k) s[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[k][e], q[i][e], s[k], 0, 0, 0);
            }
            // ---- softmax.  The reference m of a row moves only where a score passes it by kLag (log2): a weight is at most 2^kLag, and what
            // moving it costs is rarely paid.  Large values' weights are at most 1: sums reach as far as with the maximum.  The scaled score is
            // rounded before the reference is taken off, so that scores that are the same weigh the same in every tile, whatever their size
            // (scale and reference in one operation: equal scores of 10^6 3 % apart, of 10^9 an infinity, prompts with a bias 5 to 25 % further
            // off 64 bits; level in time, but 2 x 1 000 rows, 32 / 8 heads of 128, 187 us where this takes 193; with a lag of 4 errors are
            // within 1 % of the maximum's, of 8 3 %, and time is the same).  A row that has seen no key yet takes the first tile's maximum
            const bool marked = sbad[t % 3] != 0;
            const float limit = marked ? top - kLag : top;
            const float ahead = (float)(pos - base - lc * 4);
#pragma unroll
            for (int k = 0; k < KB; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[k][e] = scaled(s[k][e]);
            if (bias) {
                asm volatile("");                // (a branch: not computed and thrown away)
#pragma unroll
                for (int k = 0; k < KB; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        s[k][e] = fmaf(-r1, __builtin_amdgcn_logf(1.0f + r2 * (ahead - (float)(k * 16 + e))), s[k][e]);
            }
            if (!(base >= all_lo && base + KT - 1 <= all_hi && Rw + 16 <= nrows)) {
#pragma unroll
                for (int k = 0; k < KB; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int kp = base + k * 16 + lc * 4 + e;
                        s[k][e] = kp >= lo && kp <= hi ? s[k][e] : -INFINITY;
                    }
            }
            float mx = -INFINITY;
#pragma unroll
            for (int k = 0; k < KB; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[k][e]);
            if (__builtin_amdgcn_ballot_w64(mx > limit) != 0) {
                mx = fmaxf(mx, __shfl_xor(mx, 16));
                mx = fmaxf(mx, __shfl_xor(mx, 32));
                const float mnew = mx > limit ? mx : m, alpha = top == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mnew);
                if (mx > limit) top = mnew + kLag;
                m = mnew;
                l *= alpha;
#pragma unroll
                for (int v = 0; v < NV; ++v) o[v] *= alpha;
            }
#pragma unroll
            for (int k = 0; k < KB; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s[k][e] = __builtin_amdgcn_exp2f(s[k][e] - m);
                    l += s[k][e];
                }
            // ---- values: the weights are where the product wants them
            if (!marked) {
#pragma unroll
                for (int k = 0; k < KB; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int v = 0; v < NV; v += 4) {
                            const f32x4 va = *reinterpret_cast<const f32x4*>(sv + (k * 16 + lc * 4 + e) * VP + v * 16 + lq * 4);
#pragma unroll
                            for (int x = 0; x < 4; ++x) o[v + x] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[x], s[k][e], o[v + x], 0, 0, 0);
                        }
            } else {
                // a value that a row does not see must not reach it as 0 * infinity; one that it sees does, also with a weight that underflowed
#pragma unroll
                for (int k = 0; k < KB; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        for (int c = 0; c < 4; ++c) {
                            const float w = __shfl(s[k][e], c * 16 + lq);
                            const int key = k * 16 + c * 4 + e;
                            if (base + key >= lo && base + key <= hi) {
#pragma unroll
                                for (int v = 0; v < NV; ++v)
#pragma unroll
                                    for (int x = 0; x < 4; ++x) o[v][x] = fmaf(w, sv[key * VP + at(v, x)], o[v][x]);
                            }
                        }
            }
        }
        __syncthreads();
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    // ---- out: lane (lq, lc) holds elements d .. d + 3 of its row
    if (row >= nrows) return;
    const int64_t slot = ((((int64_t)b * p.KH + kvh) * L.nq + qg) * L.nsplit + split) * R + wave * 16 + lq;
    if (L.nsplit > 1) {
        float* ml = p.ws + (int64_t)p.B * p.KH * L.nq * L.nsplit * R * L.dvw + slot * 2;
        if (lc == 0) {
            ml[0] = top == -INFINITY ? -1e30f : m;
            ml[1] = l;
        }
#pragma unroll
        for (int v = 0; v < NV; v += 4)
#pragma unroll
            for (int x = 0; x < 4; ++x)
                *reinterpret_cast<f32x4*>(p.ws + slot * L.dvw + at(v, x)) = f32x4{o[v][x], o[v + 1][x], o[v + 2][x], o[v + 3][x]};
        return;
    }
    const float M = p.sink ? fmaxf(m, 0.f) : m, f = __builtin_amdgcn_exp2f(m - M);
    const float Z = l * f + (p.sink ? __builtin_amdgcn_exp2f(-M) : 0.f), inv = Z > 0.f ? f / Z : Z != Z ? Z : 0.f;
    T* out = reinterpret_cast<T*>(p.out) + ((int64_t)(q0 + row / g) * p.H + kvh * g + row % g) * p.DV;
    const bool wide = p.DV % 4 == 0 && reinterpret_cast<uintptr_t>(p.out) % sizeof(vec4) == 0;
#pragma unroll
    for (int v = 0; v < NV; v += 4)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const f32x4 y = f32x4{o[v][x], o[v + 1][x], o[v + 2][x], o[v + 3][x]} * inv;
            if (wide) {
                if (at(v, x) < p.DV) *reinterpret_cast<vec4*>(out + at(v, x)) = __builtin_convertvector(y, vec4);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (at(v + e, x) < p.DV) out[at(v + e, x)] = (T)y[e];
            }
        }
}

// sums the kv splits: one thread per four elements of a row
template <typename T>
__global__ __launch_bounds__(256) void xattn_f32_merge_kernel(const XattnParams p, const F32Launch L) {
    const int vpr = L.dvw / 4;
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x, rowid = id / vpr;
    const int d = (int)(id - rowid * vpr) * 4, r = (int)(rowid % L.R);
    const int64_t item = rowid / L.R;                         // (b, kvh, row group)
    const int qg = (int)(item % L.nq), pair = (int)(item / L.nq);
    if (pair >= p.B * p.KH || d >= p.DV) return;
    const int b = pair / p.KH, kvh = pair % p.KH, q0 = p.qo_indptr[b], row = qg * L.R + r;
    if (row >= (p.qo_indptr[b + 1] - q0) * p.g) return;
    const float* ml = p.ws + (int64_t)p.B * p.KH * L.nq * L.nsplit * L.R * L.dvw;
    // (eight splits' loads together: they are all there is to wait for)
    constexpr int U = 8;
    const int64_t first = item * L.nsplit * L.R + r;
    float M = p.sink ? 0.f : -1e30f;
    for (int s0 = 0; s0 < L.nsplit; s0 += U) {
        float m[U];
#pragma unroll
        for (int u = 0; u < U; ++u) m[u] = ml[(first + (int64_t)min(s0 + u, L.nsplit - 1) * L.R) * 2];
#pragma unroll
        for (int u = 0; u < U; ++u) M = fmaxf(M, m[u]);
    }
    float Z = p.sink ? __builtin_amdgcn_exp2f(-M) : 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < L.nsplit; s0 += U) {
        f32x2 x[U];
        f32x4 y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t at = first + (int64_t)min(s0 + u, L.nsplit - 1) * L.R;
            x[u] = *reinterpret_cast<const f32x2*>(ml + at * 2);
            y[u] = *reinterpret_cast<const f32x4*>(p.ws + at * L.dvw + d);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s0 + u >= L.nsplit) break;
            const float f = __builtin_amdgcn_exp2f(x[u][0] - M);
            Z += x[u][1] * f;
            o += y[u] * f;
        }
    }
    const float inv = Z > 0.f ? 1.0f / Z : Z != Z ? Z : 0.f;
    T* out = reinterpret_cast<T*>(p.out) + ((int64_t)(q0 + row / p.g) * p.H + kvh * p.g + row % p.g) * p.DV + d;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (d + e < p.DV) out[e] = (T)(o[e] * inv);
}

// The tile shapes: rows per workgroup as many as leave two workgroups per CU in 160 KB of LDS (one for the wide heads)
enum Shape { kNone, k64, k128, k256, kShared320, kShared576 };

Shape shape_of(const XattnParams& p) {
    if (p.k_cache == p.v_cache && p.ldk == p.ldv)
        return p.DKp <= 320 && p.DVp <= 256 ? kShared320 : p.DKp <= 576 && p.DVp <= 512 ? kShared576 : kNone;
    const int w = p.DKp > p.DVp ? p.DKp : p.DVp;
    return w <= 64 ? k64 : w <= 128 ? k128 : w <= 256 ? k256 : kNone;
}

// room: bytes of scratch that are enough for this call and for the same one with fewer keys, whose rounded splits may be more of them
F32Launch plan(const XattnParams& p, Shape s, long keys, size_t* room = nullptr) {
    static const int wide[] = {0, 4, 4, 2, 2, 2}, dvw[] = {0, 64, 128, 256, 256, 512}, kt[] = {0, 64, 32, 32, 32, 32};
    const int64_t rows = (int64_t)p.n_max * p.g, items = (int64_t)p.KH * p.B, tiles = (keys + kt[s] - 1) / kt[s];
    F32Launch L;
    L.dvw = dvw[s];
    auto with_rows = [&](int R) {
        L.R = R;
        L.nq = (int)((rows + R - 1) / R);
        // two workgroups per CU; a split has at least four tiles, so that its first loads and its share of the merge are a small part
        const int64_t groups = L.nq * items, want = groups > 0 ? (512 + groups - 1) / groups : 1;
        L.nsplit = (int)std::max<int64_t>(1, std::min<int64_t>({want, keys / (4 * kt[s]), 64}));
        return groups * L.nsplit;
    };
    // Sixteen rows a workgroup: a tile is 1.5 to 2 us of a step, one more split to merge 0.2, so splits go down to two tiles of the
    // longest page table, none of them without a tile there, and four tiles stay whole (130 keys 13.9 us whole, 14.8 in two).  A shorter
    // sequence beside the longest has as many splits, of fewer tiles, the last ones of none.  us, at least four tiles a split / now, 8 kv
    // heads of 64: one request of 600 keys 22.8 / 15.5, of 2 000 25.0 / 20.5, 6 of 300 20.3 / 16.5, of 1 500 29.2 / 25.3, 12 of 600 25.9 /
    // 21.5, 16 of 2 000 51.6 / 50.9.  Heads above 128, one workgroup a CU: 5 x 8 kv heads of 256, 600 keys 33.8 / 33.0, 6 of 8, 790
    // 56.9 / 40.2, but unequal sequences of more than 32 pairs level out with more splits than one round of CUs (7 x 8, to 1 587 keys 65.5 /
    // 73.8, 11 x 8 95.5 / 137): as above.
    // (returns the most splits of as many keys or fewer: 64 over 128 tiles, 43 of three over 129)
    auto few_rows = [&]() -> int64_t {
        with_rows(16);
        const int64_t groups = L.nq * items;
        const bool two = s == k64 || s == k128;
        if (groups <= 0 || (!two && groups > 32)) return L.nsplit;
        const int64_t want = two ? (512 + groups - 1) / groups : 256 / groups;
        const int64_t n = std::max<int64_t>(1, std::min<int64_t>({want, tiles < 5 ? 1 : tiles / 2, 64})), per = (tiles + n - 1) / n;
        L.nsplit = per > 0 ? (int)((tiles + per - 1) / per) : 1;
        return n;
    };
    // Wide row groups reuse a tile's keys, 16 rows are the shorter chain: ahead by a fifth to a third while the wide ones are not half as
    // many workgroups as there are CUs (32 query heads of 64, 20 rows over 20 keys: 16.2 -> 11.6 us with the keys of a tile that are not
    // there left out; 16 rows over 1 500: x 0.7).  A wavefront's own rows (heads to 128) are level at 100 workgroups (13 x 8: 22.1 and 23.3;
    // 48 x 2: 28.3 and 26.0), ahead at 128 (8 x 60 rows, 16 / 4 heads of 128: 21.5 and 19.2).  Wider heads, two tiles of 16 rows together, are
    // ahead where those tiles would be more than one a CU: 17 requests of 20 rows, heads of 256 (136) 53.4 and 34.9 us, of 32 rows 56.1 and
    // 38.7, but 16 of 32 (128) 30.2 and 33.0, 4 of 128 26.2 and 30.1.
    const long line = s == k64 || s == k128 ? 128 : 129;
    auto bytes = [&](int64_t splits) { return splits == 1 ? (size_t)0 : (size_t)(items * L.nq * splits * L.R) * (L.dvw + 2) * 4; };
    const bool few = rows <= 16 || with_rows(16 * wide[s]) < line;
    if (few) {
        const int64_t most = few_rows();
        if (room) *room = bytes(most);
    } else if (room) {
        const F32Launch W = L;
        *room = bytes(L.nsplit);
        if (W.nq * items < line) *room = std::max(*room, bytes(few_rows()));        // (behind fewer keys on 16 rows)
        L = W;
    }
    return L;
}

template <typename T, int DK, int DV, int QT, int KT, bool SHARED>
int launch(const XattnParams& p, const F32Launch& L, hipStream_t st) {
    constexpr int bytes = f32_lds_bytes<DK, DV, QT, KT, SHARED>();
    static_assert(bytes <= 160 * 1024, "LDS");
    static MdPerDeviceOnce once;
    if (bytes > 64 * 1024 && once.first()) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&xattn_f32_kernel<T, DK, DV, QT, KT, SHARED>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
            once.undo();
            md_set_error("attention: cannot raise the LDS limit to %d bytes", bytes);
            return MD_ERR_LAUNCH;
        }
    }
    hipLaunchKernelGGL((xattn_f32_kernel<T, DK, DV, QT, KT, SHARED>), dim3((unsigned)(L.nq * L.nsplit), p.KH, p.B), dim3(256), bytes,
                       st, p, L);
    if (L.nsplit > 1) {
        const int64_t threads = (int64_t)p.B * p.KH * L.nq * L.R * (L.dvw / 4);
        hipLaunchKernelGGL((xattn_f32_merge_kernel<T>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, p, L);
    }
    MD_CHECK_LAUNCH("attention(32-bit)");
    return MD_OK;
}

template <typename T, int DK, int DV, int KT, int NW, int OCC>
int launch_rows(const XattnParams& p, const F32Launch& L, hipStream_t st) {
    constexpr int bytes = rows_lds_bytes<DK, DV, KT>();
    static_assert(bytes <= 160 * 1024, "LDS");
    static MdPerDeviceOnce once;
    if (bytes > 64 * 1024 && once.first()) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&xattn_f32_rows_kernel<T, DK, DV, KT, NW, OCC>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
            once.undo();
            md_set_error("attention: cannot raise the LDS limit to %d bytes", bytes);
            return MD_ERR_LAUNCH;
        }
    }
    hipLaunchKernelGGL((xattn_f32_rows_kernel<T, DK, DV, KT, NW, OCC>), dim3((unsigned)(p.KH * p.B * L.nq * L.nsplit)), dim3(64 * NW),
                       bytes, st, p, L);
    if (L.nsplit > 1) {
        const int64_t threads = (int64_t)p.B * p.KH * L.nq * L.R * (L.dvw / 4);
        hipLaunchKernelGGL((xattn_f32_merge_kernel<T>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, p, L);
    }
    MD_CHECK_LAUNCH("attention(32-bit)");
    return MD_OK;
}

template <typename T>
int launch_shape(const XattnParams& p, Shape s, const F32Launch& L, hipStream_t st) {
    const bool few = L.R == 16;
    switch (s) {
    case k64: return few ? launch<T, 64, 64, 1, 64, false>(p, L, st) : launch_rows<T, 64, 64, 32, 4, 4>(p, L, st);
    case k128: return few ? launch<T, 128, 128, 1, 32, false>(p, L, st) : launch_rows<T, 128, 128, 32, 4, 2>(p, L, st);
    case k256: return few ? launch<T, 256, 256, 1, 32, false>(p, L, st) : launch<T, 256, 256, 2, 32, false>(p, L, st);
    case kShared320: return few ? launch<T, 320, 256, 1, 32, true>(p, L, st) : launch<T, 320, 256, 2, 32, true>(p, L, st);
    default: return few ? launch<T, 576, 512, 1, 32, true>(p, L, st) : launch<T, 576, 512, 2, 32, true>(p, L, st);
    }
}

}  // namespace

size_t md_internal_xattn_f32_workspace(const XattnParams& p, long keys) {
    const Shape s = shape_of(p);
    if (s == kNone) return 0;
    size_t room = 0;
    plan(p, s, keys, &room);
    return room;
}

bool md_internal_xattn_f32_ok(const XattnParams& p) { return shape_of(p) != kNone && p.page_size % 32 == 0; }

int md_internal_xattn_f32(const XattnParams& p, int dtype, long keys, hipStream_t st) {
    const Shape s = shape_of(p);
    F32Launch L = plan(p, s, keys);
    if (!p.ws) L.nsplit = 1;
    return dtype == MD_T_F32 ? launch_shape<float>(p, s, L, st) : launch_shape<bf16_t>(p, s, L, st);
}
