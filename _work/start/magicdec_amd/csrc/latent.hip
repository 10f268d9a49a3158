// Latent attention (gfx950): keys and values of every head are linear maps of one small latent row per token, and one rotated
// key part is shared by all heads, so a cache row is  latent (kv_rank) | rotated key part (rot_dim) | zeros up to W.
//   score(t, s, h) = (qn_th . K_h c_s + rot(qr_th) . r_s) * scale,   o_th = sum_s p_ts (V_h c_s)
// Two forms of the same sums:
//   absorbed   K_h moves to the query, V_h behind the sum: scores are (K_h^T qn | rot(qr)) . (c | r), one query of W numbers per
//              (token, head) against rows every head shares -- a multi-query attention whose value row is a prefix of its key row.
//              A cached row is read once for all heads: decoding.
//   expanded   keys and values of the context are computed (one library product over the gathered latents) and attended per
//              head with dim + rot_dim and vdim numbers: several times fewer operations per (query, key): prompts.
//
//   md_latent_append     query latent -> weighted RMS norm; latent -> weighted RMS norm, key part -> rotation, both -> cache
//   md_latent_query      both for a step's rows, and the queries of the normalised query latents, in one launch
//   md_head_linear       y[row][h] = W_h x[row][h]: the absorbed queries (+ their rotated part) and the way out of the latent
//                        (* sigmoid of the head's gate)
//   md_latent_attn       the absorbed form over the cache; 32-bit and unusual sizes run the fp32 attention kernels of xattn_f32.hip or,
//                        beyond their sizes, the plain one of xattn.hip
//   md_latent_gather     latents of a paged context as dense rows
//   md_latent_prefill    the expanded form
// Positions, angles, norms, scores, softmax weights and gates are fp32.
#include "latent.h"
#include "xattn.h"

#include <algorithm>

unsigned int* md_page_overflow_counter_device();   // kvops.hip

namespace {

constexpr int kMaxRow = 1024;

// ------------------------------------------------------------------------------------------------ norms, rotation, append
template <typename T, int VEC>
__device__ __forceinline__ void ld_piece(const T* p, float (&f)[VEC]) {
    typedef T vec __attribute__((ext_vector_type(VEC)));
    if constexpr (VEC == 1) {
        f[0] = (float)p[0];
    } else {
        const vec v = *reinterpret_cast<const vec*>(p);
#pragma unroll
        for (int e = 0; e < VEC; ++e) f[e] = (float)v[e];
    }
}
template <typename T, int VEC>
__device__ __forceinline__ void st_piece(T* p, const float (&f)[VEC]) {
    typedef T vec __attribute__((ext_vector_type(VEC)));
    if constexpr (VEC == 1) {
        p[0] = (T)f[0];
    } else {
        vec v;
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] = (T)f[e];
        *reinterpret_cast<vec*>(p) = v;
    }
}

// dst = src / sqrt(mean(src^2) + eps) * w by one wavefront
template <typename T, int VEC>
__device__ __forceinline__ void norm_row(const T* src, const T* w, T* dst, int n, float eps, int lane) {
    float ss = 0.f, f[VEC], g[VEC];
    for (int d = lane * VEC; d < n; d += 64 * VEC) {
        ld_piece<T, VEC>(src + d, f);
#pragma unroll
        for (int e = 0; e < VEC; ++e) ss += f[e] * f[e];
    }
    const float rs = 1.0f / sqrtf(wave_reduce_sum(ss) / (float)n + eps);
    for (int d = lane * VEC; d < n; d += 64 * VEC) {
        ld_piece<T, VEC>(src + d, f);
        ld_piece<T, VEC>(w + d, g);
#pragma unroll
        for (int e = 0; e < VEC; ++e) f[e] = (f[e] * rs) * g[e];
        st_piece<T, VEC>(dst + d, f);
    }
}

// element d of a rotated vector (neighbouring pairs of the first 2 * pairs elements turn, the rest pass)
template <typename T>
__device__ __forceinline__ float rotated(const T* x, int d, int pairs, const float* cs) {
    const float a = (float)x[d];
    if (d >= 2 * pairs) return a;
    const float b = (float)x[d ^ 1], c = cs[d & ~1], s = cs[d | 1];      // cs = (cos, sin) of every pair
    return d & 1 ? a * c + b * s : a * c - b * s;
}

// row j of request b, a row of z: its latent, normalised, and its key part, rotated, to its position's cache row; by one wavefront
template <typename T, int VEC>
__device__ __forceinline__ void append_row(const LatentParams& p, const T* row, int b, int j, int lane) {
    const int pos = p.pos0[b] + j, pg0 = p.page_indptr[b];
    if (pos < 0 || pos >= (p.page_indptr[b + 1] - pg0) * p.page_size || pos >= p.max_pos) {
        if (lane == 0) atomicAdd(p.overflow, 1u);
        return;
    }
    T* dst = reinterpret_cast<T*>(p.cache) +
             ((int64_t)p.page_indices[pg0 + pos / p.page_size] * p.page_size + pos % p.page_size) * p.W;
    const T* src = row + p.q_rank;
    norm_row<T, VEC>(src, reinterpret_cast<const T*>(p.kv_norm), dst, p.kv_rank, p.eps, lane);
    const float* cs = p.cos_sin + (int64_t)pos * p.rot_pairs * 2;
    for (int d = lane; d < p.W - p.kv_rank; d += 64)
        dst[p.kv_rank + d] = d < p.rot_dim ? (T)rotated(src + p.kv_rank, d, p.rot_pairs, cs) : (T)0.f;
}

// two wavefronts per row: one normalises the query latent, the other the latent and rotates the key part
template <typename T, int VEC>
__global__ __launch_bounds__(256) void latent_append_kernel(const LatentParams p) {
    const int b = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int q0 = p.qo_indptr[b], j = blockIdx.x * 2 + (wave >> 1);
    if (j >= p.qo_indptr[b + 1] - q0) return;
    const T* row = reinterpret_cast<const T*>(p.z) + (int64_t)(q0 + j) * p.ldz;
    if ((wave & 1) == 0) {
        norm_row<T, VEC>(row, reinterpret_cast<const T*>(p.dq_norm), reinterpret_cast<T*>(p.cq) + (int64_t)(q0 + j) * p.q_rank,
                         p.q_rank, p.eps, lane);
        return;
    }
    if (p.append) append_row<T, VEC>(p, row, b, j, lane);
}

// ------------------------------------------------------------------------------------------------ queries of a step
// q[M][N] = rms(query latent) * dq_norm . W^T with W in the streaming layout [N/32][K/16][64][8] (K = 256 STEPS), and beside it, in workgroups
// behind the product's, the append.  A workgroup has 32 rows x 32 columns, each of its sixteen wavefronts a sixteenth of K: all that a wavefront
// reads is requested at once, and the norm is formed of what it holds while the weight is on its way: rounded where latent_append_kernel
// rounds, its sum of squares of another order, so that a latent may round the other way.  The appended row is that kernel's bit for bit.
//
// A chain of latencies bounds a step of few rows: as launches of their own the norm and append take 4.6 us and the product 4.6 (32 rows of
// 3 072 x 768), this 5.3.
template <int STEPS>
__global__ __launch_bounds__(1024, 4) void latent_query_kernel(const LatentParams p, const bf16_t* w, bf16_t* q, int64_t ldq, int M, int N) {
    constexpr int NW = 16, K = 16 * NW * STEPS;
    __shared__ float part[NW * 32];
    extern __shared__ __attribute__((aligned(16))) float red[];            // [NW][32][32]
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), m_tiles = (M + 31) / 32, tiles = N / 32 * m_tiles;
    const bf16_t* z = reinterpret_cast<const bf16_t*>(p.z);
    if ((int)blockIdx.x >= tiles) {
        const int row = ((int)blockIdx.x - tiles) * NW + wave;
        if (row >= M) return;
        int b = 0;                                                          // requests that end in front of the row
        for (int i = 0; i < p.B; i += 64) b += __popcll(__builtin_amdgcn_ballot_w64(i + lane < p.B && p.qo_indptr[i + lane + 1] <= row));
        if (b < p.B) append_row<bf16_t, 8>(p, z + (int64_t)row * p.ldz, b, row - p.qo_indptr[b], lane);
        return;
    }
    const int tn = blockIdx.x / m_tiles, m0 = (int)blockIdx.x % m_tiles * 32, k0 = wave * STEPS * 16 + kh * 8;
    const bf16_t* xp = z + (int64_t)min(m0 + j, M - 1) * p.ldz + k0;
    const bf16_t* gp = reinterpret_cast<const bf16_t*>(p.dq_norm) + k0;
    const bf16_t* wp = w + ((int64_t)tn * (K / 16) + wave * STEPS) * 512 + lane * 8;
    bf16x8 x[STEPS], g[STEPS], b[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) x[s] = *reinterpret_cast<const bf16x8*>(xp + s * 16);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) g[s] = *reinterpret_cast<const bf16x8*>(gp + s * 16);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) b[s] = *reinterpret_cast<const bf16x8*>(wp + s * 512);
    float ss = 0.f;
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += (float)x[s][e] * (float)x[s][e];
    ss += __shfl_xor(ss, 32);
    if (kh == 0) part[wave * 32 + j] = ss;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                      // (the weight stays on its way)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) t += part[i * 32 + j];
    const float rs = 1.0f / sqrtf(t / (float)K + p.eps);
    typedef float f32x16 __attribute__((ext_vector_type(16)));
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        bf16x8 a;
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = (bf16_t)(((float)x[s][e] * rs) * (float)g[s][e]);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[s], acc, 0, 0, 0);
    }
    // acc[r]: row (r & 3) + 8 (r >> 2) + 4 kh, column j
#pragma unroll
    for (int r = 0; r < 16; ++r) red[wave * 1024 + ((r & 3) + 8 * (r >> 2) + 4 * kh) * 32 + j] = acc[r];
    __syncthreads();
    const int row = tid >> 5, col = tid & 31;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) sum += red[i * 1024 + tid];
    if (m0 + row < M) q[(int64_t)(m0 + row) * ldq + tn * 32 + col] = (bf16_t)sum;
}

template <int STEPS>
int launch_query(const LatentParams& p, const bf16_t* w, bf16_t* q, int64_t ldq, int M, int N, hipStream_t st) {
    constexpr int bytes = 16 * 4096;
    static MdPerDeviceOnce once;
    if (once.first() && hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_query_kernel<STEPS>),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
        once.undo();
        md_set_error("md_latent_query: hipFuncSetAttribute(LDS) failed");
        return MD_ERR_LAUNCH;
    }
    const int blocks = N / 32 * ((M + 31) / 32) + (p.append ? (M + 15) / 16 : 0);
    hipLaunchKernelGGL((latent_query_kernel<STEPS>), dim3(blocks), dim3(1024), bytes, st, p, w, q, ldq, M, N);
    return MD_OK;
}

// ------------------------------------------------------------------------------------------------ per-head linear
struct HeadLinearParams {
    const void* x;
    const void* w;            // [H][N][K]
    void* out;
    const void* gate;         // [M][ld_gate] or null: y *= sigmoid(gate[row][h])
    // a rotated tail behind the N outputs of a head: out[row][h][N + d] = rotated(tail[row][h])[d], zeros up to tail_pad
    const void* tail;
    const float* cos_sin;
    const int32_t* qo_indptr;
    const int32_t* pos0;
    int64_t ldx, hx, ldo, ho, ld_gate, ldt, ht;
    int M, H, N, K, B, tail_dim, tail_pad, rot_pairs, max_pos;
};

__device__ __forceinline__ float sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }

template <typename T>
__device__ __forceinline__ void head_tail(const HeadLinearParams& p, int h, int row0, int nrow) {
    // the column blocks of a row tile share its tail: this block's rows are row0 + blockIdx.x, + gridDim.x, ...
    __shared__ int s_pos[64];
    if (threadIdx.x < nrow) {
        const int row = min(row0 + (int)threadIdx.x, p.M - 1);
        int lo = 0, hi = p.B;                                       // request of the row: qo_indptr[lo] <= row < qo_indptr[lo + 1]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (p.qo_indptr[mid] <= row) lo = mid; else hi = mid;
        }
        s_pos[threadIdx.x] = min(max(p.pos0[lo] + row - p.qo_indptr[lo], 0), p.max_pos - 1);
    }
    __syncthreads();
    const int mine = (nrow - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
    for (int i = threadIdx.x; i < mine * p.tail_pad; i += 256) {
        const int r = blockIdx.x + i / p.tail_pad * gridDim.x, d = i % p.tail_pad, row = row0 + r;
        if (row >= p.M) break;
        const float v = d < p.tail_dim ? rotated(reinterpret_cast<const T*>(p.tail) + row * p.ldt + h * p.ht, d, p.rot_pairs,
                                                 p.cos_sin + (int64_t)s_pos[r] * p.rot_pairs * 2) : 0.f;
        (reinterpret_cast<T*>(p.out) + row * p.ldo + h * p.ho)[p.N + d] = (T)v;
    }
}

// 16-bit: 64 columns x 16 RT rows of one head per workgroup, 16 columns per wavefront, operands straight from memory
template <int RT, bool VEC>
__global__ __launch_bounds__(256) void head_linear_mfma_kernel(const HeadLinearParams p) {
    const int lane = threadIdx.x & 63, lq = lane & 15, lc = lane >> 4, wave = threadIdx.x >> 6;
    const int h = blockIdx.z, row0 = blockIdx.y * 16 * RT, n0 = blockIdx.x * 64 + wave * 16;
    if (p.tail) head_tail<bf16_t>(p, h, row0, 16 * RT);
    const bf16x8 z8 = {0, 0, 0, 0, 0, 0, 0, 0};
    auto piece = [&](const bf16_t* src, int k, bool ok) {
        if (VEC) return ok && k < p.K ? *reinterpret_cast<const bf16x8*>(src + k) : z8;
        bf16x8 v = z8;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (ok && k + e < p.K) v[e] = src[k + e];
        return v;
    };
    if (n0 < p.N) {
        const int n = n0 + lq;
        const bool n_ok = n < p.N;
        const bf16_t* wp = reinterpret_cast<const bf16_t*>(p.w) + ((int64_t)h * p.N + (n_ok ? n : 0)) * p.K;
        const bf16_t* xp[RT];
        bool r_ok[RT];
        f32x4 acc[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int row = row0 + r * 16 + lq;
            r_ok[r] = row < p.M;
            xp[r] = reinterpret_cast<const bf16_t*>(p.x) + (int64_t)(r_ok[r] ? row : 0) * p.ldx + h * p.hx;
            acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        for (int kb = 0; kb < p.K; kb += 128) {                     // four steps requested together (zeros past K)
            bf16x8 wf[4], xf[4][RT];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                wf[u] = piece(wp, kb + u * 32 + lc * 8, n_ok);
#pragma unroll
                for (int r = 0; r < RT; ++r) xf[u][r] = piece(xp[r], kb + u * 32 + lc * 8, r_ok[r]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int r = 0; r < RT; ++r) acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], xf[u][r], acc[r], 0, 0, 0);
        }
        // acc[r][e] = y[row0 + r * 16 + lq][n0 + lc * 4 + e]
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int row = row0 + r * 16 + lq, c = n0 + lc * 4;
            if (row >= p.M) continue;
            const float s = p.gate ? sigmoid((float)reinterpret_cast<const bf16_t*>(p.gate)[row * p.ld_gate + h]) : 1.f;
            bf16_t* o = reinterpret_cast<bf16_t*>(p.out) + row * p.ldo + h * p.ho + c;
            if (VEC && c + 4 <= p.N) {
                *reinterpret_cast<bf16x4*>(o) = __builtin_convertvector(acc[r] * s, bf16x4);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (c + e < p.N) o[e] = (bf16_t)(acc[r][e] * s);
            }
        }
    }
}

// 32-bit on the fp32 matrix instructions, laid out as above: a lane reads four k of a row at once, product e takes the e-th of each.  Dense
// 16-byte pieces only; the kernel below has a thread per value, which waits for every k (2 400 rows, 16 heads, 128 -> 512: 4 470 us, here 126; 8 rows: 50 and 5.8).
template <int RT>
__global__ __launch_bounds__(256) void head_linear_f32_mfma_kernel(const HeadLinearParams p) {
    const int lane = threadIdx.x & 63, lq = lane & 15, lc = lane >> 4, wave = threadIdx.x >> 6;
    const int h = blockIdx.z, row0 = blockIdx.y * 16 * RT, n0 = blockIdx.x * 64 + wave * 16;
    if (p.tail) head_tail<float>(p, h, row0, 16 * RT);
    if (n0 >= p.N) return;
    const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
    const int n = n0 + lq;
    const float* wp = reinterpret_cast<const float*>(p.w) + ((int64_t)h * p.N + min(n, p.N - 1)) * p.K;
    const float* xp[RT];
    f32x4 acc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        xp[r] = reinterpret_cast<const float*>(p.x) + (int64_t)min(row0 + r * 16 + lq, p.M - 1) * p.ldx + h * p.hx;
        acc[r] = z4;
    }
    for (int kb = 0; kb < p.K; kb += 64) {                          // four portions of 16 k requested together (zeros past K)
        f32x4 wf[4], xf[4][RT];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = kb + u * 16 + lc * 4;
            wf[u] = k < p.K ? *reinterpret_cast<const f32x4*>(wp + k) : z4;
#pragma unroll
            for (int r = 0; r < RT; ++r) xf[u][r] = k < p.K ? *reinterpret_cast<const f32x4*>(xp[r] + k) : z4;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int r = 0; r < RT; ++r) acc[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[u][e], xf[u][r][e], acc[r], 0, 0, 0);
    }
    // acc[r][e] = y[row0 + r * 16 + lq][n0 + lc * 4 + e]
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int row = row0 + r * 16 + lq, c = n0 + lc * 4;
        if (row >= p.M || c >= p.N) continue;
        const float s = p.gate ? sigmoid(reinterpret_cast<const float*>(p.gate)[row * p.ld_gate + h]) : 1.f;
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + row * p.ldo + h * p.ho + c) = acc[r] * s;
    }
}

// 32-bit of any sizes: a thread per output
__global__ __launch_bounds__(256) void head_linear_f32_kernel(const HeadLinearParams p) {
    const int h = blockIdx.z, row0 = blockIdx.y * 16, n = blockIdx.x * 16 + (threadIdx.x & 15), row = row0 + (threadIdx.x >> 4);
    if (n < p.N && row < p.M) {
        const float* w = reinterpret_cast<const float*>(p.w) + ((int64_t)h * p.N + n) * p.K;
        const float* x = reinterpret_cast<const float*>(p.x) + (int64_t)row * p.ldx + h * p.hx;
        float s = 0.f;
        for (int k = 0; k < p.K; ++k) s = fmaf(w[k], x[k], s);
        if (p.gate) s *= sigmoid(reinterpret_cast<const float*>(p.gate)[row * p.ld_gate + h]);
        (reinterpret_cast<float*>(p.out) + row * p.ldo + h * p.ho)[n] = s;
    }
    if (p.tail) head_tail<float>(p, h, row0, 16);
}

// ------------------------------------------------------------------------------------------------ merge, gather
// partials of the kv splits: ws = sums [slot][rows_wg][Rp], then (reference, weight) [slot][rows_wg][2]; slot =
// (b * groups + g) * nsplit + s.  Lane s knows split s's factor; Q wavefronts share 256 columns of one row, each adds every Q-th split
// (four requested together), and their sums meet in LDS in order
template <int Q>
__global__ __launch_bounds__(256) void latent_merge_kernel(const LatentParams p, int rows_wg, int Rp) {
    __shared__ f32x4 part[4][64];
    const int lane = threadIdx.x & 63, all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = Q == 4 ? all : 0;
    const int b = blockIdx.z, row = Q == 4 ? blockIdx.x : blockIdx.x * 4 + all, q0 = p.qo_indptr[b];
    if (row >= (p.qo_indptr[b + 1] - q0) * p.H) return;               // (Q == 4: whole workgroup)
    const int g = row / rows_wg, r = row - g * rows_wg, d = (blockIdx.y * 64 + lane) * 4;
    const int64_t slot0 = ((int64_t)b * p.n_groups + g) * p.nsplit;
    const float* ml = p.ws + (int64_t)p.B * p.n_groups * p.nsplit * rows_wg * Rp;
    f32x2 t = {-INFINITY, 0.f};
    if (lane < p.nsplit) t = *reinterpret_cast<const f32x2*>(ml + ((slot0 + lane) * rows_wg + r) * 2);
    const float m = wave_reduce_max(t[0]), w = t[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(t[0] - m);
    const float l = wave_reduce_sum(t[1] * w);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = wave; s0 < p.nsplit; s0 += 4 * Q) {
        f32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (s0 + Q * u < p.nsplit && d < Rp) v[u] = *reinterpret_cast<const f32x4*>(p.ws + ((slot0 + s0 + Q * u) * rows_wg + r) * Rp + d);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (s0 + Q * u < p.nsplit) {                              // uniform
                const float f = __shfl(w, s0 + Q * u);
                if (d < Rp) o += v[u] * f;
            }
    }
    if constexpr (Q == 4) {
        part[wave][lane] = o;
        __syncthreads();
        if (wave > 0) return;
        o = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    }
    if (d >= Rp) return;
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    bf16_t* op = reinterpret_cast<bf16_t*>(p.out) + ((int64_t)q0 * p.H + row) * p.kv_rank + d;
    if (p.kv_rank % 4 == 0) {
        if (d < p.kv_rank) *reinterpret_cast<bf16x4*>(op) = __builtin_convertvector(o * inv, bf16x4);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (d + e < p.kv_rank) op[e] = (bf16_t)(o[e] * inv);
    }
}

// one wavefront per context row
__global__ __launch_bounds__(256) void latent_gather_kernel(const LatentParams p, bf16_t* __restrict__ dst) {
    const int b = blockIdx.y, pos = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c0 = p.ctx_indptr[b];
    if (pos >= p.ctx_indptr[b + 1] - c0) return;
    const int pg0 = p.page_indptr[b];
    const bool fits = pos < (p.page_indptr[b + 1] - pg0) * p.page_size;
    const bf16_t* src = reinterpret_cast<const bf16_t*>(p.cache) +
                        (fits ? ((int64_t)p.page_indices[pg0 + pos / p.page_size] * p.page_size + pos % p.page_size) * p.W : 0);
    const u32x4 z = {0u, 0u, 0u, 0u};
    for (int d = lane * 8; d < p.kv_rank; d += 512)
        *reinterpret_cast<u32x4*>(dst + (int64_t)(c0 + pos) * p.kv_rank + d) = fits ? *reinterpret_cast<const u32x4*>(src + d) : z;
}

bool aligned(const void* q, int n) { return ((uintptr_t)q & (n - 1)) == 0; }
int row_width(int kv_rank, int rot_dim) { return (kv_rank + rot_dim + 31) / 32 * 32; }
int row_tiles(const md_latent_args* a) { return (long)a->n_max * a->H <= 16 ? 1 : 2; }
int row_groups(const md_latent_args* a) { return (int)(((long)a->n_max * a->H + 16 * row_tiles(a) - 1) / (16 * row_tiles(a))); }

bool mfma_ok(const md_latent_args* a) {
    return a->dtype == MD_T_BF16 && !a->force_plain && a->page_size % 64 == 0 &&
           md_internal_latent_absorbed_ok(a->kv_rank, row_width(a->kv_rank, a->rot_dim), row_tiles(a));
}

constexpr int kTargetWgs = 512;              // 16-row workgroups: two per CU (of 32 rows: one)

int kv_splits(const md_latent_args* a) {
    const long tiles = ((long)a->max_pages * a->page_size + 31) / 32, groups = (long)a->B * row_groups(a);
    const long target = kTargetWgs / row_tiles(a);
    long want = (target + groups - 1) / groups;
    // >= 256 keys per workgroup; a tile is a chain of two barriers, 2 us where nothing else runs on the CU, so while one workgroup per CU
    // is not reached 128 keys, and 64 up to one on every other.  Four layers, us: one request of 8 000 keys 316 -> 300, four of 1 000
    // 319 -> 295, twelve of 1 500 333 -> 319 (64 keys: 325); beyond, shorter chains lose to the merge: 32 of 2 049 at 128 keys 391 against
    // 380, 48 of 1 200 430 against 415
    // (not within a page, and within two only where the merge has little to do: one request of 75 keys 18.3 against 19.8, 31 of 137 with
    // a 512-wide latent 19.9 against 21.8, but 19 of 160 with a 256-wide one 23.5 -> 18.4)
    const bool worth = tiles > 8 || (tiles > 4 && (groups <= 16 || a->kv_rank <= 256));
    const long few = worth ? std::max(std::min(tiles / 4, target / 2 / groups), std::min(tiles / 2, target / 4 / groups)) : 0;
    const long cap = std::max(std::max(tiles / 8, few), 1L);
    if (want > cap) want = cap;
    return (int)(want < 1 ? 1 : want > 64 ? 64 : want);            // (the merge holds a split per lane)
}

int check_args(const char* who, const md_latent_args* a) {
    MD_CHECK_ARG(a && a->cache && a->qo_indptr && a->pos0 && a->page_indices && a->page_indptr, "%s: null pointer argument", who);
    MD_CHECK_ARG(a->B > 0 && a->B <= 65535 && a->n_max > 0 && a->H > 0 && a->H <= 65535, "%s: bad shape B=%d n_max=%d H=%d", who,
                 a->B, a->n_max, a->H);
    MD_CHECK_ARG(a->kv_rank > 0 && a->rot_dim > 0 && a->rot_pairs >= 0 && 2 * a->rot_pairs <= a->rot_dim &&
                     row_width(a->kv_rank, a->rot_dim) <= kMaxRow, "%s: kv_rank %d + rot_dim %d (<= %d)", who, a->kv_rank,
                 a->rot_dim, kMaxRow);
    MD_CHECK_ARG(a->page_size > 0 && a->page_size % 32 == 0 && a->max_pages > 0, "%s: page_size %d must be a multiple of 32", who,
                 a->page_size);
    MD_CHECK_ARG(a->dtype == MD_T_BF16 || a->dtype == MD_T_F32, "%s: dtype must be MD_T_BF16 or MD_T_F32", who);
    MD_CHECK_ARG(aligned(a->cache, 16), "%s: the cache must be 16-byte aligned", who);
    return MD_OK;
}

long keys_of(const md_latent_args* a) { return (long)a->max_pages * a->page_size; }

// the absorbed form as a one-kv-head attention whose values are the first kv_rank elements of its keys
XattnParams general_params(const md_latent_args* a) {
    XattnParams x = {};
    x.q = a->q;
    x.k_cache = a->cache;
    x.v_cache = a->cache;
    x.out = a->out;
    x.qo_indptr = a->qo_indptr;
    x.pos0 = a->pos0;
    x.page_indices = a->page_indices;
    x.page_indptr = a->page_indptr;
    x.B = a->B;
    x.n_max = a->n_max;
    x.H = x.g = a->H;
    x.KH = 1;
    x.D = x.DKp = x.ldk = x.ldv = row_width(a->kv_rank, a->rot_dim);
    x.DV = x.DVp = a->kv_rank;
    x.page_size = a->page_size;
    x.chunk = 0x7fffffff;
    x.scale = a->scale;
    x.scale_log2 = a->scale * 1.4426950408889634f;
    return x;
}

LatentParams make_params(const md_latent_args* a) {
    LatentParams p = {};
    p.z = a->z;
    p.dq_norm = a->dq_norm;
    p.kv_norm = a->kv_norm;
    p.cq = a->cq;
    p.cache = a->cache;
    p.cos_sin = a->cos_sin;
    p.qo_indptr = a->qo_indptr;
    p.pos0 = a->pos0;
    p.page_indices = a->page_indices;
    p.page_indptr = a->page_indptr;
    p.ctx_indptr = a->ctx_indptr;
    p.q = a->q;
    p.kv = a->kv;
    p.gate = a->gate;
    p.out = a->out;
    p.ldz = a->ldz;
    p.ldo = a->ldo;
    p.ld_gate = a->ld_gate;
    p.B = a->B;
    p.n_max = a->n_max;
    p.H = a->H;
    p.dim = a->dim;
    p.rot_dim = a->rot_dim;
    p.rot_pairs = a->rot_pairs;
    p.vdim = a->vdim;
    p.q_rank = a->q_rank;
    p.kv_rank = a->kv_rank;
    p.W = row_width(a->kv_rank, a->rot_dim);
    p.page_size = a->page_size;
    p.max_pos = a->max_pos;
    p.append = a->append;
    p.eps = a->eps;
    p.scale_log2 = a->scale * 1.4426950408889634f;
    p.overflow = md_page_overflow_counter_device();
    return p;
}

int prefill_dk(int n) { return n <= 64 ? 64 : n <= 128 ? 128 : n <= 192 ? 192 : n <= 256 ? 256 : 0; }

}  // namespace

extern "C" int md_latent_row_width(int kv_rank, int rot_dim) {
    return kv_rank > 0 && rot_dim > 0 && row_width(kv_rank, rot_dim) <= kMaxRow ? row_width(kv_rank, rot_dim) : 0;
}

extern "C" int md_latent_append(const md_latent_args* a, md_stream_t stream) {
    const int rc = check_args("md_latent_append", a);
    if (rc != MD_OK) return rc;
    MD_CHECK_ARG(a->z && a->dq_norm && a->cq && a->q_rank > 0, "md_latent_append: null pointer argument");
    MD_CHECK_ARG(!a->append || (a->kv_norm && a->cos_sin && a->max_pos > 0), "md_latent_append: the append needs kv_norm and the angle table");
    MD_CHECK_ARG(a->ldz >= a->q_rank + (a->append ? a->kv_rank + a->rot_dim : 0), "md_latent_append: rows of %lld elements are too short",
                 (long long)a->ldz);
    const LatentParams p = make_params(a);
    MD_CHECK_ARG(p.overflow, "md_latent_append: cannot resolve the page-overflow counter");
    const dim3 grid((a->n_max + 1) / 2, a->B);
    const bool vec = a->q_rank % 8 == 0 && a->kv_rank % 8 == 0 && a->ldz % 8 == 0 && aligned(a->z, 32) && aligned(a->cq, 32) &&
                     aligned(a->cache, 32) && aligned(a->dq_norm, 32) && (!a->append || aligned(a->kv_norm, 32));
    hipStream_t st = (hipStream_t)stream;
    if (a->dtype == MD_T_F32) {
        if (vec) hipLaunchKernelGGL((latent_append_kernel<float, 8>), grid, dim3(256), 0, st, p);
        else hipLaunchKernelGGL((latent_append_kernel<float, 1>), grid, dim3(256), 0, st, p);
    } else {
        if (vec) hipLaunchKernelGGL((latent_append_kernel<bf16_t, 8>), grid, dim3(256), 0, st, p);
        else hipLaunchKernelGGL((latent_append_kernel<bf16_t, 1>), grid, dim3(256), 0, st, p);
    }
    MD_CHECK_LAUNCH("md_latent_append");
    return MD_OK;
}

extern "C" int md_latent_query_supported(int M, int N, int q_rank) {
    MD_CHECK_ARG(M > 0 && N > 0 && q_rank > 0, "md_latent_query_supported: M=%d N=%d q_rank=%d", M, N, q_rank);
    // a workgroup a CU: 64 rows of 3 072 columns, not of 6 144 (384 workgroups: four layers 571 us a step as two launches, 582 as one)
    return M <= 64 && N % 32 == 0 && N / 32 * ((M + 31) / 32) <= 256 && q_rank % 256 == 0 && q_rank <= 1536 ? 1 : 0;
}

extern "C" int md_latent_query(const md_latent_args* a, const void* w_packed, void* q, int64_t ldq, int M, int N, md_stream_t stream) {
    const int rc = check_args("md_latent_query", a);
    if (rc != MD_OK) return rc;
    MD_CHECK_ARG(a->z && a->dq_norm && w_packed && q, "md_latent_query: null pointer argument");
    MD_CHECK_ARG(M > 0 && N > 0 && a->q_rank > 0 && md_latent_query_supported(M, N, a->q_rank) && a->dtype == MD_T_BF16 && ldq >= N,
                 "md_latent_query: M=%d N=%d q_rank=%d unsupported", M, N, a->q_rank);
    MD_CHECK_ARG(!a->append || (a->kv_norm && a->cos_sin && a->max_pos > 0), "md_latent_query: the append needs kv_norm and the angle table");
    MD_CHECK_ARG(a->ldz >= a->q_rank + (a->append ? a->kv_rank + a->rot_dim : 0) && a->ldz % 8 == 0 && a->kv_rank % 8 == 0 && aligned(a->z, 16) &&
                     aligned(a->dq_norm, 16) && aligned(w_packed, 16) && aligned(a->cache, 32) && (!a->append || aligned(a->kv_norm, 16)),
                 "md_latent_query: rows of %lld elements, or operands that are not 16-byte aligned", (long long)a->ldz);
    const LatentParams p = make_params(a);
    MD_CHECK_ARG(p.overflow, "md_latent_query: cannot resolve the page-overflow counter");
    const bf16_t* w = (const bf16_t*)w_packed;
    bf16_t* out = (bf16_t*)q;
    hipStream_t st = (hipStream_t)stream;
    int r = MD_OK;
    switch (a->q_rank / 256) {
    case 1: r = launch_query<1>(p, w, out, ldq, M, N, st); break;
    case 2: r = launch_query<2>(p, w, out, ldq, M, N, st); break;
    case 3: r = launch_query<3>(p, w, out, ldq, M, N, st); break;
    case 4: r = launch_query<4>(p, w, out, ldq, M, N, st); break;
    case 5: r = launch_query<5>(p, w, out, ldq, M, N, st); break;
    default: r = launch_query<6>(p, w, out, ldq, M, N, st);
    }
    if (r != MD_OK) return r;
    MD_CHECK_LAUNCH("md_latent_query");
    return MD_OK;
}

// 16-row tiles of a head_linear wavefront: as many as leave every CU a workgroup
static int row_tiles(const md_head_linear_args* a) {
    const long columns = (long)((a->N + 63) / 64) * a->H;
    return columns * ((a->M + 63) / 64) >= 256 ? 4 : columns * ((a->M + 31) / 32) >= 256 ? 2 : 1;
}

extern "C" int md_head_linear(const md_head_linear_args* a, md_stream_t stream) {
    MD_CHECK_ARG(a && a->x && a->w && a->out, "md_head_linear: null pointer argument");
    MD_CHECK_ARG(a->M > 0 && a->H > 0 && a->H <= 65535 && a->N > 0 && a->K > 0, "md_head_linear: bad shape M=%d H=%d N=%d K=%d", a->M,
                 a->H, a->N, a->K);
    MD_CHECK_ARG(a->dtype == MD_T_BF16 || a->dtype == MD_T_F32, "md_head_linear: dtype must be MD_T_BF16 or MD_T_F32");
    MD_CHECK_ARG(!a->tail || (a->cos_sin && a->qo_indptr && a->pos0 && a->B > 0 && a->tail_pad >= a->tail_dim && a->tail_dim > 0 &&
                              2 * a->rot_pairs <= a->tail_dim && a->rot_pairs >= 0 && a->max_pos > 0),
                 "md_head_linear: the rotated tail needs positions and the angle table");
    HeadLinearParams p = {};
    p.x = a->x;
    p.w = a->w;
    p.out = a->out;
    p.gate = a->gate;
    p.tail = a->tail;
    p.cos_sin = a->cos_sin;
    p.qo_indptr = a->qo_indptr;
    p.pos0 = a->pos0;
    p.ldx = a->ldx;
    p.hx = a->hx;
    p.ldo = a->ldo;
    p.ho = a->ho;
    p.ld_gate = a->ld_gate;
    p.ldt = a->ldt;
    p.ht = a->ht;
    p.M = a->M;
    p.H = a->H;
    p.N = a->N;
    p.K = a->K;
    p.B = a->B;
    p.tail_dim = a->tail_dim;
    p.tail_pad = a->tail_pad;
    p.rot_pairs = a->rot_pairs;
    p.max_pos = a->max_pos;
    hipStream_t st = (hipStream_t)stream;
    if (a->dtype == MD_T_F32) {
        MD_CHECK_ARG((a->M + 15) / 16 <= 65535, "md_head_linear: %d rows", a->M);
        if (a->K % 4 == 0 && a->N % 4 == 0 && a->ldx % 4 == 0 && a->hx % 4 == 0 && a->ldo % 4 == 0 && a->ho % 4 == 0 && aligned(a->x, 16) &&
            aligned(a->w, 16) && aligned(a->out, 16)) {
            const int rt = row_tiles(a);
            const dim3 grid((a->N + 63) / 64, (a->M + 16 * rt - 1) / (16 * rt), a->H);
            if (rt == 4) hipLaunchKernelGGL(head_linear_f32_mfma_kernel<4>, grid, dim3(256), 0, st, p);
            else if (rt == 2) hipLaunchKernelGGL(head_linear_f32_mfma_kernel<2>, grid, dim3(256), 0, st, p);
            else hipLaunchKernelGGL(head_linear_f32_mfma_kernel<1>, grid, dim3(256), 0, st, p);
            MD_CHECK_LAUNCH("md_head_linear");
            return MD_OK;
        }
        hipLaunchKernelGGL(head_linear_f32_kernel, dim3((a->N + 15) / 16, (a->M + 15) / 16, a->H), dim3(256), 0, st, p);
        MD_CHECK_LAUNCH("md_head_linear");
        return MD_OK;
    }
    const bool vec = a->K % 8 == 0 && a->ldx % 8 == 0 && a->hx % 8 == 0 && a->ldo % 4 == 0 && a->ho % 4 == 0 && aligned(a->x, 16) &&
                     aligned(a->w, 16) && aligned(a->out, 8);
    const int rt = row_tiles(a);
    const dim3 grid((a->N + 63) / 64, (a->M + 16 * rt - 1) / (16 * rt), a->H);
    MD_CHECK_ARG(grid.y <= 65535, "md_head_linear: %d rows", a->M);
#define MD_HL(RT)                                                                                               \
    do {                                                                                                        \
        if (vec) hipLaunchKernelGGL((head_linear_mfma_kernel<RT, true>), grid, dim3(256), 0, st, p);            \
        else hipLaunchKernelGGL((head_linear_mfma_kernel<RT, false>), grid, dim3(256), 0, st, p);               \
    } while (0)
    if (rt == 4) MD_HL(4);
    else if (rt == 2) MD_HL(2);
    else MD_HL(1);
#undef MD_HL
    MD_CHECK_LAUNCH("md_head_linear");
    return MD_OK;
}

extern "C" size_t md_latent_workspace_bytes(const md_latent_args* a) {
    if (!a) return 0;
    if (!mfma_ok(a)) return a->force_plain ? 0 : md_internal_xattn_f32_workspace(general_params(a), keys_of(a));
    const int ns = kv_splits(a);
    if (ns == 1) return 0;
    const size_t Rp = (a->kv_rank + 15) / 16 * 16;
    return (size_t)a->B * row_groups(a) * ns * 16 * row_tiles(a) * (Rp + 2) * 4;
}

extern "C" int md_latent_attn(const md_latent_args* a, md_stream_t stream) {
    int rc = check_args("md_latent_attn", a);
    if (rc != MD_OK) return rc;
    MD_CHECK_ARG(a->q && a->out && aligned(a->q, 16) && aligned(a->out, 8), "md_latent_attn: q and out (16-byte aligned) are needed");
    hipStream_t st = (hipStream_t)stream;
    LatentParams p = make_params(a);
    if (!mfma_ok(a)) {
        XattnParams x = general_params(a);
        if (a->force_plain || !md_internal_xattn_f32_ok(x)) return md_internal_xattn_plain(x, a->dtype, st);
        const size_t need = md_latent_workspace_bytes(a);
        if (need && a->workspace && a->workspace_bytes >= need && aligned(a->workspace, 16)) x.ws = (float*)a->workspace;
        return md_internal_xattn_f32(x, a->dtype, keys_of(a), st);
    }
    const int qt = row_tiles(a);
    p.n_groups = row_groups(a);
    p.nsplit = kv_splits(a);
    if (p.nsplit > 1) {
        MD_CHECK_ARG(a->workspace && a->workspace_bytes >= md_latent_workspace_bytes(a) && aligned(a->workspace, 16),
                     "md_latent_attn: workspace of %zu bytes needed, got %zu", md_latent_workspace_bytes(a), a->workspace_bytes);
        p.ws = (float*)a->workspace;
    }
    rc = md_internal_latent_absorbed(p, qt, st);
    if (rc != MD_OK) return rc;
    if (p.nsplit > 1) {
        const int Rp = (a->kv_rank + 15) / 16 * 16;
        const int rows = a->n_max * a->H, cols = (Rp + 255) / 256;
        if (p.nsplit > 8) hipLaunchKernelGGL((latent_merge_kernel<4>), dim3(rows, cols, a->B), dim3(256), 0, st, p, 16 * qt, Rp);
        else hipLaunchKernelGGL((latent_merge_kernel<1>), dim3((rows + 3) / 4, cols, a->B), dim3(256), 0, st, p, 16 * qt, Rp);
    }
    MD_CHECK_LAUNCH("md_latent_attn");
    return MD_OK;
}

extern "C" int md_latent_gather(const md_latent_args* a, int ctx_max, void* dst, md_stream_t stream) {
    const int rc = check_args("md_latent_gather", a);
    if (rc != MD_OK) return rc;
    MD_CHECK_ARG(a->ctx_indptr && dst && aligned(dst, 16) && ctx_max > 0 && a->kv_rank % 8 == 0 && a->dtype == MD_T_BF16,
                 "md_latent_gather: needs context lengths, bf16 and kv_rank %% 8 == 0");
    const LatentParams p = make_params(a);
    hipLaunchKernelGGL(latent_gather_kernel, dim3((ctx_max + 3) / 4, a->B), dim3(256), 0, (hipStream_t)stream, p, (bf16_t*)dst);
    MD_CHECK_LAUNCH("md_latent_gather");
    return MD_OK;
}

extern "C" int md_latent_prefill_supported(const md_latent_args* a) {
    return a && a->dtype == MD_T_BF16 && a->dim > 0 && a->dim % 8 == 0 && a->rot_dim % 8 == 0 && a->vdim > 0 && a->vdim % 8 == 0 &&
           a->kv_rank % 8 == 0 && prefill_dk(a->dim + a->rot_dim) && prefill_dk(a->vdim) && a->page_size % 64 == 0 ? 1 : 0;
}

extern "C" int md_latent_prefill(const md_latent_args* a, md_stream_t stream) {
    const int rc0 = check_args("md_latent_prefill", a);
    if (rc0 != MD_OK) return rc0;
    MD_CHECK_ARG(md_latent_prefill_supported(a), "md_latent_prefill: unsupported sizes (md_latent_prefill_supported)");
    MD_CHECK_ARG(a->q && a->kv && a->ctx_indptr && a->cos_sin && a->out && a->max_pos > 0 && aligned(a->q, 16) && aligned(a->kv, 16) &&
                     aligned(a->out, 8) && a->ldo % 4 == 0 && a->ldo >= (int64_t)a->H * a->vdim,
                 "md_latent_prefill: null or misaligned argument");
    LatentParams p = make_params(a);
    p.n_groups = (a->n_max + kLatentPrefillRows - 1) / kLatentPrefillRows;
    const int64_t grid = ((int64_t)a->B * a->H + 7) / 8 * 8 * p.n_groups;
    MD_CHECK_ARG(grid < ((int64_t)1 << 31), "md_latent_prefill: grid too large");
    int rc;
    switch (prefill_dk(a->dim + a->rot_dim)) {
    case 64: rc = md_internal_latent_prefill_64(p, (int)grid, (hipStream_t)stream); break;
    case 128: rc = md_internal_latent_prefill_128(p, (int)grid, (hipStream_t)stream); break;
    case 192: rc = md_internal_latent_prefill_192(p, (int)grid, (hipStream_t)stream); break;
    default: rc = md_internal_latent_prefill_256(p, (int)grid, (hipStream_t)stream);
    }
    if (rc != MD_OK) return rc;
    MD_CHECK_LAUNCH("md_latent_prefill");
    return MD_OK;
}
