// Expanded latent attention on the matrix cores (bf16, gfx950): prompts.  Keys are the context's expanded rows (dim numbers per
// head, dense) followed by the rotated part every head shares (straight from the cache pages); values are expanded rows.
// Compiled once per padded key width: -DMD_LATENT_DK=64 | 128 | 192 | 256; the value width is a template parameter.
//
// Eight wavefronts of 32 query rows share 64-key tiles through LDS images, one barrier per tile.  S^T = K Q^T and
// O^T = V^T P^T on 32x32x16: a lane owns one query row, so the running maximum is a lane-local reduction plus one exchange.  It is
// followed lazily: sums are rescaled only when a tile's maximum exceeds the reference by 8 (weights up to 2^8 are harmless in
// fp32).  Queries are rotated as they are loaded; the output is multiplied by the head's gate.  Weights enter the product as a
// bf16 part and a bf16 rest.
//
// What bounds it: a workgroup fills its CU, so that nothing else runs while it waits -- for its queries and behind its output rows, for
// tiles, and at the end of the launch for the CU that started last.  4 x 2049 rows, 32 heads of 128 + 64 / 128 (the matrix work is 110 us
// of a SIMD): 400 us with tiles through registers, query and output rows in 8- and 16-byte pieces (30 us each) and pair after pair;
// 352 with the DMA, whole rows and no wait for the page number between a tile's loads; 332 with the longest groups of every pair first;
// 306 with a prompt's odd rows at its start.  One row of 8192: 938 -> 860; 128 rows behind 4000: 163 -> 154.
#include "attn_common.h"
#include "latent.h"

#include <algorithm>

#ifndef MD_LATENT_DK
#error "compile with -DMD_LATENT_DK=<padded key size>"
#endif

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int DK = MD_LATENT_DK, KT = 64, NW = kLatentPrefillRows / 32, NT = 64 * NW;

// Places in the image (lds_place for keys): values are read transposed, two pieces of four rows at a time, and pairs stay together.
template <int N>
__device__ __forceinline__ int value_place(int ch, int row) { return ch ^ (2 * (row & (N % 16 ? 3 : 7))); }
__device__ const u32x4 kZeros = {0u, 0u, 0u, 0u};

// 16 bytes a lane from `src` to LDS bytes `to` + lane * 16
__device__ __forceinline__ void dma16(const bf16_t* src, unsigned int to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(to), "v"(src) : "memory", "m0");
}

// weights -> upper 16 bits (truncated: bf16) and the rest rounded to bf16
__device__ __forceinline__ void split(const f32x8 w, bf16x8& hi, bf16x8& lo) {
    u32x4 h;
    f32x8 r;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const unsigned int a = __float_as_uint(w[e]), b = __float_as_uint(w[e + 1]);
        h[e / 2] = __builtin_amdgcn_perm(b, a, 0x07060302);
        r[e] = w[e] - __uint_as_float(a & 0xffff0000u);
        r[e + 1] = w[e + 1] - __uint_as_float(b & 0xffff0000u);
    }
    hi = *reinterpret_cast<const bf16x8*>(&h);
    lo = __builtin_convertvector(r, bf16x8);
}

template <int DV>
constexpr int stage_bytes() { return KT * (DK + DV) * 2; }
// images: the tile in use and those on their way, two where they fit
template <int DV>
constexpr int images() { return 3 * stage_bytes<DV>() <= 160 * 1024 ? 3 : 2; }
constexpr int kQueryBytes = kLatentPrefillRows * DK * 2;
// the queries arrive beside the first tile where the CU has room for both, in front of it otherwise
template <int DV>
constexpr int query_at() { return stage_bytes<DV>() + kQueryBytes <= 160 * 1024 ? stage_bytes<DV>() : 0; }

template <int DV>
__global__ __launch_bounds__(NT, 2) void latent_prefill_kernel(const LatentParams p) {
    constexpr int KS = DK / 16, NB = DV / 16, DB = DV / 32;
    constexpr int K_BYTES = KT * DK * 2, STAGE = stage_bytes<DV>(), CK = DK / 8, CV = DV / 8, NK = KT * CK / NT, NV = KT * CV / NT, NI = images<DV>();
    static_assert(KT * CK % NT == 0 && KT * CV % NT == 0, "a tile is a whole number of pieces per thread");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // NI tile images; first the queries, last the output rows
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // blocks of one (request, head) differ by multiples of 8: same XCD.  The long ones (late rows) first, since the last one to start is the
    // last to end: of every pair where a prompt's rows are most of its context (pair after pair: 352 us for 332), one pair after the other
    // behind a long one, where its groups are about as long and read its rows together (2 x 655 behind 4000, 128 heads of 128 + 64 / 128
    // 714 us, 753 of every pair).  The first request decides: it is a matter of speed only
    const int r0 = blockIdx.x >> 3, pairs = (p.B * p.H + 7) / 8;
    const bool all = p.qo_indptr[1] - p.qo_indptr[0] > p.pos0[0];
    const int qg = p.n_groups - 1 - (all ? r0 / pairs : r0 % p.n_groups), pair = (all ? r0 % pairs : r0 / p.n_groups) * 8 + (blockIdx.x & 7);
    if (pair >= p.B * p.H) return;
    const int b = pair / p.H, h = pair % p.H;
    const int q0 = p.qo_indptr[b], n_b = p.qo_indptr[b + 1] - q0;
    if (qg * kLatentPrefillRows >= n_b) return;                   // whole workgroup
    // In more than a round of the chip groups end with the last row: rows that fill none are the first ones, with the shortest contexts (16 x
    // 868 rows, 8 heads of 256 / 256 202 us, 234 otherwise).  One round waits for the group with the longest context, and the last one may
    // have few rows: groups begin with the first row (872 rows behind 100, 8 heads of 96 / 64 40 us, 44 otherwise)
    const int g0 = qg * kLatentPrefillRows - (gridDim.x > 256 ? kLatentPrefillRows - 1 - (n_b - 1) % kLatentPrefillRows : 0);
    const int pos_b = p.pos0[b], pg0 = p.page_indptr[b], cap = (p.page_indptr[b + 1] - pg0) * p.page_size;
    const int c0 = p.ctx_indptr[b], ctx = min(p.ctx_indptr[b + 1] - c0, cap);
    const int wg_last = min(pos_b + min(g0 + kLatentPrefillRows, n_b) - 1, ctx - 1);
    if (wg_last < 0) return;
    const int w0 = g0 + wave * 32, qi = w0 + j;                     // the wave's first row, this lane's row
    const bool valid = qi >= 0 && qi < n_b;
    const int pos = pos_b + qi, lim = valid ? min(pos, ctx - 1) : 0;
    const int lim_lo = min(pos_b + max(w0, 0), ctx - 1), my_last = w0 > -32 && w0 < n_b ? min(pos_b + min(w0 + 32, n_b) - 1, ctx - 1) : -1;
    const int t1 = wg_last / KT, my1 = my_last >= 0 ? my_last / KT : -1;
    const int dq = p.dim + p.rot_dim;
    const float sl2 = fabsf(p.scale_log2);

    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] = 0.f;
    float m = -INFINITY, l = 0.f;

    // ---- tiles to LDS, without a register between: the DMA writes lane after lane, so that a lane fetches the piece that belongs at its
    // place.  In assembly, since the compiler would have every LDS read wait for it; the waits are counted by hand.  All of a wave's
    // lanes take part in every load: pieces behind a key are zeros (they meet the query's zeros), pieces behind a value any
    const int ldkv = p.H * (p.dim + p.vdim), hk = h * p.dim, hv = p.H * p.dim + h * p.vdim;
    const int pg1 = wg_last / p.page_size;
    int pages = p.page_indices[pg0 + min(lane, pg1)];               // of 64 pages, one a lane
    asm volatile("" : "+v"(pages));
    auto issue = [&](int t, int img) {
        const int kp0 = t * KT, rem = ctx - 1 - kp0, pi = kp0 / p.page_size;    // rows past the context repeat its last row: they are masked
        if (pi % 64 == 0 && pi > 0 && kp0 % p.page_size == 0) {
            pages = p.page_indices[pg0 + min(pi + lane, pg1)];
            asm volatile("" : "+v"(pages));                         // waited for here: behind the branch it would be in every tile
        }
        const int page = __builtin_amdgcn_readlane(pages, pi % 64);
        const bf16_t* kvb = reinterpret_cast<const bf16_t*>(p.kv) + (int64_t)(c0 + kp0) * ldkv;
        const bf16_t* rpb = reinterpret_cast<const bf16_t*>(p.cache) + p.kv_rank +
                            ((int64_t)page * p.page_size + kp0 % p.page_size) * p.W;
        const unsigned int to = (unsigned int)(img * STAGE + wave * 1024);
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int c = i * NT + tid, r = c / CK, row = min(r, rem), d = lds_place<CK>(c % CK, r) * 8;
            const bf16_t* src = d < p.dim ? kvb + (row * ldkv + hk + d) : rpb + (row * p.W + d - p.dim);
            if (dq < DK) src = d < dq ? src : reinterpret_cast<const bf16_t*>(&kZeros);
            dma16(src, to + i * NT * 16);
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = i * NT + tid, r = c / CV, row = min(r, rem), d = value_place<CV>(c % CV, r) * 8;
            dma16(kvb + (row * ldkv + hv + (d < p.vdim ? d : 0)), to + K_BYTES + i * NT * 16);
        }
    };
    // ---- queries: each wave its own 32 rows, dense rows of a head at a time (a lane's own row piece by piece is 64 places a load)
    const int kra0 = j * DK * 2 + lds_place<CK>(kh, j) * 16;
    auto key_at = [&](int ks) {                                     // step ks of the lane's row of 32, key or query
        constexpr int low = CK % 16 ? 127 : 255;
        return (kra0 ^ (ks * 32 & low)) + (ks * 32 & ~low);
    };
    if (query_at<DV>() != 0) issue(0, 0);
#pragma unroll
    for (int i = 0; i < CK / 2; ++i) {
        const int c = i * 64 + lane, r = c / CK, d = lds_place<CK>(c % CK, r) * 8;
        const bf16_t* src = reinterpret_cast<const bf16_t*>(p.q) + ((int64_t)(q0 + min(max(w0 + r, 0), n_b - 1)) * p.H + h) * dq + d;
        dma16(d < dq ? src : reinterpret_cast<const bf16_t*>(&kZeros), query_at<DV>() + wave * 32 * DK * 2 + i * 1024);
    }
    bf16x8 qf[KS];
    {
        const float* cs = p.cos_sin + (int64_t)min(max(pos, 0), p.max_pos - 1) * p.rot_pairs * 2;
        const float sign = p.scale_log2 < 0.f ? -1.f : 1.f;
        f32x4 ca[KS], cb[KS];                                       // (cos, sin) of the four pairs of an 8-element piece
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int e = ks * 16 + kh * 8 - p.dim;
            ca[ks] = cb[ks] = f32x4{1.f, 0.f, 1.f, 0.f};
            if (p.rot_pairs % 4 == 0) {                             // uniform: pieces are rotated as a whole or not at all
                if (e >= 0 && e < 2 * p.rot_pairs) {
                    ca[ks] = *reinterpret_cast<const f32x4*>(cs + e);
                    cb[ks] = *reinterpret_cast<const f32x4*>(cs + e + 4);
                }
            } else if (e >= 0) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (e + u < 2 * p.rot_pairs) ca[ks][u] = cs[e + u];
                    if (e + 4 + u < 2 * p.rot_pairs) cb[ks][u] = cs[e + 4 + u];
                }
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            f32x8 v = __builtin_convertvector(lds_read_b128(smem + query_at<DV>() + wave * 32 * DK * 2 + key_at(ks)), f32x8);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float c = u < 2 ? ca[ks][u * 2] : cb[ks][u * 2 - 4], s = u < 2 ? ca[ks][u * 2 + 1] : cb[ks][u * 2 - 3];
                const float x = v[u * 2], y = v[u * 2 + 1];
                v[u * 2] = (x * c - y * s) * sign;
                v[u * 2 + 1] = (y * c + x * s) * sign;
            }
            qf[ks] = __builtin_convertvector(v, bf16x8);
        }
    }
    __syncthreads();                                                // every wave has its queries
    if (query_at<DV>() == 0) issue(0, 0);
    if (NI == 3 && t1 > 0) issue(1, 1);
    const int lq = lane & 15, vrow = kh * 4 + (lq >> 2);
    int vra[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
        vra[db] = K_BYTES + vrow * DV * 2 + value_place<CV>(((lane >> 4) & 1) * NB + db * 2 + ((lq & 3) >> 1), vrow) * 16 + (lq & 1) * 8;
    // this row's largest score of tile t, keys past the row's position left out
    auto largest = [&](int t, f32x16& s0, f32x16& s1) {
        if (t * KT + KT - 1 > lim_lo) {                             // wave-uniform: the tile reaches past some row's position
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = t * KT + 4 * kh + (r & 3) + 8 * (r >> 2);
                if (key > lim) s0[r] = -INFINITY;
                if (key + 32 > lim) s1[r] = -INFINITY;
            }
        }
        float mx = s0[0];
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(fmaxf(mx, s0[r]), s1[r]);
        return fmaxf(mx, __shfl_xor(mx, 32)) * sl2;
    };
    auto rescale = [&](float mx) {
        if (__any(mx > m + 8.f)) {                                  // (the first tile holds key 0, which every row sees: m is finite)
            const float mn = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - mn);
            l *= alpha;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
            m = mn;
        }
    };
    auto weights = [&](const f32x16& s, int s16, bf16x8& ph, bf16x8& pl) {       // of keys s16 * 16 .. + 15
        f32x8 pv;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            pv[e] = __builtin_amdgcn_exp2f(fmaf(s[s16 * 8 + e], sl2, -m));
            l += pv[e];
        }
        split(pv, ph, pl);
    };
    auto add = [&](const unsigned char* img, int u, int s16, const bf16x8 ph, const bf16x8 pl) {
        bf16x8 vf[DB];
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            const unsigned char* vb = img + vra[db] + (u * 32 + s16 * 16) * DV * 2;
            const bf16x4 v0 = lds_read_tr(vb), v1 = lds_read_tr(vb + 8 * DV * 2);
            vf[db] = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
            o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[db], ph, o[db], 0, 0, 0);
        }
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[db], pl, o[db], 0, 0, 0);
    };
    // tile t lies in image t % NI; it is overwritten NI tiles later, after a barrier every wave reaches past its use
    for (int t = 0, cur = 0; t <= t1; ++t, cur = cur == NI - 1 ? 0 : cur + 1) {
        if (NI == 3 && t < t1) asm volatile("s_waitcnt vmcnt(%0)" : : "i"(NK + NV) : "memory");       // tile t + 1 may be on its way
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (t + NI - 1 <= t1) issue(t + NI - 1, cur == 0 ? NI - 1 : cur - 1);
        if (t > my1) continue;
        const unsigned char* img = smem + cur * STAGE;
        f32x16 s0 = {}, s1 = {};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const unsigned char* k = img + key_at(ks);
            s0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lds_read_b128(k), qf[ks], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lds_read_b128(k + 32 * DK * 2), qf[ks], s1, 0, 0, 0);
        }
        rescale(largest(t, s0, s1));
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            bf16x8 ph, pl;
            weights(g < 2 ? s0 : s1, g & 1, ph, pl);
            add(img, g >> 1, g & 1, ph, pl);
        }
    }

    l += __shfl_xor(l, 32);
    float inv = 1.0f / l;
    if (p.gate && valid) inv /= 1.0f + expf(-(float)reinterpret_cast<const bf16_t*>(p.gate)[(q0 + qi) * p.ld_gate + h]);
    // ---- output rows: through LDS, so that a store writes whole rows of a head
    __syncthreads();                                                // every wave is past the last image
    // With wide heads nothing below is computed, and kept, in front of the tiles: 192 / 192 has no register for it (40 spilled; 4 x 821 rows
    // behind 100, 16 heads of 128 + 64 / 192 75 -> 62 us)
    int ln = lane;
    if constexpr (DK + DV >= 320) asm volatile("" : "+v"(ln));
    const int oj = ln & 31;
    unsigned char* mine = smem + wave * 32 * DV * 2;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
            const int ch = (db + (rg >> 1) * (NB / 2)) * 2 + (rg & 1);
            const f32x4 ov = {o[db][rg * 4] * inv, o[db][rg * 4 + 1] * inv, o[db][rg * 4 + 2] * inv, o[db][rg * 4 + 3] * inv};
            *reinterpret_cast<bf16x4*>(mine + oj * DV * 2 + lds_place<CV>(ch, oj) * 16 + (ln >> 5) * 8) = __builtin_convertvector(ov, bf16x4);
        }
#pragma unroll
    for (int i = 0; i < CV / 2; ++i) {
        const int c = i * 64 + ln, r = c / CV, ch = c % CV;
        const bf16x8 v = lds_read_b128(mine + r * DV * 2 + lds_place<CV>(ch, r) * 16);
        if (w0 + r >= 0 && w0 + r < n_b && ch * 8 < p.vdim)
            *reinterpret_cast<bf16x8_a8*>(reinterpret_cast<bf16_t*>(p.out) + (q0 + w0 + r) * p.ldo + h * p.vdim + ch * 8) = v;
    }
}

template <int DV>
int launch(const LatentParams& p, int grid, hipStream_t st) {
    constexpr int tiles = images<DV>() * stage_bytes<DV>(), queries = query_at<DV>() + kQueryBytes, rows = kLatentPrefillRows * DV * 2;
    constexpr int lds = std::max(tiles, std::max(queries, rows));
    static_assert(lds <= 160 * 1024, "the tile images must fit the CU");
    auto k = latent_prefill_kernel<DV>;
    static MdPerDeviceOnce once;
    if (lds > 64 * 1024 && once.first() &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) {
        once.undo();
        md_set_error("md_latent_prefill: hipFuncSetAttribute(%d B LDS) failed", lds);
        return MD_ERR_LAUNCH;
    }
    hipLaunchKernelGGL(k, dim3(grid), dim3(NT), lds, st, p);
    return MD_OK;
}

}  // namespace

#define MD_CAT_(a, b) a##b
#define MD_CAT(a, b) MD_CAT_(a, b)

int MD_CAT(md_internal_latent_prefill_, MD_LATENT_DK)(const LatentParams& p, int grid, hipStream_t st) {
    return p.vdim <= 64 ? launch<64>(p, grid, st) : p.vdim <= 128 ? launch<128>(p, grid, st)
         : p.vdim <= 192 ? launch<192>(p, grid, st) : launch<256>(p, grid, st);
}
