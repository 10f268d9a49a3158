// StreamingLLM sink+window eviction for the draft KV cache, gfx950.
//
// reference: KVCache.prefill        Engine/StreamingLLM/model_draft.py:102-143
//            KVCache.prefill_draft  Engine/StreamingLLM/model.py:116-157
//
// The reference, per 128-token prefill chunk and per layer, builds
//   new_k = cat(cache[:, sink:kv_len], k_chunk)[:, -(kv_len-sink):]
// re-appends it, clones the WHOLE draft cache, rotates the clone's keys with
// cache-relative positions and runs attention on the clone.  Here:
//   md_streaming_shift_append : the same resulting bytes, in place (slots in
//       ascending groups, a group read before any of it is overwritten);
//   md_streaming_rotate       : rows [0,valid_len) of every request, K rotated
//       by position = slot index, V copied, into a scratch cache (or in place
//       on the last chunk == the reference's kv_cache.copy_(rotated_kv));
//   md_streaming_windows      : both for several chunks at once, where they are
//       too small to be passed one by one (few requests).
// Bug-for-bug: the shift covers the whole [sink,kv_len) slot range even while
// the tail slot has never been written (the zero row of the 2nd->3rd chunk
// transition travels exactly as in the reference).
#include "md_common.h"

namespace {

__device__ __forceinline__ int64_t slot_offset(int b, int s, int ppr, int page_size, int row_elems) {
    const int page = b * ppr + s / page_size;
    const int slot = s % page_size;
    return ((int64_t)page * 2 * page_size + slot) * row_elems;
}

// A workgroup moves COLS adjacent 16-B columns (8: one 128-B line per row) of a request's k or v rows: 256 / COLS rows at a time, 8 such
// strips in registers, requested at once, then -- when every wavefront has them -- written n_new rows further up.  Rows move towards
// lower slots only, so a strip group never overwrites a row that a later one reads.  Bound by the latency of one round trip
// per strip group while the rows fit the last-level cache: 8 columns, 256 rows a trip.  One thread per column walking the rows in eights
// (one workgroup per request at 8 kv heads of 64) took 46.8 us for 16 requests of 257 rows, 15.8 MB moved; this takes 6.7.  Beyond it
// bound by HBM, 2 x 2 x budget rows, which single lines reach less well than 512-B runs: 32 columns.
constexpr int kShiftStrips = 8;

template <int COLS>
__global__ __launch_bounds__(256) void shift_append_kernel(const bf16_t* __restrict__ k_new,
                                                           const bf16_t* __restrict__ v_new, int64_t ks, int64_t vs,
                                                           bf16_t* cache, int n_new, int kv_len, int sink, int ppr,
                                                           int KH, int D, int page_size) {
    constexpr int ROWS = 256 / COLS;
    const int b = blockIdx.y;
    const int row_elems = KH * D;
    const int cols = row_elems / 8;
    const int t = blockIdx.x * COLS + threadIdx.x % COLS, strip = threadIdx.x / COLS;
    const bool live = t < 2 * cols, isv = t >= cols;
    const int c = isv ? t - cols : t;
    const int64_t half = isv ? (int64_t)page_size * row_elems : 0;
    const bf16_t* nw = isv ? v_new : k_new;
    const int64_t ns = isv ? vs : ks;
    for (int s0 = sink; s0 < kv_len; s0 += ROWS * kShiftStrips) {
        u32x4 buf[kShiftStrips];
#pragma unroll
        for (int u = 0; u < kShiftStrips; ++u) {
            const int s = s0 + u * ROWS + strip;
            if (live && s < kv_len) {
                const int src = s + n_new;
                if (src < kv_len)
                    buf[u] = *reinterpret_cast<const u32x4*>(cache + slot_offset(b, src, ppr, page_size, row_elems) + half + c * 8);
                else
                    buf[u] = *reinterpret_cast<const u32x4*>(nw + (int64_t)(b * n_new + (src - kv_len)) * ns + c * 8);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the rows are in registers before any of them is overwritten
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kShiftStrips; ++u) {
            const int s = s0 + u * ROWS + strip;
            if (live && s < kv_len)
                *reinterpret_cast<u32x4*>(cache + slot_offset(b, s, ppr, page_size, row_elems) + half + c * 8) = buf[u];
        }
    }
}

// eight rotated elements (same arithmetic as kvops.hip rope8); c: their cos / sin pairs
__device__ __forceinline__ u32x4 rotate8(const u32x4 x, const float* __restrict__ c) {
    const f32x4 c0 = *reinterpret_cast<const f32x4*>(c);
    const f32x4 c1 = *reinterpret_cast<const f32x4*>(c + 4);
    u32x4 r;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const float xe = __uint_as_float(x[w] << 16);
        const float xo = __uint_as_float(x[w] & 0xffff0000u);
        const float co = w < 2 ? c0[(w & 1) * 2] : c1[(w & 1) * 2];
        const float si = w < 2 ? c0[(w & 1) * 2 + 1] : c1[(w & 1) * 2 + 1];
        const float ye = __fsub_rn(__fmul_rn(xe, co), __fmul_rn(xo, si));
        const float yo = __fadd_rn(__fmul_rn(xo, co), __fmul_rn(xe, si));
        const bf16x2 pk = {f32_to_bf16(ye), f32_to_bf16(yo)};
        r[w] = *reinterpret_cast<const unsigned int*>(&pk);
    }
    return r;
}

// grid (valid_len, B); K rotated by pos = slot, V copied
__global__ __launch_bounds__(256) void rotate_kernel(const bf16_t* __restrict__ cache, bf16_t* rot, int ppr, int KH, int D,
                                                     int page_size, const float* __restrict__ cos_sin, int max_pos) {
    const int b = blockIdx.y, s = blockIdx.x;
    const int row_elems = KH * D;
    const int cols = row_elems / 8;
    const int cpr = D / 8;
    const int64_t off = slot_offset(b, s, ppr, page_size, row_elems);
    const int64_t half = (int64_t)page_size * row_elems;
    const int pos = s < max_pos ? s : max_pos - 1;
    const float* cs = cos_sin + (int64_t)pos * D;
    const bool inplace = (rot == cache);
    for (int i = threadIdx.x; i < 2 * cols; i += blockDim.x) {
        if (i < cols) {
            const u32x4 x = *reinterpret_cast<const u32x4*>(cache + off + i * 8);
            const u32x4 r = rotate8(x, cs + (i % cpr) * 8);
            *reinterpret_cast<u32x4*>(rot + off + i * 8) = r;
        } else if (!inplace) {
            const int ii = i - cols;
            *reinterpret_cast<u32x4*>(rot + off + half + ii * 8) =
                *reinterpret_cast<const u32x4*>(cache + off + half + ii * 8);
        }
    }
}

// The caches that C portions of a prompt see, all at once.  What a slot holds after portion c follows from the cache before the first of
// them and from their new rows alone, so no portion waits for the one ahead of it:
//   while a portion fits, slot s < ctx is the old row and slot ctx + j new row j;
//   from portion f on, the first that does not, every slot >= sink moves up by the m tokens since then: slot s is slot s + m of
//   that moment, or new row s + m - kv_len of those m (the moment's slots past its tokens are what the cache holds there).
// blockIdx.y = c < C writes portion c's rows, keys rotated by their slot, as pages of their own; c = C writes the cache as the last
// portion leaves it (all slots) to `next`: the cache itself is still being read.  Bound by the traffic, 2 x 2 x (C + 1) x kv_len rows a
// request.
constexpr int kWindowRows = 4;

struct WindowParams {
    const bf16_t *k, *v, *cache;
    bf16_t *windows, *next;
    const float* cos_sin;
    int64_t ks, vs;
    int tokens, portion, portions, ctx, kv_len, sink, ppr, KH, D, page_size, max_pos, rotate_next;
};

__global__ __launch_bounds__(256) void windows_kernel(const WindowParams p) {
    const int b = blockIdx.z, c = min((int)blockIdx.y, p.portions - 1);
    const bool last = (int)blockIdx.y == p.portions;
    const int begin = c * p.portion, n = min(p.portion, p.tokens - begin);
    const int before = min(p.ctx + begin, p.kv_len);
    const int pre = (p.kv_len - p.ctx) / p.portion * p.portion;      // tokens ahead of portion f
    const bool over = before + n > p.kv_len;
    const int valid = over ? p.kv_len : before + n, m = over ? begin + n - pre : 0;
    const int slots = last ? p.ppr * p.page_size : valid;
    const int row = p.KH * p.D, cols = row / 8, cpr = p.D / 8;
    for (int i = threadIdx.x; i < kWindowRows * 2 * cols; i += 256) {
        const int s = blockIdx.x * kWindowRows + i / (2 * cols), t = i % (2 * cols);
        if (s >= slots) break;
        const bool isv = t >= cols;
        const int col = isv ? t - cols : t;
        const int at = over && s >= p.sink && s < valid ? s + m : s;
        int token = -1;
        if (at >= p.kv_len && s < valid)
            token = pre + at - p.kv_len;
        else if (s < valid && at >= p.ctx && at < (over ? p.ctx + pre : valid))
            token = at - p.ctx;
        const int64_t half = isv ? (int64_t)p.page_size * row : 0;
        const bf16_t* src = token >= 0 ? (isv ? p.v : p.k) + ((int64_t)b * p.tokens + token) * (isv ? p.vs : p.ks)
                                       : p.cache + slot_offset(b, at, p.ppr, p.page_size, row) + half;
        u32x4 x = *reinterpret_cast<const u32x4*>(src + col * 8);
        if (!isv && s < valid && (!last || p.rotate_next))
            x = rotate8(x, p.cos_sin + (int64_t)min(s, p.max_pos - 1) * p.D + col % cpr * 8);
        bf16_t* dst = last ? p.next + slot_offset(b, s, p.ppr, p.page_size, row)
                           : p.windows + slot_offset(b * p.portions + c, s, p.ppr, p.page_size, row);
        *reinterpret_cast<u32x4*>(dst + half + col * 8) = x;
    }
}

}  // namespace

extern "C" int md_streaming_windows(const void* k_new, const void* v_new, int64_t k_row_stride, int64_t v_row_stride, const void* cache,
                                    void* windows, void* next, int B, int tokens, int portion, int ctx, int kv_len, int sink,
                                    int pages_per_req, int KH, int D, int page_size, int rotate_next, const float* cos_sin, int max_pos,
                                    md_stream_t stream) {
    MD_CHECK_ARG(k_new && v_new && cache && windows && next && cos_sin, "md_streaming_windows: null pointer argument");
    MD_CHECK_ARG(next != cache && windows != cache && windows != next, "md_streaming_windows: the cache is read while the others are written");
    MD_CHECK_ARG(B > 0 && B <= 65535 && tokens > 0 && portion > 0 && ctx >= 0 && ctx <= kv_len && kv_len > sink && sink >= 0 && KH > 0 &&
                     D > 0 && D % 8 == 0 && page_size > 0 && (int64_t)pages_per_req * page_size >= kv_len && max_pos > 0,
                 "md_streaming_windows: bad shape tokens=%d portion=%d ctx=%d kv_len=%d sink=%d pages_per_req=%d", tokens, portion, ctx,
                 kv_len, sink, pages_per_req);
    MD_CHECK_ARG((((uintptr_t)k_new | (uintptr_t)v_new | (uintptr_t)cache | (uintptr_t)windows | (uintptr_t)next | (uintptr_t)cos_sin) & 15) == 0 &&
                     k_row_stride % 8 == 0 && v_row_stride % 8 == 0,
                 "md_streaming_windows: 16-byte alignment / stride multiple of 8 required");
    const int portions = (int)(((int64_t)tokens + portion - 1) / portion);
    MD_CHECK_ARG(portions < 65535, "md_streaming_windows: %d portions", portions);
    const WindowParams p = {(const bf16_t*)k_new, (const bf16_t*)v_new, (const bf16_t*)cache, (bf16_t*)windows, (bf16_t*)next, cos_sin,
                            k_row_stride, v_row_stride, tokens, portion, portions, ctx, kv_len, sink, pages_per_req, KH, D, page_size,
                            max_pos, rotate_next};
    const int slots = pages_per_req * page_size;
    hipLaunchKernelGGL(windows_kernel, dim3((slots + kWindowRows - 1) / kWindowRows, portions + 1, B), dim3(256), 0, (hipStream_t)stream, p);
    MD_CHECK_LAUNCH("md_streaming_windows");
    return MD_OK;
}

extern "C" int md_streaming_shift_append(const void* k_new, const void* v_new, int64_t k_row_stride,
                                         int64_t v_row_stride, void* cache, int B, int n_new, int kv_len, int sink,
                                         int pages_per_req, int KH, int D, int page_size, md_stream_t stream) {
    MD_CHECK_ARG(k_new && v_new && cache, "md_streaming_shift_append: null pointer argument");
    MD_CHECK_ARG(B > 0 && n_new > 0 && kv_len > sink && sink >= 0 && KH > 0 && D > 0 && (KH * D) % 8 == 0 &&
                     page_size > 0 && pages_per_req * page_size >= kv_len,
                 "md_streaming_shift_append: bad shape n_new=%d kv_len=%d sink=%d pages_per_req=%d", n_new, kv_len,
                 sink, pages_per_req);
    MD_CHECK_ARG((((uintptr_t)k_new | (uintptr_t)v_new | (uintptr_t)cache) & 15) == 0 && k_row_stride % 8 == 0 &&
                     v_row_stride % 8 == 0,
                 "md_streaming_shift_append: 16-byte alignment / stride multiple of 8 required");
    const int cols2 = 2 * KH * D / 8;
    // 512-B runs from two workgroups of them per CU and rows beyond the 256 MB of the last-level cache on: 64 requests of 1 025 rows, 32
    // kv heads of 128, 482 us in 128-B lines, 411 (one thread per column: 409); 128 of 257, 32 of 128, 230, 203 (207).  Below, the long
    // trips win: 128 requests of 257 rows, 8 kv heads of 64, 22 us, 26 in 512-B runs.
    const int64_t wide = (int64_t)((cols2 + 31) / 32) * B;
    const bool runs = wide >= 600 && wide * 512 * kv_len >= 266000000;
    const int cols = runs ? 32 : 8;
    hipLaunchKernelGGL(runs ? shift_append_kernel<32> : shift_append_kernel<8>, dim3((cols2 + cols - 1) / cols, B), dim3(256), 0,
                       (hipStream_t)stream, (const bf16_t*)k_new, (const bf16_t*)v_new, k_row_stride, v_row_stride, (bf16_t*)cache, n_new,
                       kv_len, sink, pages_per_req, KH, D, page_size);
    MD_CHECK_LAUNCH("md_streaming_shift_append");
    return MD_OK;
}

extern "C" int md_streaming_rotate(const void* cache, void* rot_cache, int B, int valid_len, int pages_per_req, int KH,
                                   int D, int page_size, const float* cos_sin, int max_pos, md_stream_t stream) {
    MD_CHECK_ARG(cache && rot_cache && cos_sin, "md_streaming_rotate: null pointer argument");
    MD_CHECK_ARG(B > 0 && valid_len > 0 && KH > 0 && D > 0 && D % 8 == 0 && page_size > 0 &&
                     pages_per_req * page_size >= valid_len && max_pos > 0,
                 "md_streaming_rotate: bad shape valid_len=%d pages_per_req=%d", valid_len, pages_per_req);
    MD_CHECK_ARG((((uintptr_t)cache | (uintptr_t)rot_cache | (uintptr_t)cos_sin) & 15) == 0,
                 "md_streaming_rotate: 16-byte alignment required");
    hipLaunchKernelGGL(rotate_kernel, dim3(valid_len, B), dim3(256), 0, (hipStream_t)stream, (const bf16_t*)cache,
                       (bf16_t*)rot_cache, pages_per_req, KH, D, page_size, cos_sin, max_pos);
    MD_CHECK_LAUNCH("md_streaming_rotate");
    return MD_OK;
}
