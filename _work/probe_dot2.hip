#include <hip/hip_runtime.h>
#include <stdio.h>
#include <string.h>
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
__global__ void k(const unsigned* w, float* a, float* b, int n) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    unsigned x = w[i];
    a[i] = __uint_as_float(x << 16) + __uint_as_float(x & 0xffff0000u);
    bf2 v = __builtin_bit_cast(bf2, x), one = {(__bf16)1.0f, (__bf16)1.0f};
    b[i] = __builtin_amdgcn_fdot2_f32_bf16(v, one, 0.0f, false);
}
__global__ void nanmul(const float* t, const float* c, unsigned* o, int n) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) o[i] = __float_as_uint(t[i] * c[i]);
}
int main() {
    const int n = 1 << 20;
    unsigned* w; float *a, *b;
    hipHostMalloc(&w, n * 4); hipHostMalloc(&a, n * 4); hipHostMalloc(&b, n * 4);
    unsigned s = 12345;
    for (int i = 0; i < n; i++) {
        unsigned lo, hi;
        s = s * 1664525u + 1013904223u; lo = (s >> 8) & 0x7fff; s = s * 1664525u + 1013904223u; hi = (s >> 8) & 0x7fff;
        int kind = i & 3;
        if (kind == 0) { lo &= 0x3fff; hi = (hi & 0x7f) | (lo & 0x7f80); }              // near exponents
        if (kind == 1) { lo &= 0x1ff; hi &= 0x1ff; }                                   // denormal and smallest normal
        if (kind == 2) { lo &= 0x3f80; lo |= 0x55; hi = lo > 0x400 ? lo - 0x400 + (hi & 0x7f) : hi & 0x7f; }
        if (lo >= 0x3f81) lo = 0x3f80; if (hi >= 0x3f81) hi = 0x3f80;                   // probabilities: 0..1
        w[i] = lo | hi << 16;
    }
    k<<<n / 256, 256>>>(w, a, b, n);
    hipDeviceSynchronize();
    int bad = 0, badd = 0;
    for (int i = 0; i < n; i++) if (memcmp(&a[i], &b[i], 4)) { bad++; if (a[i] < 1.2e-38f) badd++; if (bad < 6) printf("%08x %g %g\n", w[i], a[i], b[i]); }
    printf("dot2: %d of %d differ, %d of them denormal\n", bad, n, badd);
    float* t = a; unsigned nan = 0x7fc08000u; float f; memcpy(&f, &nan, 4);
    const float cs[8] = {1.0f, 0.0f, 1e-30f, 1e30f, 3.0f, f, 1e-40f, 2.0f};
    for (int i = 0; i < 8; i++) { t[i] = i == 5 ? 2.5f : f; b[i] = cs[i]; }
    nanmul<<<1, 256>>>(t, b, w, 8);
    hipDeviceSynchronize();
    for (int i = 0; i < 8; i++) printf("%08x ", w[i]);
    printf("\n");
    return 0;
}
