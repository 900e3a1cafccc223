// Standalone dequantisation: packed int4 -> fp16 W_hat [N,K], natural k order.
// Replaces dequant_W_kernel (reference:
// quantization/tianshu/backend/w4a16_gemm.cuh:1060-1154).  Pure bandwidth:
// reads N*K/2 + (K/g)*N*4 bytes, writes 2*N*K bytes.
#include "sq_common.h"
#include "sq_kernels.h"

namespace sq {

// Layout L1.  One thread = one packed word = 8 outputs = one 16-byte store, so a
// wave reads 256 contiguous bytes and writes 1 KiB contiguous bytes.  A thread has one to a few words, so what stands in front
// of its loads counts: a word's row takes a division, which in 64 bits is some hundred instructions with a branch that the word's
// own load waited behind (4128x2688 at group size 32, 6.8 -> 6.5 us).  I: 32 bits up to 2^31 words, 64 beyond (launch_indexed).
template <typename I>
__global__ __launch_bounds__(256) void dequant_l1_kernel(const uint32_t* __restrict__ w,
                                                         const half2_t* __restrict__ zs,
                                                         half8_t* __restrict__ out, int K8, int gshift8,
                                                         int groups, I total_words, int blocks) {
    const NibbleMasks nm = nibble_masks();
    const I stride = (I)blocks * 256;
    for (I i = (I)blockIdx.x * 256 + threadIdx.x; i < total_words; i += stride) {
        const uint32_t word = __builtin_nontemporal_load(w + i);
        const I n = i / (I)K8;
        const int k8 = (int)(i - n * (I)K8);
        const half2_t p = zs[(long)n * groups + (k8 >> gshift8)];
        const half2_t z64 = {p.x, p.x};
        const half2_t s = {p.y, p.y};
        __builtin_nontemporal_store(dequant8(word, z64, s, nm), out + i);
    }
}

// Closed-form position of element (n,k) inside the layout-L2 weight: the tile
// order is [K/32][N/32][32 lanes][4 words][8 nibbles] with
//   lane = (n%8)*4 + (k%8)/2, word = (k%32/16)*2 + (n%32/16),
//   nibble = (k%2)*4 + ((k/8)%2)*2 + ((n/8)%2).
// (derived from the 10-axis nibble permutation of
// quantization/nvidia/kernel/gemm_s4_f16/format.cu:66-71)
__device__ __forceinline__ uint32_t l2_nibble(const uint32_t* __restrict__ w, int n, int k, int N) {
    const int kk = k & 31, nn = n & 31;
    const int lane = (nn & 7) * 4 + ((kk & 7) >> 1);
    const int word = (kk >> 4) * 2 + (nn >> 4);
    const int nib = (kk & 1) * 4 + ((kk >> 3) & 1) * 2 + ((nn >> 3) & 1);
    const long tile = (long)(k >> 5) * (N >> 5) + (n >> 5);
    return (w[(tile * 32 + lane) * 4 + word] >> (4 * nib)) & 0xFu;
}

// Layout L2.  One thread = 8 consecutive k of one row; a one-time conversion, so
// the gather through the closed form is not tuned.
template <typename I>
__global__ __launch_bounds__(256) void dequant_l2_kernel(const uint32_t* __restrict__ w,
                                                         const half2_t* __restrict__ zs,
                                                         half8_t* __restrict__ out, int N, int K, int g,
                                                         int blocks) {
    const I K8 = (I)(K / 8);
    const I total = (I)N * K8;
    const I stride = (I)blocks * 256;
    for (I i = (I)blockIdx.x * 256 + threadIdx.x; i < total; i += stride) {
        const int n = (int)(i / K8);
        const int k0 = (int)(i - (I)n * K8) * 8;
        const half2_t p = zs[(long)(k0 / g) * N + n];
        half8_t r;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const half_t h = (half_t)(float)(64u + l2_nibble(w, n, k0 + j, N));
            r[j] = (h - p.x) * p.y;
        }
        out[i] = r;
    }
}

static int log2i(int v) {
    int s = 0;
    while ((1 << s) < v) s++;
    return s;
}

// The width of the index that `total` words need; a trip past the end must not wrap, hence 31 bits.
template <typename F>
static hipError_t launch_indexed(long total, F&& launch) {
    long blocks = (total + 255) / 256;
    if (blocks > 256 * 32) blocks = 256 * 32;
    if (total < (1l << 31))
        launch((int)blocks, (uint32_t)total);
    else
        launch((int)blocks, total);
    return hipGetLastError();
}

hipError_t launch_dequant_l1(const void* w, const void* zs, void* out, int N, int K, int g, hipStream_t st) {
    return launch_indexed((long)N * (K / 8), [&](int blocks, auto total) {
        hipLaunchKernelGGL((dequant_l1_kernel<decltype(total)>), dim3(blocks), dim3(256), 0, st, (const uint32_t*)w,
                           (const half2_t*)zs, (half8_t*)out, K / 8, log2i(g) - 3, K / g, total, blocks);
    });
}

hipError_t launch_dequant_l2(const void* w, const void* zs, void* out, int N, int K, int g, hipStream_t st) {
    return launch_indexed((long)N * (K / 8), [&](int blocks, auto total) {
        hipLaunchKernelGGL((dequant_l2_kernel<decltype(total)>), dim3(blocks), dim3(256), 0, st, (const uint32_t*)w,
                           (const half2_t*)zs, (half8_t*)out, N, K, g, blocks);
    });
}

}  // namespace sq
