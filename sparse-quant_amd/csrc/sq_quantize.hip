// Quantise and pack an fp16 weight in one pass (layouts L1 and L2): group minimum / maximum, scale, zero, codes, packed
// words and zeros/scales from one read of the weight.
//
// What bounds it.  2 bytes are read and half a byte is written per weight, so memory is the floor; the arithmetic (a
// correctly rounded quotient per weight, min / max, pack: about eleven vector instructions) comes close to it and is kept
// small: the quotient is a product with the group's reciprocal and one exact remainder step, rounding to an integer is
// one packed addition of 1536 (ulp 1 there, ties to even), clamping and packing work on pairs.
// Measured: 16384 x 4096 at 4 bits and group size 128, 172 MB moved: 41.9 us (4.1 TB/s; a large copy reaches 5.1 TB/s);
// the same result through some twenty element-wise launches took 620 us.
//
// Results are those of the torch expression over fp16 tensors, bit for bit (every operation computed in fp32 and rounded
// to fp16 once, as torch's element-wise kernels do):
//   s = fp16(clamp(fp16(max - min), 1e-5) * (1 / (2^b - 1)))      z = clamp(-round(fp16(min / s)), 0, 2^b - 1)
//   q = clamp(round(fp16(w / s)) + z, 0, 2^b - 1)
// Quotient: with r = fp32(1 / s), q0 = w r, e = w - q0 s (exact in an fma), q1 = q0 + e r lies within 2^-46 of the true
// quotient before its own rounding; a quotient of two 11-bit significands that is not itself a 25-bit number is at least
// 2^-36 away from every such number, so q1 is the correctly rounded fp32 quotient.  Groups that hold an infinity or a
// NaN, or whose range overflows fp16, take a branch of plain operations (one test per wave).
// (replaces quant_funcs.quantize_tensor and the two writers, reference: test/muxi/utils/quant_funcs.py:75-114, and the
// chain of test/nvidia/utils/quant_dequant_nvidia.py:5-32)
#include "sq_common.h"
#include "sq_kernels.h"

namespace sq {

namespace {

__device__ __forceinline__ half2_t pk_max(half2_t a, half2_t b) { return __builtin_elementwise_max(a, b); }
__device__ __forceinline__ half2_t pk_min(half2_t a, half2_t b) { return __builtin_elementwise_min(a, b); }

template <int CTRL>
__device__ __forceinline__ half2_t dpp_max(half2_t v) {
    const int i = bit_cast<int>(v);
    return pk_max(v, bit_cast<half2_t>(__builtin_amdgcn_update_dpp(i, i, CTRL, 0xF, 0xF, false)));
}

// Zero and scale of a group, and the reciprocal the codes are formed with.
struct GroupZs {
    half_t z, s;
    float sf, r;
};

template <int BITS>
__device__ __forceinline__ GroupZs group_zs(half_t hi, half_t lo) {
    constexpr float QMAX = (float)((1 << BITS) - 1);
    GroupZs g;
    half_t d = (half_t)((float)hi - (float)lo);
    if (!(d != d)) d = (half_t)fmaxf((float)d, 1e-5f);  // a NaN stays one
    g.s = (half_t)((float)d * (1.f / QMAX));
    g.sf = (float)g.s;
    const half_t t = (half_t)((float)lo / g.sf);
    half_t z = -__builtin_rintf16(t);
    if (!(z != z)) z = (half_t)fminf(fmaxf((float)z, 0.f), QMAX);
    g.z = z;
    g.r = 1.f / g.sf;
    return g;
}

// Eight weights of one group, spread with its other weights over LPG neighbouring lanes: codes as four half2 whose low
// nibbles hold them (pairs (k0, k1) .. (k6, k7)); u: the codes as fp16 values, which are NaN where the group holds one.
// Every lane of the wave has to be here.
template <int BITS, int LPG>
__device__ __forceinline__ GroupZs quantise8(half8_t w, uint32_t (&code)[4], half2_t (&u)[4], bool want_u) {
    constexpr int QMAX = (1 << BITS) - 1;
    half2_t p[4];
#pragma unroll
    for (int i = 0; i < 4; i++) p[i] = (half2_t){w[2 * i], w[2 * i + 1]};
    const half2_t hi2 = pk_max(pk_max(p[0], p[1]), pk_max(p[2], p[3]));
    const half2_t lo2 = pk_min(pk_min(p[0], p[1]), pk_min(p[2], p[3]));
    // 0 where all eight are finite
    half2_t odd = p[0] * (half2_t){(half_t)0.f, (half_t)0.f};
#pragma unroll
    for (int i = 1; i < 4; i++) odd = __builtin_elementwise_fma(p[i], (half2_t){(half_t)0.f, (half_t)0.f}, odd);
    const half_t odd1 = odd.x + odd.y;
    // (maximum, -minimum) as a pair, so that one packed maximum per step serves both
    half2_t ends = pk_max((half2_t){hi2.x, -lo2.x}, (half2_t){hi2.y, -lo2.y});
    const half_t inf = (half_t)__builtin_inff();
    if (odd1 != odd1) ends = (half2_t){inf, inf};
    ends = dpp_max<0xB1>(ends);                          // quad_perm 1,0,3,2
    ends = dpp_max<0x4E>(ends);                          // quad_perm 2,3,0,1
    if constexpr (LPG >= 8) ends = dpp_max<0x141>(ends);  // row_half_mirror: the other quad of eight lanes
    if constexpr (LPG >= 16) ends = dpp_max<0x140>(ends);  // row_mirror: the other eight of sixteen
    GroupZs g = group_zs<BITS>(ends.x, -ends.y);
    if (__builtin_amdgcn_ballot_w64(!(g.sf < __builtin_inff())) != 0) {
        bool nan = false;
        half_t hi = w[0], lo = w[0];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            nan |= w[i] != w[i];
            hi = w[i] > hi ? w[i] : hi;
            lo = w[i] < lo ? w[i] : lo;
        }
        const int lane = threadIdx.x & 63;
        const uint64_t mask = __builtin_amdgcn_ballot_w64(nan) >> (lane & ~(LPG - 1));
        ends = (half2_t){hi, -lo};
        if (nan) ends = (half2_t){inf, inf};
        ends = dpp_max<0xB1>(ends);
        ends = dpp_max<0x4E>(ends);
        if constexpr (LPG >= 8) ends = dpp_max<0x141>(ends);
        if constexpr (LPG >= 16) ends = dpp_max<0x140>(ends);
        const half_t not_a_number = (half_t)__builtin_nanf("");
        const bool group_nan = (mask & ((1ull << LPG) - 1)) != 0;
        g = group_zs<BITS>(group_nan ? not_a_number : ends.x, group_nan ? not_a_number : -ends.y);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const half_t t = (half_t)((float)w[i] / g.sf);
            half_t v = (half_t)((float)__builtin_rintf16(t) + (float)g.z);
            if (!(v != v)) v = (half_t)fminf(fmaxf((float)v, 0.f), (float)QMAX);
            u[i >> 1][i & 1] = v;
            const uint32_t c = v != v ? 0u : (uint32_t)(float)v;
            code[i >> 1] = i & 1 ? code[i >> 1] | (c << 16) : c;
        }
        return g;
    }
    constexpr float BASE = 1536.f;  // 0x6600
    const half2_t base = {(half_t)BASE, (half_t)BASE}, top = {(half_t)(BASE + QMAX), (half_t)(BASE + QMAX)};
    const half2_t z = {g.z, g.z};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        half2_t t;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const float x = (float)p[i][e];
            const float q0 = x * g.r;
            t[e] = (half_t)__builtin_fmaf(__builtin_fmaf(-q0, g.sf, x), g.r, q0);
        }
        // |t| below 512 becomes an integer above 1024; anything larger stays outside the clamp whatever it rounds to
        const half2_t v = pk_min(pk_max((t + base) + z, base), top);
        code[i] = bit_cast<uint32_t>(v);
        if (want_u) u[i] = v - base;
    }
    return g;
}

// Layout L1 nibble order k0,k2,k4,k6,k1,k3,k5,k7 from the least significant.
__device__ __forceinline__ uint32_t pack_l1_4(const uint32_t (&c)[4]) {
    return (c[0] & 0x000F000Fu) | ((c[1] & 0x000F000Fu) << 4) | ((c[2] & 0x000F000Fu) << 8) | ((c[3] & 0x000F000Fu) << 12);
}
// 2 bits: of four interleaved codes (a, b, c, d) the byte is a << 4 | b << 6 | c | d << 2; (k0,k2,k4,k6), then (k1,k3,k5,k7).
__device__ __forceinline__ uint16_t pack_l1_2(const uint32_t (&c)[4]) {
    const uint32_t t = ((c[0] & 0x00030003u) << 4) | ((c[1] & 0x00030003u) << 6) | (c[2] & 0x00030003u) | ((c[3] & 0x00030003u) << 2);
    return (uint16_t)((t & 0xFFu) | (t >> 8));
}

constexpr int Q_UNROLL = 4;  // 16-byte pieces of a thread: four loads in flight

// Everything is flat: piece i (eight weights) is word i of the packed weight, pieces LPG j .. + LPG - 1 are group j.
template <int BITS, int LPG>
__global__ __launch_bounds__(256) void quantise_l1_kernel(const half8_t* __restrict__ w, void* __restrict__ q,
                                                          half2_t* __restrict__ zs, long pieces) {
    const long i0 = (long)blockIdx.x * (256 * Q_UNROLL) + threadIdx.x;
    half8_t v[Q_UNROLL];
#pragma unroll
    for (int j = 0; j < Q_UNROLL; j++) {
        const long i = i0 + 256 * j;
        v[j] = __builtin_nontemporal_load(w + (i < pieces ? i : pieces - 1));
    }
#pragma unroll
    for (int j = 0; j < Q_UNROLL; j++) {
        const long i = i0 + 256 * j;
        uint32_t code[4];
        half2_t u[4];
        const GroupZs g = quantise8<BITS, LPG>(v[j], code, u, false);
        if (i < pieces) {
            if constexpr (BITS == 4)
                __builtin_nontemporal_store(pack_l1_4(code), (uint32_t*)q + i);
            else
                __builtin_nontemporal_store(pack_l1_2(code), (uint16_t*)q + i);
            if ((i & (LPG - 1)) == 0) zs[i / LPG] = (half2_t){(half_t)(g.z + (half_t)64.f), g.s};
        }
    }
}

// Layout L2: a workgroup takes 32 rows x 128 k (four 32 x 32 tiles of 128 words); the codes turn through LDS.
//   word `wd` of lane l of a tile, nibble b: k%32 = 16 (wd/2) + 8 ((b/2)%2) + 2 (l%4) + b/4, n%32 = 16 (wd%2) + 8 (b%2) + l/4
// The weight is read in 256-byte pieces of a row; 4-bit words of four tiles leave as 512-byte runs.
template <int BITS, int LPG>
__global__ __launch_bounds__(256) void quantise_l2_kernel(const half_t* __restrict__ w, uint32_t* __restrict__ q,
                                                          half2_t* __restrict__ zs, half_t* __restrict__ fake, int N, int K) {
    __shared__ uint32_t codes[32][17];
    const int tid = threadIdx.x;
    const int n0 = blockIdx.x * 32;
    const int k0 = blockIdx.y * 128;
    const int c = tid & 15;
    const int k = k0 + 8 * c;
    const bool inside = k < K;  // K is a multiple of 8 LPG: a group is inside or outside as a whole
    half8_t v[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int n = n0 + (tid >> 4) + 16 * j;
        v[j] = __builtin_nontemporal_load((const half8_t*)(w + (long)n * K + (inside ? k : 0)));
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int r = (tid >> 4) + 16 * j;
        const int n = n0 + r;
        uint32_t code[4];
        half2_t u[4];
        const GroupZs g = quantise8<BITS, LPG>(v[j], code, u, fake != nullptr);
        uint32_t nat = 0;  // natural order, k0 in the low nibble
#pragma unroll
        for (int i = 0; i < 4; i++) nat |= ((code[i] & 0xFu) | ((code[i] >> 12) & 0xF0u)) << (8 * i);
        codes[r][c] = nat;
        if (inside) {
            if ((c & (LPG - 1)) == 0) zs[(long)(k / (8 * LPG)) * N + n] = (half2_t){(half_t)(g.z + (half_t)64.f), g.s};
            if (fake) {
                half8_t f;
#pragma unroll
                for (int e = 0; e < 8; e++) f[e] = (half_t)((half_t)(u[e >> 1][e & 1] - g.z) * g.s);
                __builtin_nontemporal_store(f, (half8_t*)(fake + (long)n * K + k));
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int d = tid + 256 * j;
        const int t = d >> 7, lane = (d >> 2) & 31, wd = d & 3;
        if (k0 + 32 * t >= K) continue;
        uint32_t out = 0;
#pragma unroll
        for (int ch = 0; ch < 2; ch++)
#pragma unroll
            for (int rh = 0; rh < 2; rh++) {
                const uint32_t two = codes[16 * (wd & 1) + 8 * rh + (lane >> 2)][4 * t + 2 * (wd >> 1) + ch] >> (8 * (lane & 3));
                out |= ((two & 0xFu) << (4 * (2 * ch + rh))) | (((two >> 4) & 0xFu) << (4 * (4 + 2 * ch + rh)));
            }
        const long tile = (long)((k0 >> 5) + t) * (N >> 5) + blockIdx.x;
        q[tile * 128 + (d & 127)] = out;
    }
}

}  // namespace

hipError_t launch_quantise_l1(const void* w, void* q, void* zs, int N, int K, int g, int bits, hipStream_t st) {
    const long pieces = (long)N * K / 8;
    const dim3 grid((unsigned)((pieces + 256 * Q_UNROLL - 1) / (256 * Q_UNROLL)));
#define SQ_Q1(B_, L_) \
    hipLaunchKernelGGL((quantise_l1_kernel<B_, L_>), grid, dim3(256), 0, st, (const half8_t*)w, q, (half2_t*)zs, pieces)
    if (bits == 4) {
        if (g == 128) SQ_Q1(4, 16);
        else if (g == 64) SQ_Q1(4, 8);
        else SQ_Q1(4, 4);
    } else {
        if (g == 128) SQ_Q1(2, 16);
        else if (g == 64) SQ_Q1(2, 8);
        else SQ_Q1(2, 4);
    }
#undef SQ_Q1
    return hipGetLastError();
}

hipError_t launch_quantise_l2(const void* w, void* q, void* zs, void* fake, int N, int K, int g, int bits, hipStream_t st) {
    const dim3 grid(N / 32, (K + 127) / 128);
#define SQ_Q2(B_, L_)                                                                                                        \
    hipLaunchKernelGGL((quantise_l2_kernel<B_, L_>), grid, dim3(256), 0, st, (const half_t*)w, (uint32_t*)q, (half2_t*)zs, \
                       (half_t*)fake, N, K)
    if (bits == 4) {
        if (g == 128) SQ_Q2(4, 16);
        else if (g == 64) SQ_Q2(4, 8);
        else SQ_Q2(4, 4);
    } else {
        if (g == 128) SQ_Q2(2, 16);
        else if (g == 64) SQ_Q2(2, 8);
        else SQ_Q2(2, 4);
    }
#undef SQ_Q2
    return hipGetLastError();
}

}  // namespace sq
