// GEMM for 17 tokens up (any group size, any K) with layout L1: the product between a weight stream and a matrix-core
// contraction, and the contraction itself until many rounds of short K favour the two-workgroups-per-CU kernel of
// sq_gemm.hip.  At 5..16 tokens it takes the weights whose K the streaming kernel splits badly, and gate and up of a gated
// MLP in one launch (PAIR) from one token where that measures ahead; both are rules of sq_api.hip.
//
// What bounds it.  At 32..600 tokens neither HBM nor the matrix cores are full; what a CU can issue is: a
// v_mfma_f32_32x32x16_f16 takes 32 cycles and hides vector instructions of the other wave of its SIMD completely, but a
// wave gets one out every 5..6 cycles, and dequantising eight weights takes thirteen.  Beyond, the clock: with the matrix
// pipes 0.9 busy it falls to 1.5 GHz (2.4 with the same loads and no matrix instruction), so that every instruction that
// goes is time.  Hence:
//   * all waves in step, one barrier per stage (64 k of a wave), everything one slice (16 k) or two ahead in registers:
//     beside the matrix instructions of a slice stand the dequantisation of the next one's weights, the LDS reads of the
//     activations of the one after that and the stage's requests, one by one, because four waves that send theirs
//     together wait 350 cycles for the address unit.  (With two groups of waves that alternate between matrix instructions
//     and everything else, the other half, LDS trip, requests and half the dequantisation one after the other, takes 1050
//     cycles a phase against 660 of matrix instructions.  Loop cycles, alternating -> in step: 100 tokens x 15360x5120
//     42400 -> 38500, 333 x 12288x4096 83300 -> 63000, 2048 x 16384x4096 172600 -> 149500.)
//   * tiles of 32 rows alternate all the same: their two matrix instructions per slice hide no LDS trip (in step
//     against alternating, geometric means over 200 weights and token counts: 32 x 128 tiles 4.5 % slower with up to 4
//     stages, 4 % with 5..8, 2.5 % with 9..32; 32 x 64 tiles 2.5 % slower, level, 1 % faster.  800 tokens x 1024x1024 6.6 /
//     7.2 us, 32 x 8192x2048 at group size 64 8.1 / 8.5).  So does the scale on the sums (SUMS below).
//   * K is split over the waves of the workgroup (WK groups of 64 consecutive k each per stage of KS = 64 WK), so that
//     a weight row is read in 64..256-byte pieces, a stage holds 40..50 KB, and narrow weights fill the chip without
//     partial tiles in memory.  The groups' sums meet in LDS at the end.
//   * every operand goes global -> LDS by direct loads, up to ST stages ahead (three or four stages of a ring); rows past
//     M are never requested (their lanes are masked, their LDS rows are zero), so padding costs no memory traffic.
//   * where the tiles leave CUs idle, the tiles of the last, part-filled round split K over workgroups through the
//     caller's workspace.
// Measured (us per launch, cold weights, group size 128; before: sq_gemm.hip's 32..128-row tiles or the decode kernels):
//   32 tokens   4096x4096 9.9 -> 8.6, 12288x4096 14.3 -> 12.3, 4096x11008 16.5 -> 12.9, 5120x13696 27.0 -> 16.6
//   100 tokens  4096x4096 15.9 -> 11.0, 15360x5120 37.3 -> 28.8, 5120x13696 54.0 -> 30.2
//   333 tokens  4096x4096 27.0 -> 20.2, 12288x4096 65.1 -> 47.5, 5120x13696 90.3 -> 65.0
//   1024 tokens 4096x4096 46.0 -> 41, 5120x13696 202 -> 152; 2048 tokens 4096x16384 269 -> 243 (1.13 PFLOP/s)
//   in step     100 tokens 15360x5120 28.2 -> 26.9, 192 12288x4096 31.1 -> 29.8, 333 12288x4096 at group size 64
//   45.9 -> 42.7, 2048 4096x16384 246 -> 235
// Tiles of 256 x 256 with four waves of 256 x 64 (one wave per SIMD, 256 accumulation registers), which dequantise every
// weight once where eight waves of 128 x 64 did it twice, at the same loop cycles a clock of 1550 instead of 1450 MHz:
// 16384x4096 at 2048 tokens 249 -> 238, and no K groups to add up at the end.
// Tried and dropped: eight waves in step without the scheduling (8..15 % slower than alternating groups; the waits for
// LDS were not counted then, since the compiler does not see a wait in inline assembly), 32 k per wave and stage (half the
// LDS reads, no faster), four waves of 128 x 128 (250 where 256 x 64 take 238), requests between the matrix instructions
// of alternating groups (5..15 % slower), the group sums handed over in registers' order instead of row-major slices
// (1..4 % slower below 256 tokens).
//
// Operand mapping as in sq_gemm.hip: D = X W^T with activations as A (lane = row) and weights as B (lane = column);
// lane (ln, lc) of a wave holds k = 32 lc + 8 t .. + 7 of its 64 for slice t, one packed word of the weight row per
// slice; W_hat = fp16((q - z) * s) bit for bit, or with SUMS the integers q - z.
// (replaces w4a16_gemm_wmma_kernel, reference: quantization/muxi/backend/w4a16_gemm.cuh:466-600, and the role of
// turbomind::GemmS4F16, quantization/nvidia/kernel/gemm_s4_f16/gemm_template.h:358-450)
#include "sq_common.h"
#include "sq_kernels.h"

#include <type_traits>

namespace sq {

constexpr size_t RING_COUNTER_BYTES = 65536;  // start of the workspace: one uint32 per tile that splits K

struct RingPlan {
    int shape, nfull, ksplit;  // tiles below nfull are computed by one workgroup, the others by ksplit each
};

namespace {

__device__ __forceinline__ int swz8(int row) { return (row & 7) ^ ((row >> 3) & 1); }

// LDS layout of a stage: activations as WK tiles [BM rows][128 bytes], weights [BN rows][32 WK bytes], zeros/scales
// [BN columns][P pairs]; with SETS the stages hold none and behind them stand two buffers [BN columns][8 pairs].  The
// 16-byte chunks of a row are permuted (by the lane that requests them: a direct load puts lane l at 16 l) so that the
// 128-bit operand reads, lane = row, of eight and of sixteen consecutive rows fall on different banks: swz8 for rows of
// eight chunks, wswz for weight rows of 2 WK.
template <int WK>
__device__ __forceinline__ int wswz(int row) {
    if constexpr (WK == 8) return row & 15;
    if constexpr (WK == 4) return swz8(row);
    if constexpr (WK == 2) return ((row >> 1) & 3) ^ ((row >> 3) & 1);
    return ((row >> 2) & 1) ^ ((row >> 3) & 1);
}

// The largest divisor of l that is at most cap and a multiple of unit.
constexpr int ring_trip(int l, int cap, int unit) {
    int u = cap < l ? cap : l;
    while (l % u != 0 || u % unit != 0) u--;
    return u;
}

template <int MI, int NI, int WM, int WN, int WK, int GS, int ST, bool SETS>
struct RingShape {
    static constexpr int NW = WM * WN * WK, NT = 64 * NW;
    static constexpr int BM = 32 * MI * WM, BN = 32 * NI * WN, KS = 64 * WK;
    static constexpr int XB = WK * BM * 128, WB = BN * WK * 32;
    static constexpr int P = (KS >> GS) ? (KS >> GS) : 1;  // zeros/scales pairs per column and stage
    // Zeros/scales: a stage's own with its other operands, or (SETS) those of ZN stages, ZD of a row, in two buffers behind
    // the stages: see issue_set.
    static constexpr int ZD = SETS ? 8 : P, ZN = ZD / P;
    static constexpr int ZB = BN * ZD * 4;
    static constexpr int SB = XB + WB + (SETS ? 0 : ZB);
    static constexpr int XI = XB / 1024 / NW, WI = WB / 1024 / NW;
    static constexpr int ZL = BN * ZD / NW < 64 ? BN * ZD / NW : 64, ZI = BN * ZD / NW / ZL;  // lanes and instructions of a wave
    static constexpr int PER = XI + WI + (SETS ? 0 : ZI);
    static constexpr int LDS = ST * SB + (SETS ? 2 * ZB : 0);
    static constexpr int TAIL = NW * 32 * 32 * NI * 4;  // one 32-row slice of every wave's sums
    static_assert(XI * NW * 1024 == XB && WI * NW * 1024 == WB && ZI * ZL * NW == BN * ZD && (NW == 8 || NW == 4), "loads divide over the waves");
    static_assert(LDS <= 163840 && TAIL <= LDS, "fits");
    static_assert(!SETS || ZN >= ST - 1, "two buffers");
};

// EV consecutive columns of bias, multiplicand and residual, requested before the sums are there: their latency does not
// stand at the end of the kernel (bias and residual, us, without / with: 4096x4096 at 2048 tokens 76.7 / 68.9, at 100 tokens
// and 5120x5120 19.9 / 18.9; the launch without them 67.1 and 18.1).
template <int EV>
struct Cols {
    typedef _Float16 hv_t __attribute__((ext_vector_type(EV)));
    static __device__ __forceinline__ hv_t load(const half_t* p) {
        hv_t h;
        if ((reinterpret_cast<uintptr_t>(p) & (2 * EV - 1)) == 0) {
            h = *(const hv_t*)p;
        } else {
#pragma unroll
            for (int e = 0; e < EV; e++) h[e] = p[e];
        }
        return h;
    }
};
template <int EV>
struct Extra {
    typename Cols<EV>::hv_t mul, res;
    __device__ __forceinline__ void request(const Epilogue& epi, int m, int n, int N, bool inside) {
        if (epi.mul && inside) mul = Cols<EV>::load(epi.mul + (long)m * N + n);
        if (epi.residual && inside) res = Cols<EV>::load(epi.residual + (long)m * N + n);
    }
};
template <int EV>
__device__ __forceinline__ void finish_cols(float (&v)[EV], const typename Cols<EV>::hv_t& bias, const Extra<EV>& x,
                                            half_t* __restrict__ Y, int m, int n, int N, const Epilogue& epi) {
    if (epi.bias) {
#pragma unroll
        for (int e = 0; e < EV; e++) v[e] += (float)bias[e];
    }
    if (epi.act == 1) {
#pragma unroll
        for (int e = 0; e < EV; e++) v[e] = fmaxf(v[e], 0.f);
    } else if (epi.act == 2) {
#pragma unroll
        for (int e = 0; e < EV; e++) v[e] = v[e] * __builtin_amdgcn_rcpf(1.f + __expf(-v[e]));
    }
    if (epi.mul) {
#pragma unroll
        for (int e = 0; e < EV; e++) v[e] *= (float)x.mul[e];
    }
    if (epi.residual) {
#pragma unroll
        for (int e = 0; e < EV; e++) v[e] += (float)x.res[e];
    }
    typename Cols<EV>::hv_t h;
#pragma unroll
    for (int e = 0; e < EV; e++) h[e] = (half_t)v[e];
    *(typename Cols<EV>::hv_t*)(Y + (long)m * N + n) = h;
}

// silu(v[e]) * v[EO + e] for EO outputs; U (may be null) receives v[EO + e].
template <int EO>
__device__ __forceinline__ void finish_pair(const float (&v)[2 * EO], half_t* __restrict__ Y, half_t* __restrict__ U, int m, int n,
                                            int N) {
    typedef _Float16 hv_t __attribute__((ext_vector_type(EO)));
    hv_t h;
    if (U) {
#pragma unroll
        for (int e = 0; e < EO; e++) h[e] = (half_t)v[EO + e];
        *(hv_t*)(U + (long)m * N + n) = h;
    }
#pragma unroll
    for (int e = 0; e < EO; e++) h[e] = (half_t)(v[e] * __builtin_amdgcn_rcpf(1.f + __expf(-v[e])) * v[EO + e]);
    *(hv_t*)(Y + (long)m * N + n) = h;
}

// Direct loads by part of a wave's lanes (mask): the instruction is issued whatever the mask, so that the counted waits
// hold for every wave.  The wave runs with all lanes active around it.
__device__ __forceinline__ void load_to_lds_x4_masked(const void* base, uint32_t lane_byte, uint32_t lds_byte, uint64_t mask) {
    asm volatile("s_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(lane_byte), "s"(base),
                 "{m0}"(lds_byte), "s"(mask)
                 : "memory");
}

__device__ __forceinline__ void load_to_lds_x1_masked(const void* base, uint32_t lane_byte, uint32_t lds_byte, uint64_t mask) {
    asm volatile("s_mov_b64 exec, %3\n\tglobal_load_lds_dword %0, %1\n\ts_mov_b64 exec, -1" ::"v"(lane_byte), "s"(base),
                 "{m0}"(lds_byte), "s"(mask)
                 : "memory");
}

// SUMS: the matrix instructions see the integers q - z and the scale meets the sums of a stage (64 k of one group) in
// fp32, as in the decode kernels at group size 128; without it they see W_hat.  Sixteen vector instructions per 64 k and
// column tile go and sixteen per row tile come: the same count with one row tile, more with two.  Measured (us, W_hat / sums):
// 32 tokens 12288x4096 12.5 / 12.5, 5120x13696 17.1 / 17.2; 48 tokens 12288x4096 16.9 / 16.7, 5120x13696 22.4 / 22.5;
// 64 tokens 4096x11008 17.6 / 17.3, 12288x4096 17.9 / 17.3, 15360x5120 23.7 / 22.6.  Its loop keeps the two alternating groups of waves (0..3 fetch
// phase p + 1 while 4..7 compute phase p): in step it would need a second set of sums, which tiles of 64 rows (222..226 registers
// of 256) have no room for, and tiles of 32 rows are slower in step as they are.
//
// PAIR: silu(X W^T) * (X W2^T), both weights [N, K], in one launch: half of a tile's columns are W's and half W2's, the same
// outputs' in the same workgroup, so that the product is formed in the store and the tiles of both fill the chip's rounds
// together (us, two launches / one: 11008x4096 at 32 tokens 24.9 / 18.4, at 333 and group size 64 101 / 80.0; 13696x5120 at
// 100 62.7 / 43.4; 11008x4096 at 2048 396 / 329).  Nothing is rounded between the products.
template <int MI, int NI, int WM, int WN, int WK, int GS, int ST, bool SUMS, bool SETS, bool PAIR>
__global__ __launch_bounds__(64 * WM * WN * WK) __attribute__((amdgpu_waves_per_eu(WM * WN * WK / 4))) void gemm_ring_kernel(
    const uint8_t* __restrict__ W, const half2_t* __restrict__ ZS, const half_t* __restrict__ X, half_t* __restrict__ Y,
    int M, int N, int K, int mtiles, int tiles, int nfull, int ksplit, Epilogue epi, float* part, unsigned* counters,
    const uint8_t* __restrict__ W2, const half2_t* __restrict__ ZS2, half_t* __restrict__ U) {
    using S = RingShape<MI, NI, WM, WN, WK, GS, ST, SETS>;
    constexpr int BM = S::BM, BN = S::BN, KS = S::KS, SB = S::SB, XI = S::XI, WI = S::WI, ZI = S::ZI, ZL = S::ZL, PER = S::PER, P = S::P;
    constexpr int ZD = S::ZD, ZN = S::ZN;
    constexpr int X_OFF = 0, W_OFF = S::XB, Z_OFF = SETS ? ST * SB : S::XB + S::WB;
    constexpr int H = 4;  // 16-wide k slices per stage and wave
    constexpr bool ALTERNATE = SUMS || MI == 1;  // two groups of waves in turn (see the head of this file)
    static_assert(!ALTERNATE || S::NW == 8, "waves 0..3 and 4..7");
    static_assert(!SETS || (SUMS && S::P <= 2), "eight pairs of a row at once are four or eight stages'");
    static_assert(!SUMS || (MI * NI <= 4 && GS == 7 && S::NW == 8), "a stage of a wave lies in one group, and the registers suffice");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[S::LDS];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;

    const NibbleMasks nm = nibble_masks();
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31;
    const int lc = lane >> 5;
    const int kg = wave / (WM * WN);
    const int wm = (wave / WN) % WM;
    const int wn = wave % WN;

    // Which tile, and which part of K.
    int tile, z = 0, ks = 1, tr = 0;
    const int rest = tiles - nfull;
    const int id = blockIdx.x;
    if (ksplit == 1) {
        const int per = (tiles + 7) >> 3;
        tile = (id & 7) * per + (id >> 3);
        if (tile >= tiles || (id >> 3) >= per) return;
    } else if (id < nfull) {
        tile = (id & 7) * (nfull >> 3) + (id >> 3);
    } else {
        const int rid = id - nfull;
        const int per = (rest * ksplit + 7) >> 3;
        const int u = (rid & 7) * per + (rid >> 3);
        if (u >= rest * ksplit || (rid >> 3) >= per) return;
        z = u / rest;
        tr = u - z * rest;
        tile = nfull + tr;
        ks = ksplit;
    }
    const int nt = tile / mtiles;
    const int m0 = (tile - nt * mtiles) * BM;
    // PAIR: rows 0 .. BN / 2 - 1 of the stage's weights are W's, the others W2's, for outputs n0 .. n0 + BN / 2 - 1.
    constexpr int BO = PAIR ? BN / 2 : BN;
    const int n0 = nt * BO;
    const bool second = PAIR && wave >= S::NW / 2;  // this wave loads W2
    const uint8_t* const Wl = second ? W2 : W;
    const half2_t* const Zl = second ? ZS2 : ZS;
    const int groups = K >> GS;
    const int nst = (K + KS - 1) / KS;
    const int spz = (nst + ks - 1) / ks;
    const int it0 = z * spz;
    const int it1 = imin(it0 + spz, nst);

    // Byte offsets of this wave's loads; the part along K is a wave-uniform base.
    uint32_t xlane[XI], wlane[WI], zlane[ZI];
    uint64_t xmask[XI];  // lanes whose row exists; the others' LDS rows stay zero
    constexpr uint64_t zmask = ZL == 64 ? ~0ull : (1ull << (ZL & 63)) - 1;
#pragma unroll
    for (int j = 0; j < XI; j++) {
        const int ii = wave * XI + j;
        const int R = (ii % (BM / 8)) * 8 + (lane >> 3);
        xlane[j] = (uint32_t)((long)imin(m0 + R, M - 1) * K * 2) + (64 * (ii / (BM / 8)) + ((lane & 7) ^ swz8(R)) * 8) * 2;
        xmask[j] = __builtin_amdgcn_ballot_w64(m0 + R < M);
        if (m0 + R >= M) {
            const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int c = 0; c < ST; c++) *(u32x4_t*)(lds + X_OFF + c * SB + (wave * XI + j) * 1024 + lane * 16) = zero;
        }
    }
#pragma unroll
    for (int j = 0; j < WI; j++) {
        const int R = (wave * WI + j) * (32 / WK) + lane / (2 * WK);
        wlane[j] = (uint32_t)((long)imin(n0 + R % BO, N - 1) * (K >> 1)) + (((lane % (2 * WK)) ^ wswz<WK>(R)) * 16);
    }
#pragma unroll
    for (int j = 0; j < ZI; j++) {
        const int d = (wave * ZI + j) * ZL + (lane & (ZL - 1));
        zlane[j] = (uint32_t)((long)imin(n0 + d / ZD % BO, N - 1) * groups * 4) + (SETS ? 0 : d % P * 4);
    }
    // A stage's own zeros/scales are 4 or 8 bytes of a row, each in a line of its own: with 32 rows per tile a third of the lines
    // that a stage asks for, and the loads come back in order.  So, where that is ahead (ring_sets), 32 bytes of a row at once, in
    // front of the first of the ZN stages that they serve (gate and up of 11008x4096 at 32 tokens: 1.52 M accesses of the L1s
    // instead of 2.14, 0.82 M requests to the L2s instead of 1.05, the same reads from memory; us: 64 tokens 12288x4096 in tiles
    // of 64 x 128 23.2 -> 21.9, 64 x 256 split in two 26.5 -> 25.4; 32 tokens 4096x11008 in tiles of 32 x 128 split in two 24.4 ->
    // 22.7, gate and up of 11008x4096 19.4 -> 17.8).
    // Two buffers: set s goes out when all have read stage ZN s - ST, which is no earlier than the last one of set s - 2.  Not for
    // the waves in step: the branch in their loop costs what it saves (100 tokens 15360x5120 in tiles of 96 x 128 32.3 -> 33.8, 200
    // 12288x4096 in 96 x 256 34.9 -> 37.3, 333 at group size 64 41.4 -> 42.3).
    auto issue_set = [&](int set) {
        const int g = ((it0 * KS) >> GS) + set * ZD;
#pragma unroll
        for (int j = 0; j < ZI; j++)
            load_to_lds_x1_masked(Zl, zlane[j] + imin(g + lane % ZD, groups - 1) * 4,
                                  lds0 + Z_OFF + (set & 1) * S::ZB + (wave * ZI + j) * ZL * 4, zmask);
    };
    // Loads of stage it into slot c.  EDGE: the last stage of a K that ends inside it; weights that are missing re-read
    // the end of the row (and meet a scale of 0), activations are zeros in LDS (an infinity at the end of a row, re-read,
    // would be a NaN in every column.  Clearing the operands in the last stages' registers instead cost the 256 x 256 tiles
    // 0.9 % whatever K was: 16384x4096 at 4096 tokens 493 -> 498 us).
    auto issue = [&](int it, int c, auto EDGE_, int lo = 0, int hi = 1 << 20) __attribute__((always_inline)) {  // requests lo .. hi - 1
        constexpr bool EDGE = decltype(EDGE_)::value;
        const int k0 = it * KS, left = K - k0;
        const uint8_t* xb = (const uint8_t*)X + (long)k0 * 2;
        const uint8_t* wb = Wl + (k0 >> 1);
        const uint8_t* zb = (const uint8_t*)Zl + (k0 >> GS) * 4;
        const uint32_t l0 = lds0 + c * SB;
        constexpr int ZP = SETS ? 0 : ZI;
#pragma unroll
        for (int j = 0; j < (SETS ? 0 : ZI); j++) {
            if (j < lo || j >= hi) continue;
            uint32_t o = zlane[j];
            if constexpr (EDGE) {
                const int p = ((wave * ZI + j) * ZL + (lane & (ZL - 1))) % P;
                o = o - p * 4 + imin(p, groups - 1 - (k0 >> GS)) * 4;
            }
            load_to_lds_x1_masked(zb, o, l0 + Z_OFF + (wave * ZI + j) * ZL * 4, zmask);
        }
#pragma unroll
        for (int j = 0; j < WI; j++) {
            if (ZP + j < lo || ZP + j >= hi) continue;
            uint32_t o = wlane[j];
            if constexpr (EDGE) {
                const int R = (wave * WI + j) * (32 / WK) + lane / (2 * WK);
                const int p = ((lane % (2 * WK)) ^ wswz<WK>(R)) * 16;
                o = o - p + imin(p, (left - 32) >> 1);
            }
            load_to_lds_x4(wb, o, l0 + W_OFF + (wave * WI + j) * 1024);
        }
#pragma unroll
        for (int j = 0; j < XI; j++) {
            if (ZP + WI + j < lo || ZP + WI + j >= hi) continue;
            uint64_t mask = xmask[j];
            if constexpr (EDGE) {
                const int ii = wave * XI + j;
                const int R = (ii % (BM / 8)) * 8 + (lane >> 3);
                const bool past = 64 * (ii / (BM / 8)) + ((lane & 7) ^ swz8(R)) * 8 >= left;
                if (past) *(u32x4_t*)(lds + X_OFF + c * SB + ii * 1024 + lane * 16) = (u32x4_t){0u, 0u, 0u, 0u};
                mask &= __builtin_amdgcn_ballot_w64(!past);
            }
            load_to_lds_x4_masked(xb, xlane[j], l0 + X_OFF + (wave * XI + j) * 1024, mask);
        }
    };
    auto issue_any = [&](int it, int c) {
        if constexpr (SETS) {
            if ((it - it0) % ZN == 0) issue_set((it - it0) / ZN);
        }
        if (it * KS + KS <= K)
            issue(it, c, std::false_type{});
        else
            issue(it, c, std::true_type{});
    };

    const int xrow = X_OFF + kg * (BM * 128) + (wm * 32 * MI + ln) * 128;
    int xoff[4];
#pragma unroll
    for (int t = 0; t < 4; t++) xoff[t] = xrow + (((4 * lc + t) ^ swz8(ln)) * 16);
    // Row of the stage's weights (and column of the sums on their way out) of the wave's first 32 columns; CN to the next 32.
    constexpr int CN = PAIR ? BO : 32;
    const int wcol = (PAIR ? (NI == 2 ? 32 * wn : (wn & 1) * BO + 32 * (wn >> 1)) : wn * 32 * NI) + ln;
    static_assert(!PAIR || NI == 2 || (NI == 1 && WN % 2 == 0), "both weights of an output column in one wave or in neighbours");
    const int woff = W_OFF + wcol * (32 * WK) + (((2 * kg + lc) ^ wswz<WK>(ln)) * 16);
    const int zoff = Z_OFF + (wcol * ZD + ((64 * kg + (GS == 5 ? 32 * lc : 0)) >> GS)) * 4;

    float16_t acc[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[mi][ni][v] = 0.f;

    auto wait_lds = []() { __builtin_amdgcn_s_waitcnt(0xC07F); };  // lgkmcnt(0), where the compiler sees it: later waits stay counted
    if constexpr (!ALTERNATE) {
        half8_t a[4][MI], b[2][NI];               // activations of slice t in a[t], weights of slice t in b[t & 1]
        uint32_t q[NI][4], q3[NI], qn[NI][4];     // packed words of the stage (the last one apart), and of the next stage
        half2_t zs[NI], zn[NI], z1024[NI];
        uint32_t hi8[NI];
        auto read_weights = [&](int c) {
            const uint8_t* l = lds + c * SB;
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                zn[ni] = *(const half2_t*)(l + zoff + ni * (CN * P * 4));
                const u32x4_t v = *(const u32x4_t*)(l + woff + ni * (CN * 32 * WK));
#pragma unroll
                for (int t = 0; t < 4; t++) qn[ni][t] = v[t];
            }
        };
        auto read_rows = [&](int c, int t, int lo, int hi) __attribute__((always_inline)) {
#pragma unroll
            for (int r = lo; r < hi; r++) a[t][r] = *(const half8_t*)(lds + c * SB + xoff[t] + r * 4096);
        };
        // Weights past the end of K get the scale 0 (only the last stage can hold any).
        auto clip = [&](int it) {
            if (it * KS + 64 * kg + (GS == 5 ? 32 * lc : 0) >= K) {
#pragma unroll
                for (int ni = 0; ni < NI; ni++) zn[ni].y = (half_t)0.f;
            }
        };
        // Pair j of a word, i.e. two of its eight weights, as dequant8 gives them.
        auto dequantise_pair = [&](int slot, int ni, int j, uint32_t w, half2_t z) __attribute__((always_inline)) {
            const half2_t z64 = {z.x, z.x}, sc = {z.y, z.y};
            if (j == 0) z1024[ni] = z64 + (half2_t){(half_t)960.f, (half_t)960.f};
            if (j == 2) hi8[ni] = w >> 8;
            const uint32_t src = j < 2 ? w : hi8[ni];
            u32x4_t v = bit_cast<u32x4_t>(b[slot][ni]);
            v[j] = (j & 1) ? dequant_pair((src & nm.hi) | 0x54005400u, z64, sc)
                           : dequant_pair((src & nm.lo) | 0x64006400u, z1024[ni], sc);
            b[slot][ni] = bit_cast<half8_t>(v);
        };
        // The next stage becomes readable in the middle of a stage, in front of row block BAR of slice 2: by then the last
        // rows of the stage, requested from LDS in slice 1, have arrived without a wait, and its slot is free.
        constexpr int BAR = MI >= 4 ? 1 : 0;
        constexpr int PAIRS = 4 * NI;  // of a slice
        constexpr int NB = 4 * MI;     // row blocks of a stage, counted from slice 2 for the requests
        // Slice t of the stage in slot c, row block by row block: matrix instructions, beside them a share of the next
        // slice's dequantisation and of the rows of the slice after that (from slot cn past the middle); behind them the
        // requests(row block).
        auto slice = [&](auto t_, int c, int cn, auto middle, auto requests) __attribute__((always_inline)) {
            constexpr int t = decltype(t_)::value;
#pragma unroll
            for (int mi = 0; mi < MI; mi++) {
                if (t == 2 && mi == BAR) middle();
                constexpr int first = t == 2 ? BAR : 0, n = MI - first;
                if (mi >= first) read_rows(t < 2 ? c : cn, (t + 2) & 3, (mi - first) * MI / n, (mi - first + 1) * MI / n);
#pragma unroll
                for (int ni = 0; ni < NI; ni++)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t][mi], b[t & 1][ni], acc[mi][ni], 0, 0, 0);
#pragma unroll
                for (int k = mi * PAIRS / MI; k < (mi + 1) * PAIRS / MI; k++) {
                    const int ni = k / 4;
                    if constexpr (t < 2)
                        dequantise_pair((t + 1) & 1, ni, k & 3, q[ni][t + 1], zs[ni]);
                    else if constexpr (t == 2)
                        dequantise_pair(1, ni, k & 3, mi < BAR ? q[ni][3] : q3[ni], zs[ni]);
                    else
                        dequantise_pair(0, ni, k & 3, qn[ni][0], zn[ni]);
                }
                constexpr int VA = (14 * NI + MI * NI - 1) / (MI * NI);
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, VA, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                requests(((t + 2) & 3) * MI + mi);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {  // finished here, not where the matrix instructions want it
                u32x4_t v = bit_cast<u32x4_t>(b[(t + 1) & 1][ni]);
                asm volatile("" : "+v"(v));
                b[(t + 1) & 1][ni] = bit_cast<half8_t>(v);
            }
        };
        auto keep_last_word = [&]() {
#pragma unroll
            for (int ni = 0; ni < NI; ni++) q3[ni] = q[ni][3];
        };
        auto take = [&]() {
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                zs[ni] = zn[ni];
#pragma unroll
                for (int t = 0; t < 4; t++) q[ni][t] = qn[ni][t];
            }
        };
        // Middle of a stage: the next one has landed (full: all but the ST - 2 younger ones), and every wave has read this one.
        auto landed = [&](bool full) {
            wait_lds();
            if (full)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((ST - 2) * PER) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        };
        using T0 = std::integral_constant<int, 0>;
        using T1 = std::integral_constant<int, 1>;
        using T2 = std::integral_constant<int, 2>;
        using T3 = std::integral_constant<int, 3>;
        using Yes = std::true_type;
        using No = std::false_type;
        if (it0 < it1) {
            // The first stage's loads of all waves before any wave's second, and the last slot's behind the first reads.
#pragma unroll
            for (int s = 0; s < ST - 1; s++) {
                if (it0 + s < it1) issue_any(it0 + s, s);
                if (s == 0) __builtin_amdgcn_s_barrier();
            }
            landed(it0 + ST - 1 <= it1);
            read_weights(0);
            read_rows(0, 0, 0, MI);
            read_rows(0, 1, 0, MI);
            if (it0 + ST - 1 < it1) issue_any(it0 + ST - 1, ST - 1);
            clip(it0);
#pragma unroll
            for (int k = 0; k < PAIRS; k++) dequantise_pair(0, k / 4, k & 3, qn[k / 4][0], zn[k / 4]);
            take();
            int c = 0, cp = ST - 1, it = it0;
            auto nothing = []() {};
            auto no_requests = [](int) {};
            // A stage that requests stage it + ST, a whole one, into its own slot from the middle on, the rest of it in the
            // stage after (FIRST: none of it is left from the stage before).  No branch inside: the waits for LDS stay counted.
            const int plain = it1 * KS > K ? it1 - 1 : it1;
            auto stage = [&](auto first_) {
                constexpr bool FIRST = decltype(first_)::value;
                const int cn = c == ST - 1 ? 0 : c + 1;
                auto rest = [&](int o) __attribute__((always_inline)) {
                    if constexpr (!FIRST) issue(it + ST - 1, cp, std::false_type{}, o * PER / NB, (o + 1) * PER / NB);
                };
                auto begin = [&](int o) __attribute__((always_inline)) {
                    if (o >= BAR) issue(it + ST, c, std::false_type{}, o == BAR ? 0 : o * PER / NB, (o + 1) * PER / NB);
                };
                auto middle = [&]() {
                    keep_last_word();
                    landed(true);
                    read_weights(cn);
                };
                slice(T0{}, c, cn, nothing, rest);
                slice(T1{}, c, cn, nothing, rest);
                slice(T2{}, c, cn, middle, begin);
                slice(T3{}, c, cn, nothing, begin);
                take();
                cp = c;
                c = cn;
                it++;
            };
            if (it + ST < plain) {
                stage(Yes{});
                while (it + ST < plain) stage(No{});
                issue(it + ST - 1, cp, std::false_type{}, 2 * MI * PER / NB, PER);
            }
            // The last ST stages, and one more where K ends inside the last: nothing left to request but that one.  The slices
            // are those of the loop above, so the last stage reads a slot that nobody multiplies.  (Where a workgroup has no
            // more stages than these, reading the next stage's operands all at once behind the barrier is time: 256 x 256
            // tiles with 9..16 stages 1.5 % of the launch, 96 x 128 and 128 x 128 with 8 or fewer 1 %.)
            for (; it < it1; it++) {
                const int cn = c == ST - 1 ? 0 : c + 1;
                auto middle = [&]() {
                    keep_last_word();
                    landed(it + ST - 1 < it1);
                    if (it + ST < it1) issue_any(it + ST, c);
                    read_weights(cn);
                };
                slice(T0{}, c, cn, nothing, no_requests);
                slice(T1{}, c, cn, nothing, no_requests);
                slice(T2{}, c, cn, middle, no_requests);
                clip(it + 1);
                slice(T3{}, c, cn, nothing, no_requests);
                take();
                c = cn;
            }
        }
    } else {
        half8_t a[H][MI], b[H][NI];
        half2_t zs[NI];
        uint32_t q[NI][H];
        float16_t part_sum[SUMS ? MI : 1][SUMS ? NI : 1];  // of the stage before, and its scales
        float part_scale[SUMS ? NI : 1];
        if constexpr (SUMS) {
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                part_scale[ni] = 0.f;
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
#pragma unroll
                    for (int v = 0; v < 16; v++) part_sum[mi][ni][v] = 0.f;
            }
        }
        // (pinned, so that the wait for the matrix instructions' results is not moved in front of the barrier)
        auto fold = [&]() {
            if constexpr (SUMS) {
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
#pragma unroll
                    for (int ni = 0; ni < NI; ni++) {
                        asm volatile("" : "+v"(part_sum[mi][ni]));
#pragma unroll
                        for (int v = 0; v < 16; v++)
                            acc[mi][ni][v] = __builtin_fmaf(part_sum[mi][ni][v], part_scale[ni], acc[mi][ni][v]);
                    }
            }
        };
        auto unpack = [&](int t) {
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                const half2_t z = {zs[ni].x, zs[ni].x};
                b[t][ni] = SUMS ? integers8(q[ni][t], z, nm) : dequant8(q[ni][t], z, (half2_t){zs[ni].y, zs[ni].y}, nm);
            }
        };
        // The wave's operands of the stage in slot c into registers.
        auto fetch = [&](int it, int c) {
            const uint8_t* l = lds + c * SB;
            const uint8_t* zl = l;
            if constexpr (SETS) zl = lds + (it - it0) / ZN % 2 * S::ZB + (it - it0) % ZN * (P * 4);
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                zs[ni] = *(const half2_t*)(zl + zoff + ni * (CN * ZD * 4));
                const u32x4_t v = *(const u32x4_t*)(l + woff + ni * (CN * 32 * WK));
#pragma unroll
                for (int t = 0; t < 4; t++) q[ni][t] = v[t];
            }
#pragma unroll
            for (int t = 0; t < H; t++)
#pragma unroll
                for (int mi = 0; mi < MI; mi++) a[t][mi] = *(const half8_t*)(l + xoff[t] + mi * 4096);
        };
        // Weights past the end of K get the scale 0 (only the last stage can hold any).
        auto clip = [&](int it) {
            if (it * KS + 64 * kg + (GS == 5 ? 32 * lc : 0) >= K) {
#pragma unroll
                for (int ni = 0; ni < NI; ni++) zs[ni].y = (half_t)0.f;
            }
        };
        // the first half of the stage's weights, finished in front of the barrier that follows
        auto unpack_first = [&]() {
            fold();
#pragma unroll
            for (int t = 0; t < H / 2; t++) {
                unpack(t);
#pragma unroll
                for (int ni = 0; ni < NI; ni++) {
                    u32x4_t v = bit_cast<u32x4_t>(b[t][ni]);
                    asm volatile("" : "+v"(v));
                    b[t][ni] = bit_cast<half8_t>(v);
                }
            }
        };
        // Matrix instructions of the stage; those of its first half hide the unpacking of the second.
        auto compute = [&]() {
#pragma unroll
            for (int ni = 0; ni < NI; ni++)
#pragma unroll
                for (int t = H / 2; t < H; t++) asm volatile("" : "+v"(q[ni][t]));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = H / 2; t < H; t++) unpack(t);
#pragma unroll
            for (int t = 0; t < H; t++)
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
#pragma unroll
                    for (int ni = 0; ni < NI; ni++) {
                        if constexpr (SUMS)
                            part_sum[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                a[t][mi], b[t][ni], t == 0 ? (float16_t){} : part_sum[mi][ni], 0, 0, 0);
                        else
                            acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t][mi], b[t][ni], acc[mi][ni], 0, 0, 0);
                    }
            if constexpr (SUMS) {
#pragma unroll
                for (int ni = 0; ni < NI; ni++) part_scale[ni] = (float)zs[ni].y;
            }
            constexpr int MF = H / 2 * MI * NI, VA = ((SUMS ? 10 : 14) * NI * (H / 2) + MF - 1) / MF;
#pragma unroll
            for (int i = 0; i < MF; i++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, VA, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x8, MF, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        if (it0 < it1) {
#pragma unroll
            for (int s = 0; s < ST - 1; s++)
                if (it0 + s < it1) issue_any(it0 + s, s);
            // Stage it + 1 has landed: all but the loads of the younger stages are done.
            auto landed_full = [&](int it) {
                if (SETS && (it - it0 + ST - 1) % ZN < ST - 2)  // a set went out with one of the younger ones
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((ST - 2) * PER + ZI) : "memory");
                else
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((ST - 2) * PER) : "memory");
            };
            auto landed_all = []() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
            auto turn = []() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
            if (it0 + ST - 1 <= it1)
                landed_full(it0 - 1);
            else
                landed_all();
            int c = 0, cp = ST - 1, it = it0;
            auto next = [&]() {
                cp = c;
                c = c == ST - 1 ? 0 : c + 1;
            };
            const int full = it1 - (ST - 1);  // stages below it still have a stage to request
            // Both branches pass the same barriers, two per stage: waves 0..3 fetch stage it + 1 while waves 4..7 compute
            // stage it.  A fetch also requests stage it + ST - 1 into the slot of stage it - 1, which both groups have
            // read by then.
            if (wave < 4) {
                fetch(it, 0);
                if (it < full)
                    issue_any(it + ST - 1, ST - 1);
                else
                    clip(it);
                unpack_first();
                turn();
                for (; it + 1 < full; it++) {
                    compute();
                    landed_full(it);
                    next();
                    fetch(it + 1, c);
                    issue_any(it + ST, cp);
                    unpack_first();
                    turn();
                }
                for (; it < it1; it++) {
                    compute();
                    landed_all();
                    next();
                    if (it + 1 < it1) {
                        fetch(it + 1, c);
                        clip(it + 1);
                        unpack_first();
                    }
                    turn();
                }
            } else {
                turn();
                for (; it < full; it++) {
                    fetch(it, c);
                    issue_any(it + ST - 1, cp);
                    unpack_first();
                    landed_full(it);
                    compute();
                    next();
                    turn();
                }
                for (; it < it1; it++) {
                    fetch(it, c);
                    clip(it);
                    unpack_first();
                    landed_all();
                    compute();
                    next();
                    turn();
                }
            }
            fold();
        }
    }

    // One test in front of all requests of multiplicand and residual: a launch without them otherwise passes a branch for
    // every chunk (256 x 256 tiles with 9..16 stages 4 % slower, 64 x 256 and 128 x 128 with up to four 2 %).
    const bool extras = !PAIR && (epi.mul || epi.residual);
    if constexpr (WK == 1) {
        if (ks == 1) {
            // No sums to add: every wave turns its own half slices (16 rows) row-major through a region of its own, two in
            // turn, so that nothing waits for another wave.
            constexpr int HC = 32 * NI;                             // columns of a wave, PAIR: of 32 outputs
            constexpr int CH = HC / (PAIR ? 16 : 8), RP = 64 / CH;  // chunks of a row, rows per pass
            constexpr int EO = PAIR ? 16 : 8;                       // sums of a chunk
            static_assert(S::NW * 2 * 16 * HC * 4 <= S::LDS && 16 % RP == 0, "fits");
            float* own = reinterpret_cast<float*>(lds) + wave * (2 * 16 * HC);
            float v[2][16 / RP][EO];
            auto turn_over = [&](int hs) __attribute__((always_inline)) {
                float* o = own + (hs & 1) * (16 * HC);
#pragma unroll
                for (int ni = 0; ni < NI; ni++)
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        o[(8 * (e >> 2) + 4 * lc + (e & 3)) * HC + 32 * ni + ln] = acc[hs >> 1][ni][8 * (hs & 1) + e];
                asm volatile("" ::: "memory");
#pragma unroll
                for (int g = 0; g < 16 / RP; g++)
#pragma unroll
                    for (int e = 0; e < EO; e++)
                        v[hs & 1][g][e] = o[(g * RP + lane / CH) * HC + (lane % CH) * 8 + (e & 7) + (e >> 3) * 32];
                asm volatile("" ::: "memory");
            };
            const int n = n0 + wn * (PAIR ? 32 : HC) + (lane % CH) * 8;
            // bias, multiplicand and residual of a half slice are requested DEEP half slices ahead
            constexpr int DEEP = 3;
            half8_t bias = {};
            Extra<8> extra[DEEP + 1][16 / RP];
            auto row_of = [&](int hs, int g) { return m0 + wm * (32 * MI) + 16 * hs + g * RP + lane / CH; };
            auto request = [&](int hs) __attribute__((always_inline)) {
                if constexpr (!PAIR) {
#pragma unroll
                    for (int g = 0; g < 16 / RP; g++) extra[hs % (DEEP + 1)][g].request(epi, row_of(hs, g), n, N, row_of(hs, g) < M && n < N);
                }
            };
            if (!PAIR && epi.bias && n < N) bias = Cols<8>::load(epi.bias + n);
            if (extras) {
#pragma unroll
                for (int hs = 0; hs < DEEP; hs++) request(hs);
            }
            __syncthreads();
            turn_over(0);
#pragma unroll
            for (int hs = 0; hs < 2 * MI; hs++) {
                if (extras && hs + DEEP < 2 * MI) request(hs + DEEP);
                if (hs + 1 < 2 * MI) turn_over(hs + 1);
#pragma unroll
                for (int g = 0; g < 16 / RP; g++) {
                    const int m = row_of(hs, g);
                    if (m < M && n < N) {
                        if constexpr (PAIR)
                            finish_pair<8>(v[hs & 1][g], Y, U, m, n, N);
                        else
                            finish_cols<8>(v[hs & 1][g], bias, extra[hs % (DEEP + 1)][g], Y, m, n, N, epi);
                    }
                }
            }
            return;
        }
    }

    // The K groups' sums meet in LDS, one 32-row slice of every row group at a time, and leave row-major, EV consecutive
    // columns per thread.
    constexpr int PT = 16 * NI / WK;     // sums per thread and slice
    constexpr int EO = PAIR ? (PT < 16 ? PT / 2 : 8) : (PT < 8 ? PT : 8);  // outputs of a chunk
    constexpr int EV = PAIR ? 2 * EO : EO;                                 // its sums
    constexpr int G = PT / EV;
    constexpr int CPR = BN / EV;         // chunks per row
    constexpr int L = MI * PT / 4;       // float4 per thread
    float* red = reinterpret_cast<float*>(lds);
    const long tsz = (long)BM * BN;
    float* mine = part + ((long)z * rest + tr) * tsz + tid * 4;
    static_assert(S::NT % CPR == 0, "the column chunk of a thread is the same in every slice");
    const int n_out = n0 + tid % CPR * EO;
    auto row_of = [&](int mi, int g) {
        const int r = (tid + g * S::NT) / CPR;
        return m0 + (r >> 5) * (32 * MI) + 32 * mi + (r & 31);
    };
    typename Cols<EO>::hv_t bias = {};
    // (where K is split only the last of the workgroups needs it, and asks then: 17..32 tokens at group size 128 0.5 % less)
    if (ks == 1 && !PAIR && epi.bias && n_out < N) bias = Cols<EO>::load(epi.bias + n_out);
    auto request = [&](Extra<EO>& x, int mi, int g) __attribute__((always_inline)) {
        if constexpr (!PAIR) x.request(epi, row_of(mi, g), n_out, N, row_of(mi, g) < M && n_out < N);
    };
    auto finish = [&](int mi, int g, float (&v)[EV], const Extra<EO>& x) {
        const int m = row_of(mi, g);
        if (m < M && n_out < N) {
            if constexpr (PAIR)
                finish_pair<EO>(v, Y, U, m, n_out, N);
            else
                finish_cols<EV>(v, bias, x, Y, m, n_out, N, epi);
        }
    };
    auto column = [](int cc, int e) __attribute__((always_inline)) { return cc * EO + e % EO + (e / EO) * BO; };
    // Slices at once: several behind one barrier where a slice is one chunk a thread (tiles of 128 columns, 96 and 128 rows:
    // one by one 0.5..1 % slower); else one, so that a slice's stores go out while the next one's sums are added (64 x 256
    // tiles with up to 4 stages 2 % slower with all slices at once, 128 x 256 1 %).
    constexpr int SL = NI > 1 || MI < 3 ? 1 : S::LDS / S::TAIL < MI ? S::LDS / S::TAIL : MI;
    constexpr int SF = S::TAIL / 4;
    Extra<EO> extra[SL][G];
#pragma unroll
    for (int mi = 0; mi < MI; mi++) {
        if (mi % SL == 0) {
            if (extras && ks == 1) {
#pragma unroll
                for (int sl = 0; sl < SL && mi + sl < MI; sl++)
#pragma unroll
                    for (int g = 0; g < G; g++) request(extra[sl][g], mi + sl, g);
            }
            __syncthreads();
#pragma unroll
            for (int sl = 0; sl < SL && mi + sl < MI; sl++)
#pragma unroll
                for (int ni = 0; ni < NI; ni++)
#pragma unroll
                    for (int v = 0; v < 16; v++)
                        red[sl * SF + ((kg * WM + wm) * 32 + 8 * (v >> 2) + 4 * lc + (v & 3)) * BN + wcol + CN * ni] = acc[mi + sl][ni][v];
            __syncthreads();
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int ch = tid + g * S::NT;
            const int r = ch / CPR, cc = ch % CPR;  // r: row of the WM * 32 of this slice
            float v[EV];
#pragma unroll
            for (int e = 0; e < EV; e++) v[e] = red[mi % SL * SF + r * BN + column(cc, e)];
#pragma unroll
            for (int q = 1; q < WK; q++)
#pragma unroll
                for (int e = 0; e < EV; e++) v[e] += red[mi % SL * SF + (q * WM * 32 + r) * BN + column(cc, e)];
            if (ks == 1) {
                finish(mi, g, v, extra[mi % SL][g]);
            } else {
#pragma unroll
                for (int h = 0; h < EV / 4; h++)
                    store_coherent_x4(mine + ((mi * G + g) * (EV / 4) + h) * (S::NT * 4),
                                      (float4_t){v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]});
            }
        }
    }
    if (ks > 1) {
        // Partial tiles meet in the workspace: device-coherent stores, one counter per tile.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        unsigned* last_flag = reinterpret_cast<unsigned*>(lds);
        if (tid == 0) {
            const unsigned old = __hip_atomic_fetch_add(&counters[tr], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *last_flag = (old == (unsigned)(ks - 1)) ? 1u : 0u;
        }
        __syncthreads();
        if (!*last_flag) return;
        if (!PAIR && epi.bias && n_out < N) bias = Cols<EO>::load(epi.bias + n_out);
        // The last of the tile's workgroups adds the partial sums in the order of the K ranges (bit-reproducible whoever
        // comes last); up to 32 loads per thread are in flight, nothing else hides their latency.
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(part, 0, 0x7FFFFFFF, 0x00027000);
        auto reduce = [&](auto NZ_) {
            constexpr int NZ = decltype(NZ_)::value;          // ranges, rounded up
            constexpr int U = ring_trip(L, 32 / NZ, EV / 4);  // float4 per thread and trip
            static_assert(L % U == 0 && U % (EV / 4) == 0, "whole trips");
#pragma unroll 1
            for (int l0 = 0; l0 < L; l0 += U) {
                u32x4_t pv[U][NZ];
                Extra<EO> px[U / (EV / 4)];
                if (extras) {
#pragma unroll
                    for (int i0 = 0; i0 < U; i0 += EV / 4)
                        request(px[i0 / (EV / 4)], (l0 + i0) / (EV / 4) / G, (l0 + i0) / (EV / 4) % G);
                }
                const uint32_t base = (uint32_t)(((long)tr * tsz + (long)l0 * (S::NT * 4) + tid * 4) * 4);
                const uint32_t zstep = (uint32_t)((long)rest * tsz * 4);
#pragma unroll
                for (int q = 0; q < NZ; q++)
#pragma unroll
                    for (int i = 0; i < U; i++)
                        pv[i][q] = __builtin_amdgcn_raw_buffer_load_b128(rs, base + i * (S::NT * 16), q < ks ? q * zstep : 0, 16);
#pragma unroll
                for (int i0 = 0; i0 < U; i0 += EV / 4) {
                    float v[EV];
#pragma unroll
                    for (int i = i0; i < i0 + EV / 4; i++) {
                        float4_t sum = bit_cast<float4_t>(pv[i][0]);
#pragma unroll
                        for (int q = 1; q < NZ; q++)
                            if (q < ks) sum += bit_cast<float4_t>(pv[i][q]);
#pragma unroll
                        for (int e = 0; e < 4; e++) v[4 * (i - i0) + e] = sum[e];
                    }
                    const int chunk = (l0 + i0) / (EV / 4);
                    finish(chunk / G, chunk % G, v, px[i0 / (EV / 4)]);
                }
            }
        };
        if (ks <= 2)
            reduce(std::integral_constant<int, 2>{});
        else if (ks <= 4)
            reduce(std::integral_constant<int, 4>{});
        else
            reduce(std::integral_constant<int, 8>{});
        if (tid == 0) __hip_atomic_store(&counters[tr], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

}  // namespace

// The shapes that are built: {MI, NI, WM, WN, WK, stages}, i.e. a (32 MI WM) x (32 NI WN) tile and 64 WK columns of K
// per stage.  LDS holds three or four stages.  Tiles of 32 and 64 rows also with the scale on the sums.
#define SQ_RING_LOW_SHAPES(X_) \
    X_(1, 1, 2, 1, 1, 8, 3) X_(2, 1, 2, 1, 2, 4, 4) X_(3, 2, 2, 1, 2, 4, 3) X_(5, 2, 2, 1, 4, 2, 4)
#define SQ_RING_SHAPES(X_)                                                                               \
    SQ_RING_LOW_SHAPES(X_) X_(4, 3, 1, 1, 4, 2, 4) X_(6, 3, 2, 1, 4, 2, 3) X_(7, 4, 1, 1, 4, 2, 3)        \
        X_(8, 4, 2, 1, 4, 2, 3) X_(9, 8, 2, 1, 4, 1, 3)

template <int MI, int NI, int WM, int WN, int WK, int GS, int ST, bool SUMS, bool SETS, bool PAIR>
static hipError_t launch_shape(const void* x, const void* w, const void* zs, const void* w2, const void* zs2, void* y, void* u, int M,
                               int N, int K, int nfull, int ksplit, Epilogue epi, void* ws, hipStream_t st) {
    using S = RingShape<MI, NI, WM, WN, WK, GS, ST, SETS>;
    const int mt = (M + S::BM - 1) / S::BM;
    constexpr int BO = PAIR ? S::BN / 2 : S::BN;
    const int tiles = mt * ((N + BO - 1) / BO);
    if (ksplit == 1) nfull = tiles;
    const int grid = ksplit == 1 ? (tiles + 7) / 8 * 8 : nfull + ((tiles - nfull) * ksplit + 7) / 8 * 8;
    hipLaunchKernelGGL((gemm_ring_kernel<MI, NI, WM, WN, WK, GS, ST, SUMS, SETS, PAIR>), dim3(grid), dim3(S::NT), 0, st, (const uint8_t*)w,
                       (const half2_t*)zs, (const half_t*)x, (half_t*)y, M, N, K, mt, tiles, nfull, ksplit, epi,
                       ws ? (float*)((char*)ws + RING_COUNTER_BYTES) : nullptr, (unsigned*)ws, (const uint8_t*)w2,
                       (const half2_t*)zs2, (half_t*)u);
    return hipGetLastError();
}

// What a shape costs, in us: a workgroup takes `step0 + step1 * a` per stage of K and `fixed` besides (first loads, sums,
// stores), a = the share of the 256 CUs that its round keeps busy (memory and clock are shared), and no less per stage than the
// rows that the eight XCDs ask for take at 6.5 TB/s (consecutive tiles of a column are one XCD's, so that narrow weights at
// thousands of tokens read the activations once for every column); a K split adds the
// exchange of the partial tiles, `ex0 + ex1 * parts + exmb` per MB of them, and every round of 256 after the first `round`.
// One workgroup fills a CU.  Least-squares
// fits: tiles of 32 rows to 9000 timings of 18 weights (3072 x 1024 .. 28672 x 8192) x 23 token counts (12 .. 4096), the
// others then adjusted for the choice alone on all shapes and splits of 13500 weights (512 .. 20480 rows, K 768 .. 16384) with
// a token count each (17 .. 4096): on 1350 that were kept back 0.25 % above the best in the geometric mean, 1.1 % of them by
// more than 5 %, at worst 11 % (with constants fitted to 26 weights from 1536 rows up, and without the rate, 0.5 %, 3 % and
// 30 %: 3272 tokens x 1024x1152 20.2 us where they take 14.5).
struct RingTile {
    int bm, bn, ks;
    float fixed, step0, step1, ex0, ex1, exmb, round;
};
static const RingTile kRingTiles[] = {
    {32, 64, 512, 1.723f, 0.829f, 0.160f, 0.301f, 0.226f, 0.861f, 0.f},
    {32, 128, 256, 1.498f, 0.754f, 0.096f, 0.448f, 0.304f, 0.649f, 0.f},
    {64, 128, 256, 2.774f, 0.734f, 0.380f, 0.702f, 0.545f, 0.299f, 0.747f},
    {96, 128, 128, 2.255f, 0.472f, 0.337f, 1.219f, 0.605f, 0.272f, 2.082f},
    {64, 256, 128, 2.615f, 0.799f, 0.277f, 1.381f, 0.949f, 0.188f, 1.770f},
    {96, 256, 128, 4.013f, 0.701f, 0.594f, 1.226f, 1.557f, 0.188f, 1.946f},
    {128, 128, 128, 2.247f, 0.548f, 0.340f, 0.853f, 1.153f, 0.353f, 3.134f},
    {128, 256, 128, 4.966f, 0.881f, 0.734f, 2.088f, 1.086f, 0.201f, 2.056f},
    {256, 256, 64, 9.097f, 0.833f, 0.661f, 0.f, 0.f, 0.f, 1.343f},  // never split, see plan_ring
};
// The same with the scale on the sums (up to 64 tokens), where other constants hold: shapes 1..5, of which the fourth is
// not built for it; the second's at 17..32 tokens alone.  There its stages are faster with the zeros/scales of several at once
// (ring_sets), and where 0.706 for 0.754 changes the plan of random weights (256 .. 32768 rows, K 768 .. 16384) it takes 0.979 of
// the time in the geometric mean (12 of 1300, at worst 1.06); at fewer tokens most plans have them by the stage (with 0.706 there
// and sets 1.045 at 1..4 tokens, 1.025 at 5..16), at 33..64 the two constants are level (0.99 and 1.01 of 30 each).  Against the
// best of all shapes and splits of those 1300 (1..64 tokens, one weight or gate and up): 0.5 % in the geometric mean, 5 % of them
// more than 4.1 %.
static const RingTile kRingSumsTiles[] = {
    kRingTiles[0], {32, 128, 256, 1.498f, 0.706f, 0.096f, 0.448f, 0.304f, 0.649f, 0.f},
    {64, 128, 256, 2.615f, 0.896f, 0.244f, 0.211f, 0.515f, 0.409f, 0.f},
    kRingTiles[3], {64, 256, 128, 2.020f, 0.843f, 0.222f, 0.814f, 0.857f, 0.394f, 0.f},
};
static const RingTile& ring_tile(int s, int M, bool sums) {
    return sums && s < 5 && (s != 1 || (M > 16 && M <= 32)) ? kRingSumsTiles[s] : kRingTiles[s];
}
constexpr int RING_SHAPES = sizeof(kRingTiles) / sizeof(kRingTiles[0]);
#define X_(id, MI, NI, WM, WN, WK, ST)                                                                              \
    static_assert(id >= 1 && id <= RING_SHAPES, "a row of kRingTiles per shape");
SQ_RING_SHAPES(X_)
#undef X_

bool gemm_ring_applies(int M, int N, int K) {
    // operands are addressed with 32-bit byte offsets per lane
    return (long)M * K * 2 < (1L << 32) && (long)N * (K / 2) < (1L << 32) && (long)M * N < (1L << 36);
}

static size_t ring_bytes(const RingPlan& p, int M, int N) {
    if (p.ksplit <= 1) return 0;
    const RingTile& t = kRingTiles[p.shape - 1];
    const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    return RING_COUNTER_BYTES + (size_t)(tiles - p.nfull) * p.ksplit * t.bm * t.bn * sizeof(float);
}

// The cheapest shape and K split whose partial tiles fit `ws_bytes`.  Where the tiles come in full rounds of 256 and a
// rest, only the rest splits K.
static RingPlan plan_ring(int M, int N, int K, size_t ws_bytes, bool sums) {
    RingPlan best{1, 0, 1};
    float best_us = 3.4e38f;
    const int rows32 = (M + 31) / 32 * 32;
    for (int s = 0; s < RING_SHAPES; s++) {
        const RingTile& t = ring_tile(s, M, sums);
        const int mt = (M + t.bm - 1) / t.bm;
        // a third of the matrix work would be padding; up to 64 rows the others are the ones with the scale on the sums
        if (t.bm > 64 && (M <= 64 || mt * t.bm * 2 > rows32 * 3)) continue;
        const long tiles = (long)mt * ((N + t.bn - 1) / t.bn);
        const int stages = (K + t.ks - 1) / t.ks;
        const int full = (int)(tiles >> 8), rest = (int)(tiles & 255);
        auto step = [&](int wgs) {  // of a round of wgs workgroups
            const float rows = 8.f * ((wgs + 7) / 8 < mt ? (wgs + 7) / 8 : mt) * (t.bm < M ? t.bm : M);
            const float busy = t.step0 + t.step1 * wgs * (1.f / 256), read = rows * t.ks * (2e-6f / 6.5f);
            return busy > read ? busy : read;
        };
        const float full_step = step(256);
        const float one = stages * full_step + t.fixed;
        const float base = 2.f + full * one;
        auto consider = [&](float us, int rounds, int nfull, int ks) {
            if (rounds > 1) us += (rounds - 1) * t.round;
            if (us >= best_us) return;
            const RingPlan p{s + 1, nfull, ks};
            if (ks > 1 && ring_bytes(p, M, N) > ws_bytes) return;
            best_us = us;
            best = p;
        };
        consider(base + (rest ? stages * step(rest) + t.fixed : 0.f), full + (rest != 0), 0, 1);
        // (256 x 256 tiles split over K were behind smaller tiles wherever they were timed: partial tiles of 256 KB)
        if (ws_bytes == 0 || rest == 0 || t.bm == 256) continue;
        static const int splits[5] = {2, 3, 4, 6, 8};
        for (int ks : splits) {
            const long w = (long)rest * ks;
            if (ks > stages || w > RING_PARTS_MAX) break;
            const int st = (stages + ks - 1) / ks;
            const float ex = t.ex0 + t.ex1 * ks + t.exmb * (4e-6f * w * t.bm * t.bn);
            const int r = (int)(w >> 8), last = (int)(w & 255);
            consider(base + r * (st * full_step + t.fixed) + (last ? st * step(last) + t.fixed : 0.f) + ex, full + r + (last != 0),
                     full * 256, ks);
        }
    }
    return best;
}

size_t gemm_ring_workspace_bytes(int M, int N, int K) {
    if (!gemm_ring_applies(M, N, K)) return 0;
    const size_t b = ring_bytes(plan_ring(M, N, K, (size_t)64 << 20, false), M, N);
    const size_t sums = M <= 64 ? ring_bytes(plan_ring(M, N, K, (size_t)64 << 20, true), M, N) : 0;
    return b > sums ? b : sums;
}

// With the scale on the sums and tiles of 128 or 256 columns: zeros/scales of several stages at once (SETS of the kernel), or a
// stage's with its other operands.  `k`: columns of K of a workgroup.  A set is a burst in front of its first stage, which a K of
// one or two sets shows, and so does a loop that waits for latency; it saves lines, which counts where the rows of a tile ask
// for many, and more of them where a row has an odd number of pairs, so that a stage's two are no aligned 8 bytes.  Time with
// sets / without, 32 x 128 tiles, 16..256 workgroups, geometric means (an even number of groups; an odd one has 1 more):
//   k        512  1024  1536  2048  2560  3072  4096  5120  6144  8192 12288     an odd number of groups
//   2 rows  1.04  1.06  1.06  1.07  1.07  1.07  1.08  1.01  1.03  1.03  1.03     1.06 1.07 1.03 1.05 1.06 1.03 1.00 1.00 0.97 0.97 0.94
//   8       1.05  1.07  1.07  1.06  1.06  1.06  1.05  0.99  1.00  1.01  1.01     1.05 1.06 1.03 1.03 1.03 1.01 0.98 0.97 0.96 0.94 0.91
//   16      1.05  1.06  1.06  1.06  1.04  1.03  1.02  0.95  0.98  0.98  0.96     1.06 1.06 1.03 1.00 1.00 0.98 0.96 0.95 0.94 0.92 0.88
//   24      1.04  1.07  1.05  1.04  1.02  1.01  0.99  0.93  0.94  0.95  0.92     1.05 1.06 1.02 1.00 0.98 0.97 0.94 0.91 0.91 0.90 0.86
//   32      1.04  1.05  1.04  1.03  0.98  0.97  0.96  0.89  0.92  0.92  0.88     1.04 1.04 1.00 0.98 0.96 0.95 0.91 0.91 0.90 0.88 0.84
// 64 x 128 tiles by the share of rows that are there are within 0.03 of that, 64 x 256 tiles lose less and gain up to twice as
// much (64 rows of an odd number of groups 0.97 0.96 0.97 0.97 0.95 0.92 0.87 0.81 0.81 0.78 0.77).  Over 1050 random weights,
// token counts and K splits, one weight and gate and up: by this rule 0.965, 0.978 and 0.905 of the time without for the three
// tiles, always with sets 0.972, 0.979 and 0.905, the better one each time 0.961, 0.973 and 0.903.
static bool ring_sets(const RingTile& t, int M, int K, int parts) {
    const int k = K / parts;
    const long rows = (long)(M + t.bm - 1) / t.bm * t.bm;
    if (K / 128 % 2) return k > (4L * M <= rows ? 4096 : 2048);
    return 2L * M > rows && k > (4L * M <= 3 * rows ? 4096 : 2048);
}

// tune = 0 for the cost model's choice, else shape id | 0x10: only the tiles of the last, part-filled round of 256
// workgroups split K | K split << 8; RING_SUMS: the scale on the sums (also with the model's choice; group size 128, tiles
// of 32 and 64 rows).  hipErrorInvalidValue: not applicable (or the workspace is missing or too small).
// PAIR: N outputs of two weights, planned as 2 N columns.
template <bool PAIR>
static hipError_t launch_ring(const void* x, const void* w, const void* zs, const void* w2, const void* zs2, void* y, void* u, void* ws,
                              size_t ws_bytes, int M, int N, int K, int g, int tune, Epilogue epi, hipStream_t st) {
    const int cols = PAIR ? 2 * N : N;
    if ((PAIR && N > (1 << 29)) || !gemm_ring_applies(M, cols, K)) return hipErrorInvalidValue;
    RingPlan p{tune & 0xF, 0, (tune >> 8) & 0xFF};
    if (p.shape == 0) {
        p = plan_ring(M, cols, K, ws ? ws_bytes : 0, (tune & RING_SUMS) != 0);
    } else {
        if (p.shape > RING_SHAPES || p.ksplit > 8) return hipErrorInvalidValue;
        const RingTile& t = kRingTiles[p.shape - 1];
        const long tiles = (long)((M + t.bm - 1) / t.bm) * ((cols + t.bn - 1) / t.bn);
        if (tiles > (1L << 24)) return hipErrorInvalidValue;
        if (p.ksplit < 1) p.ksplit = 1;
        if (tune & 0x10) p.nfull = (int)(tiles / 256 * 256);
        if (p.ksplit > 1) {
            const size_t need = ring_bytes(p, M, cols);
            if (tiles == p.nfull || tiles - p.nfull > (long)(RING_COUNTER_BYTES / 4) || p.ksplit > (K + t.ks - 1) / t.ks ||
                need - RING_COUNTER_BYTES >= 0x7FFFFFFFu || !ws || ws_bytes < need)
                return hipErrorInvalidValue;
        }
    }
#define SQ_RING_LAUNCH(MI, NI, WM, WN, WK, GS, ST, SUMS, SETS) \
    launch_shape<MI, NI, WM, WN, WK, GS, ST, SUMS, SETS, PAIR>(x, w, zs, w2, zs2, y, u, M, N, K, p.nfull, p.ksplit, epi, ws, st)
    if (tune & RING_SUMS) {
        if (g != 128) return hipErrorInvalidValue;
        const bool sets = ring_sets(kRingTiles[p.shape - 1], M, K, p.nfull ? 1 : p.ksplit);
        switch (p.shape) {
#define X_(id, MI, NI, WM, WN, WK, ST)                                           \
    case id:                                                                     \
        return sets ? SQ_RING_LAUNCH(MI, NI, WM, WN, WK, 7, ST, true, (WK <= 4)) \
                    : SQ_RING_LAUNCH(MI, NI, WM, WN, WK, 7, ST, true, false);
            SQ_RING_LOW_SHAPES(X_)
#undef X_
        }
        return hipErrorInvalidValue;
    }
    switch (p.shape) {
#define X_(id, MI, NI, WM, WN, WK, ST)                                              \
    case id:                                                                        \
        if (g == 128) return SQ_RING_LAUNCH(MI, NI, WM, WN, WK, 7, ST, false, false);      \
        if (g == 64) return SQ_RING_LAUNCH(MI, NI, WM, WN, WK, 6, ST, false, false);       \
        return SQ_RING_LAUNCH(MI, NI, WM, WN, WK, 5, ST, false, false);
        SQ_RING_SHAPES(X_)
#undef X_
    }
#undef SQ_RING_LAUNCH
    return hipErrorInvalidValue;
}

hipError_t launch_gemm_ring(const void* x, const void* w, const void* zs, void* y, void* ws, size_t ws_bytes, int M, int N,
                            int K, int g, int tune, Epilogue epi, hipStream_t st) {
    return launch_ring<false>(x, w, zs, nullptr, nullptr, y, nullptr, ws, ws_bytes, M, N, K, g, tune, epi, st);
}

hipError_t launch_gemm_ring_pair(const void* x, const void* w_gate, const void* zs_gate, const void* w_up, const void* zs_up,
                                 void* y, void* up, void* ws, size_t ws_bytes, int M, int N, int K, int g, int tune, hipStream_t st) {
    return launch_ring<true>(x, w_gate, zs_gate, w_up, zs_up, y, up, ws, ws_bytes, M, N, K, g, tune, Epilogue{nullptr, nullptr, 0},
                             st);
}

}  // namespace sq
