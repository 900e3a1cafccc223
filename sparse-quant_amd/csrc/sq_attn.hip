// LUT block-sparse attention, prefill (fp16 in/out, fp32 softmax and accumulation).
// For query block i of head h only the key blocks lut[h][i][0..nnz) are visited
// (64 x 64 blocks; a LUT entry equal to its predecessor is padding and is skipped);
// inside a block an optional causal mask and the sequence-length mask apply.
// (replaces _sparse_attention_prefill_fwd_kernel, reference:
// sparse-attention/nvidia/playground/kernels/block_sparse_attention_lut.py:22-172, and
// sparse_attention_prefill_fwd_p, sparse-attention/muxi/playground/kernels/csrc/include/
// block_sparse_attention_lut.cuh:30-236)
//
// Mapping.  A workgroup of two waves owns one 64-row query block of one (batch, head) and goes through the visited
// blocks in steps of 32 keys; a wave owns 32 queries.  Both products are computed transposed with
// v_mfma_f32_32x32x16_f16 so that a lane always owns ONE query (column l % 32):
//   S^T = K Q^T : A = K tile (row = key, 128-bit LDS reads), B = Q^T (registers, as given);
//                 D: lane holds keys 8 (v / 4) + 4 (l / 32) + v % 4 of the 32.  The scores are scaled in fp32.
//   softmax     : over a lane's 16 values and the lane pair {l, l ^ 32}; the reference maximum of a query moves
//                 lazily (only when a score exceeds it by more than 2^8), the row sum stays split over the lane
//                 pair until the end: in the common case nothing is exchanged or rescaled.
//   O^T = V^T P^T: B = P^T is what the lane already holds, keys in that order; A = V^T by transposing 64-bit LDS
//                 reads (ds_read_b64_tr_b16: four keys of one column per lane) of the V tile as it lies in memory.
// K and V tiles go global -> LDS by direct loads, one step ahead, and are never touched by vector instructions on
// the way; the 16-byte chunks of a row are permuted by the lane that requests them so that the operand reads of
// neighbouring rows fall on different banks.  The visited blocks of a row come from the table 64 entries at a time,
// in one load: which of them are padding is a ballot, so no step waits for the table.
//
// What bounds it.  Per step of D = 128 a wave needs 512 cycles of its matrix pipe and about 600 of vector issue (16
// exponentials at a quarter of the rate among them); the operand reads take 512 LDS cycles per 64 x 64 block (32
// queries per wave: each K and V value is read twice; with 16 per wave it is four times, and 1024 cycles were the
// bound).  Four workgroups of 32 KB share a CU, two waves per SIMD, each at its own point of the step, so that one's
// softmax and first loads run beside another's products.  Where there are too few workgroups for that, four waves take
// steps of 64 keys and split them (SPLIT_WGS below).
// Measured (us; before: 16 queries per wave, K through registers, V transposed by vector instructions):
//   32 heads x 4096 x 128, causal, 26 % of the blocks   125 -> 85 (matrix pipes busy 0.41 of the cycles)
//   8 x 16 heads x 4096 x 64, 25 %                       225 -> 181
//   8 x 32 heads x 512 x 128, causal, 26 %               38.5 -> 34 (134 MB to move: 22 at the rate of a copy)
//   8 x 16 heads x 512 x 64, 25 %                        10.2 -> 8.1
//   16 heads x 1674 x 128, causal, 42 %                  26.6 -> 17.3;   12 heads x 128 x 64  4.2 -> 4.2
// Outputs and cache rows are nontemporal stores: they are not read here again, and as ordinary ones they push K and V
// rows out of the L2s (5 x 32 heads x 365 x 128 15.1 -> 13.8, 8 x 16 x 512 x 64 8.8 -> 8.1).
// Of a small call's time 0.5 us was the fetch of the kernel's arguments in front of the first request: those that the
// request of the table needs are scalars now, which arrive with the wave.
// A model's prompt reads q, k and v where the fused projection left them and stores the cache rows and a [batch, row,
// hidden] output: the element-wise copies around the kernel cost three times its own time (8 prompts of 512 tokens, 32
// heads of 128, per layer: six copies of 21 us and 35 -> 42 in all; without a table, against torch's attention and its
// copies, 157 -> 59).
#include "sq_common.h"
#include "sq_kernels.h"

#include <type_traits>

namespace sq {

namespace {

// What a workgroup needs after its first request (of the table) is out.
struct LutAttnArgs {
    half_t* o;
    half_t* kc;       // caches that receive the K and V rows, or null
    half_t* vc;
    LutAttnStrides st;
    float qk_scale;  // sm_scale * log2(e)
    float lazy;      // log2 of how far a score may exceed the reference maximum
};

// Chunk permutations inside a tile row of D halves (D / 8 chunks of 16 bytes).
// K is read 128 bits wide by 32 lanes = rows at one chunk: 16 consecutive rows (256 bytes of LDS banks) must differ.
template <int D>
__device__ __forceinline__ int k_swz(int row) {
    return D == 128 ? (row & 15) : ((row & 7) ^ ((row >> 3) & 1));
}
// V is read 64 bytes of a row by 8 lanes, four consecutive rows by a transposing read: the rows' 64-byte pieces must differ.
template <int D>
__device__ __forceinline__ int v_swz(int row) {
    return D == 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1);
}

typedef short short4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ short4_t lds_read_tr(const uint8_t* p) {
    typedef __attribute__((address_space(3))) short4_t* lp;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(p));
}

// KG = 1: two waves, steps of 32 keys.  KG = 2: four waves, steps of 64 keys, wave (qg, kg) on keys 32 kg .. + 31 of each
// with a softmax state of its own; the two states of a query meet at the end.
// WPS: waves per SIMD the registers are limited to.
template <int D, int KG, int WPS>
__global__ __launch_bounds__(128 * KG, WPS) void lut_attn_kernel(
    const void* __restrict__ lut, int lut_is_64, int nblk, int nnz, int nvisit, int H, int S, int causal, int total_wg,
    const half_t* __restrict__ q, const half_t* __restrict__ k, const half_t* __restrict__ v, LutAttnArgs a) {
    // (the scalars and q, k, v arrive in registers with the wave; a structure has to be fetched)
    constexpr int ROW = D * 2;              // bytes of a tile row
    constexpr int STEP = 32 * KG;           // keys of a step
    constexpr int TILE = STEP * ROW;        // K or V of one step
    constexpr int SB = 2 * TILE;            // a stage: K tile, V tile
    constexpr int NK = D / 16;              // matrix steps of S^T
    constexpr int DT = D / 32;              // 32-row tiles of O^T
    constexpr int NL = 16 * ROW / 1024;     // direct loads per wave, operand and stage
    constexpr int RPL = 1024 / ROW;         // tile rows per load
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * SB];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31;
    const int lc = lane >> 5;
    const int qg = wave / KG;
    const int kg = wave % KG;
    // Workgroups are handed to the eight XCDs round-robin by their linear id, and every XCD has its own L2.
    // The id is therefore re-read as (XCD, slot): XCD x works through the x-th eighth of the (head, query block)
    // list, so that all query blocks of a head, which visit the same K and V rows, share one L2
    // instead of pulling those rows into all eight.  Causal: the long rows first.
    const int per_xcd = (total_wg + 7) >> 3;
    const int work = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (work >= total_wg) return;
    const int zh = work / nblk;
    const int qr = work - zh * nblk;
    const int qb = causal ? nblk - 1 - qr : qr;
    const int h = zh % H;
    const int z = zh / H;
    const half_t* kz = k + z * a.st.kv[0] + h * a.st.kv[1];
    const half_t* vz = v + z * a.st.kv[0] + h * a.st.kv[1];
    const int kv_row = (int)a.st.kv[2] * 2;  // bytes
    const int m = qb * 64 + 32 * qg + ln;  // this lane's query

    // The visited blocks, 64 table entries at a time: lane j holds entry j, `todo` has a bit for each that is visited.
    const long lut_row = ((long)h * nblk + qb) * nnz;
    const int entries = lut ? nvisit : (causal ? qb + 1 : nblk);
    int entry = 0, jbase = 0, last = -1;
    uint64_t todo = 0;
    auto table = [&](int j) {
        int blk = -1;
        if (j < entries) {
            blk = j;
            if (lut) blk = lut_is_64 ? (int)((const long long*)lut)[lut_row + j] : ((const int*)lut)[lut_row + j];
        }
        return blk;
    };
    auto take = [&](int blk) {
        const int up = __shfl_up(blk, 1);
        const int prev = lane == 0 ? last : up;
        todo = __builtin_amdgcn_ballot_w64(blk != prev && blk >= 0 && (long)blk * 64 < S);
        entry = blk;
        last = __builtin_amdgcn_readlane(blk, 63);
        jbase += 64;
    };
    auto next_block = [&]() {  // its first key, or -1
        while (todo == 0) {
            if (jbase >= entries) return -1;
            take(table(jbase + lane));
        }
        const int j = __builtin_ctzll(todo);
        todo &= todo - 1;
        return __builtin_amdgcn_readlane(entry, j) * 64;
    };
    const int first = table(lane);  // requested ahead of the queries

    half8_t qf[NK];
    {
        const half_t* qp = q + z * a.st.q[0] + h * a.st.q[1] + imin(m, S - 1) * a.st.q[2] + 8 * lc;
#pragma unroll
        for (int s = 0; s < NK; s++) qf[s] = *(const half8_t*)(qp + 16 * s);
    }

    take(first);
    int n0 = next_block();

    // Byte offsets of this wave's loads inside a step; load j covers tile rows RPL * (NL * wave + j) .. + RPL - 1.
    const int lrow = lane / (D / 8);
    const int lchunk = lane % (D / 8);
    auto lane_offset = [&](int j, int row_max, bool is_v) {
        const int row = RPL * (NL * wave + j) + lrow;
        const int c = lchunk ^ (is_v ? v_swz<D>(row) : k_swz<D>(row));
        return (uint32_t)(imin(row, row_max) * kv_row + c * 16);
    };
    uint32_t koff[NL], voff[NL];
#pragma unroll
    for (int j = 0; j < NL; j++) {
        koff[j] = lane_offset(j, STEP - 1, false);
        voff[j] = lane_offset(j, STEP - 1, true);
    }
    auto issue = [&](int n, int slot) {
        const uint8_t* kb = (const uint8_t*)(kz + n * a.st.kv[2]);
        const uint8_t* vb = (const uint8_t*)(vz + n * a.st.kv[2]);
        const uint32_t l0 = lds0 + slot * SB + wave * (NL * 1024);
        if (n + STEP <= S) {
#pragma unroll
            for (int j = 0; j < NL; j++) load_to_lds_x4(kb, koff[j], l0 + j * 1024);
#pragma unroll
            for (int j = 0; j < NL; j++) load_to_lds_x4(vb, voff[j], l0 + TILE + j * 1024);
        } else {  // rows past the end re-read the last one (their scores are masked)
#pragma unroll
            for (int j = 0; j < NL; j++) load_to_lds_x4(kb, lane_offset(j, S - 1 - n, false), l0 + j * 1024);
#pragma unroll
            for (int j = 0; j < NL; j++) load_to_lds_x4(vb, lane_offset(j, S - 1 - n, true), l0 + TILE + j * 1024);
        }
    };
    if (n0 >= 0) issue(n0, 0);

    // LDS byte offsets of the operand reads.
    int kread[NK], vread[DT];
#pragma unroll
    for (int s = 0; s < NK; s++) kread[s] = (32 * kg + ln) * ROW + (((2 * s + lc) ^ k_swz<D>(ln)) * 16);
    {
        const int key = 4 * lc + ((lane & 15) >> 2);  // + 32 kg + 16 s + 8 i, which leave v_swz unchanged
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
            vread[dt] = TILE + (32 * kg + key) * ROW + (((4 * dt + 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1)) ^ v_swz<D>(key)) * 16) +
                        8 * (lane & 1);
    }

    // Reference maximum of the query (0 while unset), the score above it at which it moves (any score while unset), and
    // this lane's share of the row sum.
    const float lazy = a.lazy;
    float ref = 0.f, limit = -INFINITY, l_i = 0.f;
    float16_t acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[dt][v] = 0.f;

    // Step n from slot SLOT; `next` (or -1) is requested into the other one.
    auto visit = [&](int n, auto slot_, int next) {
        constexpr int SLOT = decltype(slot_)::value;
        const uint8_t* l = lds + SLOT * SB;
        float16_t st;
#pragma unroll
        for (int v = 0; v < 16; v++) st[v] = 0.f;
        // All K operands are requested at once, and all V operands ahead of the softmax: a wave has one other wave on its
        // SIMD to hide LDS latency behind, which is not enough for a read per product.
        half8_t kf[NK];
#pragma unroll
        for (int s = 0; s < NK; s++) kf[s] = *(const half8_t*)(l + kread[s]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (KG == 2) __builtin_amdgcn_s_setprio(0);
        // The products of S^T are a chain, and requests that go out one by one between them do not wait for the address unit
        // (together with the counted waits of `landed`: 16 heads x 1674 x 128 19.1 -> 18.6 us on one box, 18.9 -> 18.0 on another).
        // With two waves per step another workgroup's waves fill that time (32 heads x 4096 x 128 86.9 -> 86.7).
        if (KG == 2 && next >= 0 && next + STEP <= S) {
            const uint8_t* kb = (const uint8_t*)(kz + next * a.st.kv[2]);
            const uint8_t* vb = (const uint8_t*)(vz + next * a.st.kv[2]);
            const uint32_t l0 = lds0 + (1 - SLOT) * SB + wave * (NL * 1024);
#pragma unroll
            for (int s = 0; s < NK; s++) {
                st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[s], qf[s], st, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = s * 2 * NL / NK; j < (s + 1) * 2 * NL / NK; j++) {
                    if (j < NL)
                        load_to_lds_x4(kb, koff[j], l0 + j * 1024);
                    else
                        load_to_lds_x4(vb, voff[j - NL], l0 + TILE + (j - NL) * 1024);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            if (next >= 0) issue(next, 1 - SLOT);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < NK; s++) st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[s], qf[s], st, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        short4_t vf[2][DT][2];
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int i = 0; i < 2; i++) vf[s][dt][i] = lds_read_tr(l + vread[dt] + (16 * s + 8 * i) * ROW);
        __builtin_amdgcn_sched_barrier(0);
        // (the four waves of a step wait for each other: the one in its softmax goes first.  By itself, before the requests
        // went between the products: 16 heads x 1674 x 128 17.8 -> 17.2 us, 2 x 16 x 567 x 128 8.6 -> 8.4; with two waves per step
        // it changes nothing)
        if constexpr (KG == 2) __builtin_amdgcn_s_setprio(1);
        // scores relative to the reference maximum, in units of log2
#pragma unroll
        for (int v = 0; v < 16; v++) st[v] = __builtin_fmaf(st[v], a.qk_scale, -ref);
        // Masks (only where the step touches the end of the sequence or the causal diagonal; the test is uniform).
        const int nk = n + 32 * kg;
        if (nk + 32 > S || (causal && nk + 31 > qb * 64 + 32 * qg)) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int key = nk + 8 * (v >> 2) + 4 * lc + (v & 3);
                const bool keep = (key < S) && (!causal || key <= m);
                st[v] = keep ? st[v] : -INFINITY;
            }
        }
        // The reference maximum of a query moves only when a score exceeds it by more than 2^lazy (or when it is still
        // unset): until then p = exp2(score) stays below 2^lazy, well inside fp16, the final O = acc / l does not depend
        // on the reference, and neither the accumulators nor the scores need rescaling.  The test is made per lane and
        // voted over the wave; the maximum over a query's two lanes is formed only when it is needed.
        float mx = -INFINITY;
#pragma unroll
        for (int v = 0; v < 16; v++) mx = fmaxf(mx, st[v]);
        if (__builtin_amdgcn_ballot_w64(mx > limit) != 0) {
            const float mq = fmaxf(mx, __shfl_xor(mx, 32));
            const bool upd = mq > limit;
            const float delta = upd ? mq : 0.f;
            // a query without a reference so far has l = 0 and acc = 0: nothing to rescale
            const float alpha = (upd && limit != -INFINITY) ? __builtin_amdgcn_exp2f(-delta) : 1.f;
            ref += delta;
            limit = upd ? lazy : limit;
            l_i *= alpha;
#pragma unroll
            for (int v = 0; v < 16; v++) st[v] -= delta;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[dt][v] *= alpha;
        }
        // p = exp2(score) (bare v_exp_f32: exp2(-inf) = 0 for masked entries), rounded to fp16 for the second product
        // like the reference; the lane's share of the row sum is taken from the rounded pairs with one dot instruction
        // per pair and stays in the lane until the end.
        half8_t pk[2];
        float rs = 0.f;
#pragma unroll
        for (int v = 0; v < 16; v += 2) {
            const half2_t pp = {(half_t)__builtin_amdgcn_exp2f(st[v]), (half_t)__builtin_amdgcn_exp2f(st[v + 1])};
            rs = __builtin_amdgcn_fdot2(pp, (half2_t){(half_t)1.f, (half_t)1.f}, rs, false);
            pk[v >> 3][v & 7] = pp.x;
            pk[v >> 3][(v & 7) + 1] = pp.y;
        }
        l_i += rs;
        if constexpr (KG == 2) __builtin_amdgcn_s_setprio(0);
        // O^T += V^T P^T
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
                const u32x2_t lo2 = bit_cast<u32x2_t>(vf[s][dt][0]), hi2 = bit_cast<u32x2_t>(vf[s][dt][1]);
                const u32x4_t vt = {lo2.x, lo2.y, hi2.x, hi2.y};
                acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bit_cast<half8_t>(vt), pk[s], acc[dt], 0, 0, 0);
            }
    };

    // One barrier per step: behind it this step's tiles have landed for every wave and nobody reads the other slot any
    // more, which the next step's loads may then fill.
    auto landed = []() {
        // (the same wait where the compiler sees it, so that the step's waits for LDS stay counted: with two waves per step
        // no difference)
        if constexpr (KG == 2) __builtin_amdgcn_s_waitcnt(0x0070);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    // The query operands are waited for here, together with the first tiles: left to the loop, the compiler's wait for
    // them would sit at the first product and drain the direct loads, which it cannot count, on every iteration.
#pragma unroll
    for (int s = 0; s < NK; s++) {
        u32x4_t t = bit_cast<u32x4_t>(qf[s]);
        asm volatile("" : "+v"(t));
        qf[s] = bit_cast<half8_t>(t);
    }
    if constexpr (KG == 1) {
        while (n0 >= 0) {
            const int n1 = next_block();
            const bool whole = n0 + 32 < S;  // the block has a second half
            landed();
            visit(n0, std::integral_constant<int, 0>{}, whole ? n0 + 32 : -1);
            landed();
            if (whole)
                visit(n0 + 32, std::integral_constant<int, 1>{}, n1);
            else if (n1 >= 0)
                issue(n1, 0);
            n0 = n1;
        }
    } else {
        while (n0 >= 0) {
            const int n1 = next_block();
            landed();
            visit(n0, std::integral_constant<int, 0>{}, n1);
            if (n1 < 0) break;
            n0 = next_block();
            landed();
            visit(n1, std::integral_constant<int, 1>{}, n0);
        }
    }

    // The row sum of a query is split over its two lanes.  A query row without any visible key has l = 0 and acc = 0:
    // 0 * inf = NaN, which is also what the reference's running sums produce for such a row.
    // The 32 x D outputs of a query group leave through LDS (16-byte chunks permuted like K's) as whole rows: a lane
    // holds four columns at a time, and 8-byte stores would cost the L2 eight times the write requests.
    l_i += __shfl_xor(l_i, 32);
    __syncthreads();
    uint8_t* out = lds + qg * (32 * ROW);
    auto park = [&](int dt, int i, half4_t o) {
        *(half4_t*)(out + ln * ROW + (((4 * dt + i) ^ k_swz<D>(ln)) * 16) + 8 * lc) = o;
    };
    if constexpr (KG == 1) {
        const float inv = 1.f / l_i;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                half4_t o;
#pragma unroll
                for (int j = 0; j < 4; j++) o[j] = (half_t)(acc[dt][4 * i + j] * inv);
                park(dt, i, o);
            }
        __builtin_amdgcn_wave_barrier();
    } else {
        // Each wave hands half of its output columns to the other key half's wave, with its reference maximum and row
        // sum, and finishes the others.
        constexpr int HALF = DT / 2;
        float4_t* red = reinterpret_cast<float4_t*>(lds + 64 * ROW);                // [wave][HALF][4][64]
        float2* stat = reinterpret_cast<float2*>(lds + 64 * ROW + 4 * HALF * 4096);  // [wave][64]
        static_assert(64 * ROW + 4 * HALF * 4096 + 4 * 512 <= 2 * SB, "fits");
        const float m_i = limit == -INFINITY ? -INFINITY : ref;
#pragma unroll
        for (int d = 0; d < HALF; d++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float4_t t;
#pragma unroll
                for (int j = 0; j < 4; j++) t[j] = kg == 0 ? acc[HALF + d][4 * i + j] : acc[d][4 * i + j];
                red[((wave * HALF + d) * 4 + i) * 64 + lane] = t;
            }
        stat[wave * 64 + lane] = make_float2(m_i, l_i);
        __syncthreads();
        const int peer = wave ^ 1;
        const float2 ps = stat[peer * 64 + lane];
        const float mm = fmaxf(m_i, ps.x);
        const float f_own = (m_i == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m_i - mm);
        const float f_peer = (ps.x == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(ps.x - mm);
        const float inv = 1.f / (l_i * f_own + ps.y * f_peer);
        const float w_own = f_own * inv, w_peer = f_peer * inv;
#pragma unroll
        for (int d = 0; d < HALF; d++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float4_t t = red[((peer * HALF + d) * 4 + i) * 64 + lane];
                half4_t o;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float mine = kg == 0 ? acc[d][4 * i + j] : acc[HALF + d][4 * i + j];
                    o[j] = (half_t)(mine * w_own + t[j] * w_peer);
                }
                park(d + (kg ? HALF : 0), i, o);
            }
        __syncthreads();
    }
    constexpr int PASSES = 32 * ROW / 1024 / KG;  // 1 KB of whole rows per wave and pass
#pragma unroll
    for (int j = 0; j < PASSES; j++) {
        const int row = RPL * (PASSES * kg + j) + lrow;
        const u32x4_t t = *(const u32x4_t*)(out + row * ROW + ((lchunk ^ k_swz<D>(row)) * 16));
        const int mr = qb * 64 + 32 * qg + row;
        if (mr < S)
            __builtin_nontemporal_store(t, (u32x4_t*)(a.o + z * a.st.o[0] + h * a.st.o[1] + mr * a.st.o[2] + 8 * lchunk));
    }
    // The workgroup's own 64 rows of K and V go to the caches (their lines are in this XCD's L2).
    if (a.kc) {
        half_t* kcz = a.kc + z * a.st.c[0] + h * a.st.c[1];
        half_t* vcz = a.vc + z * a.st.c[0] + h * a.st.c[1];
#pragma unroll
        for (int j = 0; j < PASSES; j++) {
            const int mr = qb * 64 + 32 * qg + RPL * (PASSES * kg + j) + lrow;
            if (mr < S) {
                const u32x4_t kr = *(const u32x4_t*)(kz + mr * a.st.kv[2] + 8 * lchunk);
                const u32x4_t vr = *(const u32x4_t*)(vz + mr * a.st.kv[2] + 8 * lchunk);
                __builtin_nontemporal_store(kr, (u32x4_t*)(kcz + mr * a.st.c[2] + 8 * lchunk));
                __builtin_nontemporal_store(vr, (u32x4_t*)(vcz + mr * a.st.c[2] + 8 * lchunk));
            }
        }
    }
}

// Workgroups up to which the four-wave form is launched: two of them per CU, so that all are resident at once and what
// counts is how soon each is through its own blocks.  Two against four waves (us): 16 heads x 1674 x 128, 432 workgroups,
// 22.3 / 17.3; 2 x 12 x 1138 x 64, 432, 9.5 / 7.8; 12 x 128 x 64, 24, 4.7 / 4.2; 5 x 32 x 145 x 64 with one block per
// row, 480, 5.3 / 5.4; beyond: 6 x 32 x 159 x 128, 576, 8.7 / 11.2; 2 x 16 x 1669 x 128, 864, 19.6 / 23.2.
constexpr int SPLIT_WGS = 512;
// D = 64 takes 132 registers left to itself: three waves per SIMD, 1536 workgroups on the chip at once.  Four (128
// registers, 2048 workgroups) are a little slower where three hold the whole grid and save the second round beyond (us,
// three / four): 8 x 16 heads x 640, 1280 workgroups, 9.7 / 10.0; 4 x 32 x 768, 1536, 17.8 / 19.5; 8 x 16 x 1024, 2048,
// 22.4 / 19.1; 4 x 16 x 2048, 2048, 32.5 / 28.6; 8 x 16 x 1536, 3072, 39.1 / 39.2; 8 x 16 x 4096, 8192, 188 / 181.
constexpr int THREE_WAVE_WGS = 1536;

}  // namespace

hipError_t launch_lut_attention(const void* q, const void* k, const void* v, void* o, void* k_cache, void* v_cache,
                                const void* lut, int lut_elem_bytes, int Z, int H, int S, int D, int nnz,
                                const LutAttnStrides& strides, float sm_scale, int causal, hipStream_t st) {
    LutAttnArgs a;
    a.o = (half_t*)o;
    a.kc = (half_t*)k_cache;
    a.vc = (half_t*)v_cache;
    a.st = strides;
    a.qk_scale = sm_scale * 1.44269504f;
    // Without a table the reference is the running maximum itself, whose probability 1 is exact in fp16: the error of a
    // dense softmax with it (2.43e-4 of the result at 512 keys, 2.51e-4 with the lazy one) at the price of more rescaling
    // (8 x 32 heads x 512 x 128: 51 -> 59 us).
    a.lazy = lut ? 8.f : 0.f;
    const int nblk = (S + 63) / 64;
    const int nvisit = lut && nnz < nblk ? nnz : nblk;  // the reference clamps NNZ to ceil(S / 64) as well (the row pitch stays nnz)
    const int total_wg = nblk * Z * H;
    const dim3 grid(((total_wg + 7) / 8) * 8);
    const bool split = total_wg <= SPLIT_WGS;
#define SQ_ATTN_LAUNCH(D_, KG_, WPS_)                                                                                    \
    hipLaunchKernelGGL((lut_attn_kernel<D_, KG_, WPS_>), grid, dim3(128 * KG_), 0, st, lut, (int)(lut_elem_bytes == 8), nblk, \
                       nnz, nvisit, H, S, causal, total_wg, (const half_t*)q, (const half_t*)k, (const half_t*)v, a)
    if (D == 64) {
        if (split) SQ_ATTN_LAUNCH(64, 2, 2);
        else if (total_wg <= THREE_WAVE_WGS) SQ_ATTN_LAUNCH(64, 1, 2);
        else SQ_ATTN_LAUNCH(64, 1, 4);
    } else {
        if (split) SQ_ATTN_LAUNCH(128, 2, 2);
        else SQ_ATTN_LAUNCH(128, 1, 2);
    }
#undef SQ_ATTN_LAUNCH
    return hipGetLastError();
}

}  // namespace sq
