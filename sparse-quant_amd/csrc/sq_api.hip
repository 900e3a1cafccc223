// C ABI of libsq_w4a16.so: argument validation and kernel dispatch.  Declarations
// and the contract of every entry point are in include/sq_w4a16.h.
#include "../../include/sq_w4a16.h"

#include <atomic>
#include <mutex>

#include "sq_kernels.h"

// Workspace of sq_w4a16_gemm_static_ws: device memory that belongs to the library, so that the
// call allocates nothing.  Every GPU the library runs on holds its own copy of the array until the
// process ends; the name below is only the host-side handle of the symbol, the device address is
// looked up once per device with hipGetSymbolAddress and that pointer is what the kernels get.
// It holds every plan of the ring kernel: within less, that kernel would split K otherwise than with a caller's workspace.
constexpr size_t SCRATCH_BYTES = sq::RING_WORKSPACE_MAX > SQ_STATIC_WS_BYTES ? sq::RING_WORKSPACE_MAX : SQ_STATIC_WS_BYTES;
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

namespace {

__global__ void zero_words_kernel(unsigned* p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

constexpr int MAX_DEVICES = 64;
void* g_scratch[MAX_DEVICES];
std::mutex g_scratch_mutex;

// Device address of `scratch` on the current device (null on failure).  The array needs no clearing: a
// file-scope __device__ array without an initialiser is zero when its code object is loaded, and every kernel
// leaves the counters at its start zero.
void* static_workspace() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
        g_scratch[dev] = p;
    }
    return g_scratch[dev];
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline int launch_code(hipError_t e) { return e == hipSuccess ? SQ_OK : SQ_ERR_LAUNCH; }
inline bool pow2(int v) { return v > 0 && (v & (v - 1)) == 0; }

// Shape rules shared by gemm and dequant.
int check_weight(int N, int K, int g, int layout) {
    if (layout != SQ_LAYOUT_L1 && layout != SQ_LAYOUT_L2) return SQ_ERR_BAD_LAYOUT;
    if (N <= 0 || K <= 0) return SQ_ERR_BAD_SHAPE;
    if (layout == SQ_LAYOUT_L1) {
        if (g != 32 && g != 64 && g != 128) return SQ_ERR_BAD_GROUP;
        if (N % 8 != 0 || K % 32 != 0 || K % g != 0) return SQ_ERR_BAD_SHAPE;
    } else {
        if (g != 128) return SQ_ERR_BAD_GROUP;
        if (N % 32 != 0 || K % 32 != 0 || K % g != 0) return SQ_ERR_BAD_SHAPE;
    }
    if ((long)N * (long)K > (1L << 40)) return SQ_ERR_BAD_SHAPE;
    return SQ_OK;
}

// One dispatcher behind every GEMM entry point.  `workspace` may be null: then the kernels
// that need one are not considered (and an explicit SQ_ALGO_SKINNY_WS is an error).
// Measured kernel choices (sq_w4a16_autotune): shape -> kernel word, consulted before the built-in rules.
// Entries are only ever appended (under the mutex); readers scan without it up to the published count.
struct TunedEntry {
    int M, N, K, g, has_ws, algo;
    float us;
};
constexpr int TUNED_MAX = 1024;
TunedEntry g_tuned[TUNED_MAX];
std::atomic<int> g_tuned_count{0};
std::mutex g_tuned_mutex;

inline bool full_workspace(const void* workspace, size_t workspace_bytes, int M, int N, int K) {
    return workspace && (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0 &&
           workspace_bytes >= sq_w4a16_workspace_bytes(M, N, K);
}

// Whether the decode kernels can split K through this workspace.
inline bool decode_workspace(const void* workspace, size_t workspace_bytes, int M, int N, int K) {
    return workspace && aligned16(workspace) && workspace_bytes >= sq::skinny2_workspace_bytes(M > 32 ? 32 : M, N, K) &&
           (N + 63) / 64 <= 16384;
}

int tuned_lookup(int M, int N, int K, int g, bool has_ws) {
    const int n = g_tuned_count.load(std::memory_order_acquire);
    for (int i = n - 1; i >= 0; i--) {  // the latest measurement of a shape wins
        const TunedEntry& e = g_tuned[i];
        if (e.M == M && e.N == N && e.K == K && e.g == g && e.has_ws == (int)has_ws) return e.algo;
    }
    return 0;
}

// The built-in kernel choice as a table: the first row whose token range contains M, whose `need` properties all
// hold and whose `forbid` properties all fail names the kernel.  Every row carries the measurement it rests on
// (MI355X, cold weights, OPT-6.7B / Llama-2-7B shapes, us per launch).  sq_w4a16_autotune overrides the table per
// shape with a measurement of that shape.
enum : unsigned {
    P_LARGE = 1u << 0,      // N * K >= 2^25 elements (fc1 / fc2 class)
    P_WS = 1u << 1,         // a workspace for the decode kernels' K split is at hand
    P_G128_64 = 1u << 2,    // group size 128 or 64
    P_K128 = 1u << 3,       // K a multiple of 128
    P_K_LE_4096 = 1u << 4,
    P_K_LE_8192 = 1u << 5,
    P_K_LE_32768 = 1u << 6,
    P_SMALL = 1u << 7,        // N * K <= 2^22 elements and K <= 1536
    P_OVER_16M = 1u << 8,     // N * K > 2^24 elements
    P_CHUNK_FILL = 1u << 9,   // the least K split of the streaming kernel fills 3/4 or more of a workgroup's 32 chunks
    P_RING = 1u << 10,        // the ring kernel can address the operands
    P_SMALL_K2048 = 1u << 11,   // N * K <= 2^22 elements and K <= 2048
    P_G64 = 1u << 13,           // group size 64
    // the streaming kernel's 64-row workgroups times K ranges come to 257..400 (336 with four K ranges: 42 tiles of 128 columns,
    // the last that the ring kernel's six parts of K keep in one round): a second round, part empty
    P_SPILL = 1u << 14,
    P_PARTS4 = 1u << 15,        // four K ranges of the streaming kernel or more
    P_PARTS5 = 1u << 16,        // five
    P_OVER_128 = 1u << 17,    // more than 128 of those workgroups
    P_FEW_OVER = 1u << 18,      // at most 160 of them, or K ranges filled less than 0.6: two K ranges either way
    P_SHORT_ROUNDS = 1u << 12,  // many rounds of 128 x 256 tiles over a short K (see builtin_choice)
    // what the streaming kernel needs of a K that it splits
    P_STREAM_SPLIT = P_G128_64 | P_K128 | P_WS | P_K_LE_32768,
};
struct ChoiceRule {
    int m_lo, m_hi;
    unsigned need, forbid;
    int kernel;
    const char* measured;
};
const ChoiceRule kChoiceRules[] = {
    // 5..16 tokens where a K range of the streaming kernel would leave its chunk slots part empty, and at group size 32
    {5, 16, P_LARGE | P_G128_64 | P_RING, P_CHUNK_FILL | P_K_LE_4096, SQ_ALGO_RING,
     "8 / 16 tokens: 15360x5120 13.9 vs 16.0 / 19.0 (streaming kernel), 13696x5120 13.4 vs 15.7 / 19.3"},
    // (in place of the streaming kernel alone: where that does not run, the GEMV keeps the scale in fp32 at 5..8 tokens and
    // group size 64, and without a workspace the ring kernel leaves most of the chip idle: 3136x5888 at 9 tokens 13.5 vs 8.3
    // (16-column kernel), 4672x6016 at 8 14.1 vs 10.7 (GEMV))
    {5, 8, P_OVER_16M | P_G64 | P_STREAM_SPLIT | P_OVER_128 | P_FEW_OVER | P_RING, P_CHUNK_FILL | P_K_LE_4096, SQ_ALGO_RING,
     "group size 64, 8 tokens: 4608x4608 9.3 vs 10.2 (streaming kernel), 5120x5120 10.3 vs 10.4, 5376x4608 0.92 of it, 4736x5376 at 5 "
     "0.95; but 3072x6016 1.16, 3008x5888 at 5 1.12, 5696x5888 at 6 1.06, 2432x8576 1.13; at group size 128 5120x5120 10.4 vs 9.9"},
    {9, 16, P_OVER_16M | P_G64 | P_STREAM_SPLIT | P_OVER_128 | P_RING, P_CHUNK_FILL | P_K_LE_4096, SQ_ALGO_RING,
     "group size 64, 16 tokens: 4608x4608 9.6 vs 11.2 (streaming kernel), 5120x5120 10.7 vs 11.3, 3200x8704 0.93 of it; but 3648x4992 "
     "1.07, 2688x8576 1.08, 4096x6016 at 10 1.14; at group size 128 5120x5120 10.5 vs 10.4"},
    // K ranges and row blocks that make a second round of few workgroups
    {5, 8, P_G64 | P_SPILL | P_PARTS5 | P_STREAM_SPLIT | P_RING, P_K_LE_4096, SQ_ALGO_RING,
     "group size 64, 8 tokens: 4352x17408 16.5 vs 19.8 (streaming kernel), 15 weights of five ranges 0.78..0.94 of it; of four ranges "
     "0.95..1.09 (5120x13824 14.6 vs 15.4, 4288x15872 at 6 16.7 vs 15.3)"},
    {9, 16, P_SPILL | P_PARTS4 | P_STREAM_SPLIT | P_RING, P_K_LE_4096, SQ_ALGO_RING,
     "16 tokens: 4352x17408 17.3 vs 19.4 (streaming kernel), 5120x13824 14.6 vs 15.9, 5120x16384 17.0 vs 17.4; but 5504x15232 at 10 "
     "1.22 of it, 5632x16000 at group size 64 21.6 vs 20.4; 8 tokens 5120x20480 18.7 vs 18.0"},
    {9, 16, P_G64 | P_SPILL | P_STREAM_SPLIT | P_RING, P_K_LE_4096, SQ_ALGO_RING,
     "16 tokens, group size 64: 10240x8192 17.6 vs 21.0 (streaming kernel), 6144x12288 17.9 vs 19.9; at group size 128 17.4 vs 16.9, "
     "17.7 vs 16.2"},
    {9, 16, P_OVER_16M | P_RING, P_G128_64, SQ_ALGO_RING,
     "16 tokens, group size 32: 5120x5120 10.3 vs 19.2, 12288x4096 12.2 vs 15.4, 4096x11008 13.0 vs 15.4; 4096x4096 8.6 vs 8.4; "
     "9 tokens: 5120x4096 9.4 vs 11.8 (16-column kernel), 16000x2048 8.2 vs 11.3, 6144x3072 8.6 vs 9.6; the other way where that "
     "kernel's N / 16 workgroups just fill their rounds: 8192x2176 8.6 vs 7.1, 4096x4608 9.0 vs 7.5"},
    // (5..8 tokens: what the GEMV below does not take.  The GEMV applies the scale to its sums in fp32)
    {5, 8, P_LARGE | P_WS | P_RING, P_G128_64, SQ_ALGO_RING,
     "8 tokens, group size 32: 12288x4096 11.7 vs 14.7 (split-K kernel) and 15.2 (GEMV), 4096x11008 12.6 vs 14.9 / 13.7, "
     "4096x8192 10.8 vs 12.3 / 10.9, 4096x16384 14.9 vs 17.5 / 18.8"},
    {5, 8, P_OVER_16M | P_RING, P_G128_64 | P_K_LE_8192, SQ_ALGO_RING,
     "8 tokens, group size 32: 2048x11008 10.3 vs 12.2 (split-K kernel), 1536x16384 10.7 vs 12.1"},
    // the streaming decode kernel, 5..16 tokens (3..4 on large weights); K beyond 4096 is split through the workspace
    {5, 16, P_G128_64 | P_K128 | P_K_LE_4096, 0, SQ_ALGO_STREAM,
     "8 tokens: fc1 10.0 vs 13.3 (split-K kernel), q/k/v in one launch 8.6 vs 12.1, 4096x4096 4.9 vs 6.5 (GEMV)"},
    {5, 16, P_STREAM_SPLIT, 0, SQ_ALGO_STREAM, "8 tokens: fc2 12.7 vs 14.6 (split-K kernel)"},
    {3, 4, P_LARGE | P_G128_64 | P_K128 | P_K_LE_4096, 0, SQ_ALGO_STREAM, "4 tokens: fc1 9.7 vs 10.7 (GEMV)"},
    {3, 4, P_LARGE | P_G128_64 | P_K128 | P_WS | P_K_LE_32768 | P_CHUNK_FILL, 0, SQ_ALGO_STREAM,
     "4 tokens: fc2 11.9 vs 13.6 (GEMV); 13824x5120, whose K ranges fill 20 of a workgroup's 32 chunks: 14.6 vs 13.9 (GEMV)"},
    // small weights at 17..32 tokens: the 16-column kernel (one launch, no exchange between workgroups)
    {17, 32, P_SMALL, 0, SQ_ALGO_SKINNY, "24 tokens: 3072x1024 4.9 vs 5.2 (ring kernel); 2048x2048 at 32 tokens 7.4 vs 6.8"},
    {17, 28, P_SMALL_K2048, 0, SQ_ALGO_SKINNY,
     "2048x1664 at 17 / 24 / 28 / 32 tokens 5.1 / 5.9 / 6.3 / 6.7 vs 7.2 / 7.2 / 7.3 / 7.3 (ring kernel, four stages of K); 1536x1792 "
     "5.2 / 5.8 / 6.2 / 6.8 vs 6.8 / 6.9 / 6.9 / 6.9; 2048x2048 5.9 / 6.4 / 6.7 / 7.0 vs 7.2 / 7.2 / 7.2 / 7.1; 1024x2048 at 28 "
     "tokens and group size 64 6.6 vs 6.5"},
    // everything else from 17 tokens up
    {17, 1 << 30, P_RING, P_SHORT_ROUNDS, SQ_ALGO_RING,
     "see sq_gemm_ring.hip: 1.25x at 24..32 tokens, 1.4x at 40..160, 1.2x at 256..700, 1.1x at 1024..2048 (geometric means over 18 weights)"},
    // group size 32 and long K at 5..16 tokens: the split-K decode kernel
    {5, 16, P_WS | P_LARGE, 0, SQ_ALGO_SKINNY_WS, "16 tokens: fc1 12.5, fc2 14.7 vs 16-column kernel 19.6 / 21.7"},
    {5, 16, P_WS, P_K_LE_8192, SQ_ALGO_SKINNY_WS, "long K: one workgroup per 16 rows cannot stage the activations in one round"},
    // the decode GEMV: up to 4 tokens, up to 8 while its staged activations fit one round
    {1, 4, 0, 0, SQ_ALGO_GEMV_FIXUP, "1 token: the four-launch layer step 27.3 per step; 4096x4096 at 4 tokens 4.4"},
    {5, 8, P_K_LE_8192, 0, SQ_ALGO_GEMV_FIXUP, "8 tokens at group size 32 (no streaming kernel): 6.5 vs 8.1 (16-column kernel)"},
    // the 16-column kernel: no workspace
    {5, 16, 0, 0, SQ_ALGO_SKINNY, "no workspace: the only kernel of this range that needs none"},
    {1, 1 << 30, 0, 0, SQ_ALGO_GEMM, "everything else: the tiled GEMM (plan_gemm picks tile height, staging and split)"},
};

int builtin_choice(int M, int N, int K, int g, bool ws_ok) {
    unsigned p = 0;
    const long nk = (long)N * (long)K;
    if (nk >= (1L << 25)) p |= P_LARGE;
    if (nk > (1L << 24)) p |= P_OVER_16M;
    if (ws_ok) p |= P_WS;
    if (g == 128 || g == 64) p |= P_G128_64;
    if (g == 64) p |= P_G64;
    if (K % 128 == 0) p |= P_K128;
    if (nk <= (1L << 22) && K <= 1536) p |= P_SMALL;
    if (nk <= (1L << 22) && K <= 2048) p |= P_SMALL_K2048;
    {
        const int chunks = K / 128, ks0 = (chunks + 31) / 32;
        if (ks0 > 0 && chunks * 4 >= ks0 * 32 * 3) p |= P_CHUNK_FILL;
        const long wgs = (long)((N + 63) / 64) * ks0;
        if (wgs > 256 && wgs <= (ks0 == 4 ? 336 : 400)) p |= P_SPILL;
        if (ks0 >= 4) p |= P_PARTS4;
        if (ks0 >= 5) p |= P_PARTS5;
        if (wgs > 128) p |= P_OVER_128;
        if (ks0 <= 2 && (wgs <= 160 || chunks * 10 < ks0 * 32 * 6)) p |= P_FEW_OVER;
    }
    if (K <= 4096) p |= P_K_LE_4096;
    if (K <= 8192) p |= P_K_LE_8192;
    if (K <= 32768) p |= P_K_LE_32768;
    if (sq::gemm_ring_applies(M, N, K)) p |= P_RING;
    if (M > 1024 && K <= 2048 && K % 256 == 0 && g >= 64) {
        // One workgroup per CU pays its first loads and its stores in full every round, two per CU hide them behind each
        // other; the ring kernel's 256 x 256 tiles make that up where they fill their last round (us, two per CU against
        // the ring kernel: 6144x1536 at 4096 tokens, 384 of its tiles, 85 against 96; 8192x1024 at 5000, 640 tiles, 97
        // against 116; 24576x1024 at 5000, 1920 tiles, 273 against 287; but 5120x2048 at 3000, 240 tiles, 71 against 63).
        // With fewer rounds or a longer K the ring kernel is ahead whatever they fill (13312x4096 at 5000, 1040 tiles, 545
        // against 533; 16384x3072 at 3000 291 against 269).
        const long tiles = (long)((N + 255) / 256) * ((M + 127) / 128);
        const long wide = (long)((N + 255) / 256) * ((M + 255) / 256), rounds = (wide + 255) / 256;
        if (tiles >= 384 && rounds > 1 && wide * 20 < rounds * 256 * 17) p |= P_SHORT_ROUNDS;
    }
    for (const ChoiceRule& r : kChoiceRules)
        if (M >= r.m_lo && M <= r.m_hi && (p & r.need) == r.need && (p & r.forbid) == 0) return r.kernel;
    return SQ_ALGO_GEMM;
}

// At group size 128 the decode kernels (up to 64 tokens) apply the scale to their sums in fp32, and so does the ring kernel
// there: W_hat would round every weight to fp16 (error against (q - z) s as real numbers, 32 tokens x 4096 columns: 2.1e-4
// with the scale on the sums, which is the rounding of the output, 2.9e-4 with W_hat).
int ring_tune(int M, int g) { return g == 128 && M <= 64 ? sq::RING_SUMS : 0; }

// Gate and up of a gated MLP in one ring launch at up to 16 tokens, us, two launches / one.  The lines were drawn through a sweep
// of 1200 weights (256..33000 rows, K 768..10500) x 1..16 tokens, with and without a workspace: where one launch is taken it takes
// 0.8 of the two in the geometric mean, at worst 1.05.
// Group size 64, 5 tokens up, where the two would be the streaming or the ring kernel's (W_hat there as here): 7680x2560 17.6 /
// 9.9, 2816x1024 6.3 / 5.7, 13824x4608 29.2 / 22.8, 12288x4096 20.4 / 19.8; but 24576x2048 at 5 20.7 / 21.1, 8512x3968 17.0 / 18.1.
// Group size 128 (the scale on the sums here as there; timed again after the lines were drawn, with zeros/scales as ring_sets has
// them and the streaming kernel's short arguments: 163 random weights where it is taken 0.82 in the geometric mean, at worst 1.10):
//   the streaming kernel's K ranges leave its chunk slots part empty: 13696x5120 at 8 tokens 29.7 / 23.5, 5632x2048 9.5 / 8.2,
//   2816x1024 6.2 / 6.1, 28672x5120 46.7 / 45.3; but at 3 19072x4992 without a workspace 33.6 / 38.7, 26112x5504 43.6 / 46.5
//   they fill them: one launch where its 32 x 128 tiles leave neither half the chip nor most of a round idle: 8192x4096 at 8 14.6 /
//   11.9, 14336x4096 18.3 / 18.6, at 16 19.0 / 19.1, 16384x4096 at 8 19.5 / 19.2, at 16 20.5 / 19.9; but at 8 8256x4096 14.6 / 17.4
//   (129 tiles), 11008x4096 16.1 / 17.8 (172), 2048x4096 9.3 / 8.9 (32; at 16 10.9 / 9.0, where the line is behind), and at 3
//   without a workspace 8384x10112 32.8 / 34.6
//   1 and 2 tokens (the GEMV): at 2 8192x5120 18.7 / 13.6, 15360x5120 30.6 / 22.7; but at 1 7680x3072 10.3 / 10.0, 9856x5120 18.5 /
//   20.6 (154 tiles), 12992x5248 22.1 / 21.9 (203)
// With few tokens a last stage of K that is half empty (K % 256 != 0) is time: 11584x5760 at 3 22.7 / 23.1, 11200x3712 at 5 and
// group size 64 17.5 / 18.4.
// Up to 8 tokens and 64 tiles the latency of two decode launches stands against one ring launch's and the exchange of its K
// ranges, or a K that is not split: 2048x2048 at 3 6.4 / 7.7, at 5 and group size 64 7.1 / 7.7; 1408x2304 at 3 7.1 / 7.8;
// 4096x3328 at 5 and group size 64 9.9 / 10.9, without a workspace 512x3840 8.7 / 10.8; 3520x2944 at 5 9.3 / 9.2;
// 3328x3712 at 16 and group size 64 without a workspace 11.3 / 12.2.
bool pair_at_few_tokens(int M, int N, int K, int g, int each, bool ws_ok) {  // each: the kernel of the two launches
    const long tiles = (2L * N + 127) / 128;
    const bool half_stage = K % 256 != 0;
    if (g == 64) {
        if (M < 5 || (tiles > 256 && K <= 4096) || (each != SQ_ALGO_STREAM && each != SQ_ALGO_RING)) return false;
        if (K > 4096) return true;
        if (M > 8) return tiles > 64 || K <= 3328 || ws_ok;
        if (K > 3328 && half_stage) return false;
        if (tiles > 64) return tiles <= 128 || tiles > 140 || K <= 3840;
        return K <= 1024 || (K <= 1536 && tiles > 16) || (K > 2048 && (K <= 2560 || (ws_ok && tiles <= 32)));
    }
    if (g != 128) return false;
    const int chunks = K / 128, parts = (chunks + 31) / 32;
    const bool filled = chunks * 100 >= parts * 32 * (parts == 1 && M > 4 && M <= 8 ? 70 : 75);
    if (M <= 2) {
        if (filled || K <= 4096 || tiles > 256 || (half_stage && tiles > 128)) return false;
        return tiles == 128 || tiles >= (K <= 4608 ? (M == 1 ? 176 : 128) : (M == 1 ? 208 : 176));
    }
    if (filled) {
        const bool spilled = K > 4096 ? M <= 4 && !ws_ok : K > (M <= 4 ? 3584 : 3328);  // tiles past 128 cost a round
        const bool whole = !half_stage || M > 8 || K > 4096;
        return (tiles > 64 && tiles <= (spilled || !whole ? 128 : 140)) || (whole && tiles >= 224 && tiles <= 256);
    }
    if (M <= 4 && K > 4096 && tiles > 128 && (half_stage || (!ws_ok && K > 5632))) return false;
    if (tiles > 256) return K > 4096 && (M > 4 || (ws_ok && K <= 5120));
    if (M > 8 || tiles > 64 || K <= 1024 || K > 4096) return M > 8 || tiles > 64 || K <= 8192 || ws_ok;
    if (K <= 2048) return tiles == 64 && K <= 1536;
    if (K <= 2560) return M > 4 || tiles > 31;
    return ws_ok && (M <= 4 ? tiles > 48 : !half_stage || tiles <= 32);
}

int gemm_dispatch(const void* x, const void* w, const void* zs, void* y, int M, int N, int K, int group_size,
                  int layout, int algo, sq::Epilogue epi, void* workspace, size_t workspace_bytes, void* stream) {
    if (M < 0) return SQ_ERR_BAD_SHAPE;
    const int rc = check_weight(N, K, group_size, layout);
    if (rc != SQ_OK) return rc;
    // The GEMM kernels consume layout L1; an L2 weight is converted once with
    // sq_repack_l2_to_l1 by the caller (the `quant` extension caches the result).
    if (layout != SQ_LAYOUT_L1) return SQ_ERR_BAD_LAYOUT;
    if (M == 0) return SQ_OK;
    if (!x || !w || !zs || !y) return SQ_ERR_NULL_POINTER;
    if (!aligned16(x) || !aligned16(w) || !aligned16(zs) || !aligned16(y)) return SQ_ERR_MISALIGNED;
    if ((long)M * (long)K > (1L << 40) || (long)M * (long)N > (1L << 40)) return SQ_ERR_BAD_SHAPE;
    hipStream_t st = static_cast<hipStream_t>(stream);

    int kernel = algo & 0xFF;
    int tune = (algo >> 8) & 0xFFFF;
    if (kernel == SQ_ALGO_AUTO && g_tuned_count.load(std::memory_order_relaxed) > 0) {
        const int word = tuned_lookup(M, N, K, group_size, full_workspace(workspace, workspace_bytes, M, N, K));
        if (word != 0) {
            kernel = word & 0xFF;
            tune = (word >> 8) & 0xFFFF;
        }
    }
    if (kernel == SQ_ALGO_AUTO) {
        kernel = builtin_choice(M, N, K, group_size, decode_workspace(workspace, workspace_bytes, M, N, K));
        if (kernel == SQ_ALGO_RING) tune = ring_tune(M, group_size);
    }
    switch (kernel) {
        case SQ_ALGO_GEMV:
        case SQ_ALGO_GEMV_FIXUP:
            if (M > 8) return SQ_ERR_BAD_ALGO;
            return launch_code(sq::launch_gemv2_tuned(x, w, zs, y, M, N, K, group_size,
                                                      kernel == SQ_ALGO_GEMV_FIXUP, tune, epi, st));
        case SQ_ALGO_SKINNY:
            if (M > 64) return SQ_ERR_BAD_ALGO;
            return launch_code(sq::launch_skinny_tuned(x, w, zs, y, M, N, K, group_size, tune, epi, st));
        case SQ_ALGO_SKINNY_WS:
            if (M > 32) return SQ_ERR_BAD_ALGO;
            if (!workspace || !aligned16(workspace) || workspace_bytes < sq::skinny2_workspace_bytes(M, N, K) ||
                (N + 63) / 64 > 16384)
                return SQ_ERR_WORKSPACE;
            return launch_code(sq::launch_skinny2_tuned(x, w, zs, y, workspace, M, N, K, group_size, tune, epi, st));
        case SQ_ALGO_STREAM: {
            if (M > 16 && M <= 32 && group_size == 128) {
                // The two-tile streaming kernel lives on in the grouped launch of the sequence entry point; for one
                // linear the ring kernel has taken its place (32 tokens: fc1 15.6 -> 13.4 us, 4096x11008 16.5 -> 12.9) on the
                // shapes this id takes.
                const bool ws_fits = workspace && aligned16(workspace) &&
                                     workspace_bytes >= sq::skinny2_workspace_bytes(M, N, K);
                if (!sq::skinny3_wide_applies(N, K, ws_fits) || !sq::gemm_ring_applies(M, N, K)) return SQ_ERR_WORKSPACE;
                return launch_code(sq::launch_gemm_ring(x, w, zs, y, aligned16(workspace) ? workspace : nullptr,
                                                        workspace_bytes, M, N, K, group_size, ring_tune(M, group_size), epi, st));
            }
            if (M > 16 || (group_size != 128 && group_size != 64)) return SQ_ERR_BAD_ALGO;
            const bool ws_fits = workspace && aligned16(workspace) &&
                                 workspace_bytes >= sq::skinny2_workspace_bytes(M, N, K);
            const hipError_t e =
                sq::launch_skinny3_tuned(x, w, zs, y, ws_fits ? workspace : nullptr, M, N, K, group_size, tune, epi, nullptr, st);
            return e == hipErrorInvalidValue ? SQ_ERR_WORKSPACE : launch_code(e);
        }
        case SQ_ALGO_GEMM:
            return launch_code(sq::launch_gemm_tuned(x, w, zs, y, aligned16(workspace) ? workspace : nullptr,
                                                     workspace_bytes, M, N, K, group_size, tune, epi, st));
        case SQ_ALGO_RING: {
            const hipError_t e = sq::launch_gemm_ring(x, w, zs, y, aligned16(workspace) ? workspace : nullptr, workspace_bytes,
                                                      M, N, K, group_size, tune, epi, st);
            return e == hipErrorInvalidValue ? SQ_ERR_WORKSPACE : launch_code(e);
        }
        default:
            return SQ_ERR_BAD_ALGO;
    }
}

}  // namespace

extern "C" {

int sq_version(void) { return 100; }

const char* sq_strerror(int code) {
    switch (code) {
        case SQ_OK: return "ok";
        case SQ_ERR_NULL_POINTER: return "null pointer argument";
        case SQ_ERR_BAD_SHAPE: return "unsupported shape (need N % 8 == 0, K % 32 == 0, K % group_size == 0)";
        case SQ_ERR_BAD_GROUP: return "unsupported group size";
        case SQ_ERR_BAD_LAYOUT: return "unknown or unsupported weight layout";
        case SQ_ERR_BAD_ALGO: return "unknown kernel id or kernel not applicable to this shape";
        case SQ_ERR_MISALIGNED: return "pointer is not 16-byte aligned";
        case SQ_ERR_LAUNCH: return "HIP kernel launch failed";
        case SQ_ERR_WORKSPACE: return "workspace missing or too small";
        case SQ_ERR_STATIC_WS: return "problem needs a larger workspace than the library's static buffer (SQ_STATIC_WS_BYTES)";
        case SQ_ERR_SEQ_TIMEOUT: return "a one-launch sequence gave up waiting for another workgroup's output (results of that call are undefined)";
        default: return "unknown error code";
    }
}

int sq_w4a16_gemm_ex(const void* x, const void* w, const void* zs, void* y, int M, int N, int K, int group_size,
                     int layout, int algo, void* stream) {
    return gemm_dispatch(x, w, zs, y, M, N, K, group_size, layout, algo, sq::Epilogue{nullptr, nullptr, 0}, nullptr, 0,
                         stream);
}

size_t sq_w4a16_workspace_bytes(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const size_t a = sq::skinny2_workspace_bytes(M > 32 ? 32 : M, N, K);
    const size_t b = M > 16 ? sq::gemm_workspace_bytes(M, N, K) : 0;
    const size_t c = M > 4 ? sq::gemm_ring_workspace_bytes(M, N, K) : 0;
    return a > b ? (a > c ? a : c) : (b > c ? b : c);
}

size_t sq_w4a16_gemm_silu_dot_workspace_bytes(int M, int N, int K) {
    const size_t each = sq_w4a16_workspace_bytes(M, N, K);
    if (each == 0 || N > (1 << 29)) return each;
    const size_t both = sq::gemm_ring_workspace_bytes(M, 2 * N, K);  // (the one launch is always the ring kernel's)
    return each > both ? each : both;
}

int sq_w4a16_gemm_ws(const void* x, const void* w, const void* zs, void* y, int M, int N, int K, int group_size,
                     int layout, int algo, void* workspace, size_t workspace_bytes, void* stream) {
    return gemm_dispatch(x, w, zs, y, M, N, K, group_size, layout, algo, sq::Epilogue{nullptr, nullptr, 0}, workspace,
                         workspace_bytes, stream);
}

// Kernel words worth timing for a shape: every family that can run it, with the tunings its launcher accepts.
// A word the launcher refuses (a K split that does not divide, a missing workspace) is skipped by the caller.
static int autotune_candidates(int M, int K, int g, bool has_ws, int* out, int cap) {
    int n = 0;
    auto add = [&](int kernel, int tune) {
        if (n < cap) out[n++] = kernel | (tune << 8);
    };
    if (M <= 8)
        for (int ks = 1; ks <= 4; ks *= 2)
            for (int nr = 2; nr <= 8; nr *= 2)
                if (nr * ks <= 16) add(SQ_ALGO_GEMV_FIXUP, nr | (ks << 4));
    if (M <= 16 && (g == 128 || g == 64) && K % 128 == 0) {
        const int rows[3] = {1, 3, 4};
        for (int r = 0; r < 3; r++)
            for (int ks = 1; ks <= 8; ks *= 2)
                if (ks == 1 ? K <= 4096 : (has_ws && K / ks >= 1024 && K / ks <= 4096)) add(SQ_ALGO_STREAM, rows[r] | (ks << 4));
    }
    if (M > 2 && M <= 32 && has_ws)
        for (int ks = 1; ks <= 8; ks *= 2) add(SQ_ALGO_SKINNY_WS, ks);
    if (M > 2 && M <= 64) add(SQ_ALGO_SKINNY, 0);
    if (M > 16) {
        for (int lds = 0; lds <= (K % 256 == 0 ? 1 : 0); lds++)
            for (int mi = 1; mi <= 4; mi *= 2) {
                if (M <= 64 && mi == 4) continue;
                for (int ks = 1; ks <= (has_ws ? 8 : 1); ks *= 2) add(SQ_ALGO_GEMM, mi | (lds ? 0x80 : 0) | (ks << 8));
            }
        if (M > 64)
            for (int v = 8; v <= 10; v++) add(SQ_ALGO_GEMM, v);
    }
    const int sums = ring_tune(M, g);  // (shapes that cannot put the scale on the sums are refused)
    if (M > 4)
        for (int shape = 1; shape <= 8; shape++)
            for (int rest = 0; rest <= (has_ws ? 1 : 0); rest++)
                for (int ks = rest ? 2 : 1; ks <= (has_ws ? 8 : 1); ks += ks < 4 ? 1 : 2)
                    add(SQ_ALGO_RING, shape | (rest ? 0x10 : 0) | sums | (ks << 8));
    if (M > 128) add(SQ_ALGO_RING, 9 | (1 << 8));  // 256 x 256 tiles: never ahead when split
    return n;
}

int sq_w4a16_autotune(const void* x, const void* w, const void* zs, void* y, int M, int N, int K, int group_size,
                      int layout, void* workspace, size_t workspace_bytes, int copies, size_t w_stride, size_t zs_stride,
                      int reps, void* stream, int* best_algo, float* best_us, float* auto_us) {
    if (M <= 0) return SQ_ERR_BAD_SHAPE;
    if (copies < 1 || copies > 4096 || reps < 1 || reps > 100000) return SQ_ERR_BAD_SHAPE;
    if (copies > 1 && (w_stride % 16 != 0 || zs_stride % 16 != 0 || w_stride < (size_t)N * K / 2)) return SQ_ERR_MISALIGNED;
    const sq::Epilogue none{nullptr, nullptr, 0};
    hipStream_t st = static_cast<hipStream_t>(stream);
    // A recorded word has to fit every workspace that counts as full later on: no candidate sees more than that.
    const bool has_ws = full_workspace(workspace, workspace_bytes, M, N, K);
    if (!has_ws) workspace = nullptr;
    workspace_bytes = has_ws ? sq_w4a16_workspace_bytes(M, N, K) : 0;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        if (e0) (void)hipEventDestroy(e0);
        return SQ_ERR_LAUNCH;
    }
    // One candidate: a launch that has to succeed, a short warm-up, then `reps` launches between two events,
    // walking through the `copies` weights so that a pool larger than the last-level cache is read from HBM.
    auto run = [&](int word, int i) {
        const size_t c = (size_t)(i % copies);
        return gemm_dispatch(x, static_cast<const uint8_t*>(w) + c * w_stride, static_cast<const uint8_t*>(zs) + c * zs_stride,
                             y, M, N, K, group_size, layout, word, none, workspace, workspace_bytes, stream);
    };
    int status = SQ_OK;
    auto time_word = [&](int word, float* us) {
        int rc = run(word, 0);
        if (rc != SQ_OK) return rc;
        // as many untimed launches as timed ones: clocks and caches are in the candidate's own steady state
        for (int i = 1; i < reps; i++) (void)run(word, i);
        if (hipEventRecord(e0, st) != hipSuccess) return (int)SQ_ERR_LAUNCH;
        for (int i = 0; i < reps; i++) rc |= run(word, i + reps);
        if (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess) return (int)SQ_ERR_LAUNCH;
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, e0, e1) != hipSuccess) return (int)SQ_ERR_LAUNCH;
        *us = ms * 1000.f / (float)reps;
        return rc;
    };
    // the built-in choice first (with any earlier measurement of this shape out of the way)
    float t_auto = 0.f;
    {
        std::lock_guard<std::mutex> lock(g_tuned_mutex);
        const int n = g_tuned_count.load(std::memory_order_relaxed);
        for (int i = 0; i < n; i++) {
            TunedEntry& e = g_tuned[i];
            if (e.M == M && e.N == N && e.K == K && e.g == group_size && e.has_ws == (int)has_ws) e.M = -1;
        }
    }
    for (int i = 0; i < 2 * reps; i++) (void)run(SQ_ALGO_AUTO, i);  // out of the idle state before anything is timed
    status = time_word(SQ_ALGO_AUTO, &t_auto);
    int best = 0;
    float t_best = t_auto;
    if (status == SQ_OK) {
        int words[192];
        const int n = autotune_candidates(M, K, group_size, has_ws, words, 192);
        for (int i = 0; i < n; i++) {
            float t = 0.f;
            const int rc = time_word(words[i], &t);
            if (rc == SQ_ERR_LAUNCH) {
                status = rc;
                break;
            }
            if (rc == SQ_OK && t < t_best) {
                t_best = t;
                best = words[i];
            }
        }
    }
    if (status == SQ_OK && best != 0) {
        // A candidate has to beat the built-in choice twice, the second time against a fresh timing of both (the
        // clocks of this part move with the load, and an early window can read a few percent off).
        float t_auto2 = 0.f, t_best2 = 0.f;
        if (time_word(SQ_ALGO_AUTO, &t_auto2) == SQ_OK && time_word(best, &t_best2) == SQ_OK) {
            if (t_auto2 < t_auto) t_auto = t_auto2;
            if (t_best2 > t_best) t_best = t_best2;
            if (t_best >= 0.99f * t_auto) {
                best = 0;
                t_best = t_auto;
            }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (status != SQ_OK) return status;
    // leave the caller's output as the chosen kernel writes it
    status = run(best, 0);
    if (status != SQ_OK) return status;
    if (best != 0) {
        std::lock_guard<std::mutex> lock(g_tuned_mutex);
        const int n = g_tuned_count.load(std::memory_order_relaxed);
        if (n < TUNED_MAX) {
            g_tuned[n] = TunedEntry{M, N, K, group_size, (int)has_ws, best, t_best};
            g_tuned_count.store(n + 1, std::memory_order_release);
        }
    }
    if (best_algo) *best_algo = best;
    if (best_us) *best_us = t_best;
    if (auto_us) *auto_us = t_auto;
    return SQ_OK;
}

int sq_w4a16_autotune_clear(void) {
    std::lock_guard<std::mutex> lock(g_tuned_mutex);
    const int n = g_tuned_count.load(std::memory_order_relaxed);
    int live = 0;
    for (int i = 0; i < n; i++) {  // readers may be scanning: entries are voided, never moved
        if (g_tuned[i].M >= 0) live++;
        g_tuned[i].M = -1;
    }
    return live;
}

int sq_w4a16_gemm_static_ws(const void* x, const void* w, const void* zs, void* y, int M, int N, int K, int group_size,
                            int layout, int algo, void* stream) {
    // Validate before touching the device, so that argument errors launch nothing.
    if (M < 0) return SQ_ERR_BAD_SHAPE;
    const int rc = check_weight(N, K, group_size, layout);
    if (rc != SQ_OK) return rc;
    if (layout != SQ_LAYOUT_L1) return SQ_ERR_BAD_LAYOUT;
    // What the kernels of this token count would take from a workspace: nothing up to 2 tokens (the GEMV has
    // no workspace form), the split-K decode kernels' counters and partial tiles up to 32, the tiled GEMM's K
    // split beyond (the ring kernel's always fits).  A shape that wants more than the static
    // buffer is refused rather than served by a slower workspace-free kernel behind the caller's back.
    const size_t need = M <= 2 ? 0 : (M <= 32 ? sq::skinny2_workspace_bytes(M, N, K) : sq::gemm_workspace_bytes(M, N, K));
    if (need > (size_t)SQ_STATIC_WS_BYTES) return SQ_ERR_STATIC_WS;
    if (M == 0) return SQ_OK;
    if (!x || !w || !zs || !y) return SQ_ERR_NULL_POINTER;
    if (!aligned16(x) || !aligned16(w) || !aligned16(zs) || !aligned16(y)) return SQ_ERR_MISALIGNED;
    void* ws = static_workspace();
    if (!ws) return SQ_ERR_LAUNCH;
    return gemm_dispatch(x, w, zs, y, M, N, K, group_size, layout, algo, sq::Epilogue{nullptr, nullptr, 0}, ws,
                         SCRATCH_BYTES, stream);
}

int sq_workspace_reset(void* workspace, size_t bytes, void* stream) {
    if (!workspace) return SQ_ERR_NULL_POINTER;
    if (!aligned16(workspace) || bytes % 4 != 0) return SQ_ERR_MISALIGNED;
    if (bytes == 0) return SQ_OK;
    if (bytes > ((size_t)1 << 30)) return SQ_ERR_BAD_SHAPE;
    const int words = (int)(bytes / 4);
    hipLaunchKernelGGL(zero_words_kernel, dim3((words + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<unsigned*>(workspace), words);
    return launch_code(hipGetLastError());
}

int sq_workspace_check(const void* workspace, size_t bytes, void* stream) {
    if (!workspace) return SQ_ERR_NULL_POINTER;
    if (bytes % 4 != 0) return SQ_ERR_MISALIGNED;
    if (bytes > 65536) bytes = 65536;
    static thread_local unsigned host[65536 / 4];
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (hipMemcpyAsync(host, workspace, bytes, hipMemcpyDeviceToHost, st) != hipSuccess) return SQ_ERR_LAUNCH;
    if (hipStreamSynchronize(st) != hipSuccess) return SQ_ERR_LAUNCH;
    for (size_t i = 0; i < bytes / 4; i++)
        if (host[i] != 0u) return SQ_ERR_WORKSPACE;
    return SQ_OK;
}

static void to_problems(const sq_linear_desc* linears, int count, sq::SeqProblem* probs) {
    for (int l = 0; l < count; l++) {
        const sq_linear_desc& d = linears[l];
        probs[l] = sq::SeqProblem{d.x, d.w, d.zs, d.bias, d.residual, d.y, d.N, d.K, d.group_size, d.act, d.depends};
    }
}

// A sequence's workspace: first what the split-K kernels of the launch-per-linear path want (64 KiB of counters
// and the partial tiles; nothing beyond the counters up to 2 tokens), then, 256-byte aligned, the region of the
// one-launch kernel (control block and exchange words), which no other kernel writes.
static size_t sequence_splitk_bytes(const sq_linear_desc* linears, int count, int M) {
    const size_t base = 65536;
    if (!linears || count <= 0 || count > SQ_SEQUENCE_MAX || M <= 2) return base;
    // more than 2 tokens: what sq_w4a16_gemm_ws wants for the largest run of linears that may share a launch
    // (their rows concatenated, each rounded up to a 64-row block) and for every single linear
    // (the ring kernel splits K of a narrow weight further than that of a wide one: one linear can want more than the run)
    long rows = 0;
    int kmax = 0;
    size_t need = base;
    for (int l = 0; l < count; l++) {
        if (linears[l].N <= 0 || linears[l].K <= 0) return base;
        rows += ((long)linears[l].N + 63) / 64 * 64;
        if (linears[l].K > kmax) kmax = linears[l].K;
    }
    if (rows > (1L << 30)) return base;
    for (int l = -1; l < count; l++) {
        const size_t a = l < 0 ? sq_w4a16_workspace_bytes(M, (int)rows, kmax)
                               : sq_w4a16_workspace_bytes(M, linears[l].N, linears[l].K);
        if (a > need) need = a;
    }
    return (need + 255) & ~(size_t)255;
}

size_t sq_w4a16_gemv_sequence_workspace_bytes(const sq_linear_desc* linears, int count, int M) {
    sq::SeqProblem probs[SQ_SEQUENCE_MAX];
    const bool listed = linears && count > 0 && count <= SQ_SEQUENCE_MAX;
    if (listed) to_problems(linears, count, probs);
    return sequence_splitk_bytes(linears, count, M) + sq::gemv_seq_workspace_bytes(listed ? probs : nullptr, count, M);
}

int sq_w4a16_gemv_sequence_status(const sq_linear_desc* linears, int count, int M, void* workspace,
                                  size_t workspace_bytes, int clear, void* stream) {
    if (!linears || !workspace) return SQ_ERR_NULL_POINTER;
    if (count <= 0 || count > SQ_SEQUENCE_MAX) return SQ_ERR_BAD_SHAPE;
    const size_t off = sequence_splitk_bytes(linears, count, M);
    if (!aligned16(workspace) || workspace_bytes < off + 256) return SQ_ERR_WORKSPACE;
    unsigned* ctrl = reinterpret_cast<unsigned*>(static_cast<uint8_t*>(workspace) + off);
    unsigned host[4] = {0, 0, 0, 0};
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (hipMemcpyAsync(host, ctrl, sizeof(host), hipMemcpyDeviceToHost, st) != hipSuccess) return SQ_ERR_LAUNCH;
    if (hipStreamSynchronize(st) != hipSuccess) return SQ_ERR_LAUNCH;
    if (clear && host[1] != 0u) {
        hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(64), 0, st, ctrl + 1, 1);
        if (hipGetLastError() != hipSuccess) return SQ_ERR_LAUNCH;
    }
    if (host[2] != 0u) return SQ_ERR_WORKSPACE;  // an exit counter that is not back at zero: a launch did not finish
    return host[1] != 0u ? SQ_ERR_SEQ_TIMEOUT : SQ_OK;
}

// Tuning of the persistent sequence kernel (sq_w4a16_gemv_sequence_tune): polls allowed for another workgroup's
// output, and loads a streaming wave keeps in flight (0: the kernel's default).
static unsigned g_seq_spin_limit = 1u << 16;
static int g_seq_lim = 0;

int sq_w4a16_gemv_sequence_tune(unsigned spin_limit, int loads_in_flight) {
    if (loads_in_flight < 0 || loads_in_flight > 16) return SQ_ERR_BAD_SHAPE;
    g_seq_spin_limit = spin_limit;
    g_seq_lim = loads_in_flight;
    return SQ_OK;
}

int sq_w4a16_gemv_sequence(const sq_linear_desc* linears, int count, int M, int layout, int mode, void* workspace,
                           size_t workspace_bytes, void* stream) {
    if (count < 0 || count > SQ_SEQUENCE_MAX) return SQ_ERR_BAD_SHAPE;
    if (mode != SQ_SEQ_AUTO && mode != SQ_SEQ_ONE_LAUNCH) return SQ_ERR_BAD_ALGO;
    if (count == 0) return SQ_OK;
    if (!linears) return SQ_ERR_NULL_POINTER;
    if (M < 0) return SQ_ERR_BAD_SHAPE;
    if (layout != SQ_LAYOUT_L1) return SQ_ERR_BAD_LAYOUT;
    sq::SeqProblem probs[SQ_SEQUENCE_MAX];
    for (int l = 0; l < count; l++) {
        const sq_linear_desc& d = linears[l];
        const int rc = check_weight(d.N, d.K, d.group_size, layout);
        if (rc != SQ_OK) return rc;
        if (d.act != SQ_ACT_NONE && d.act != SQ_ACT_RELU) return SQ_ERR_BAD_ALGO;
        if (M > 0) {
            if (!d.x || !d.w || !d.zs || !d.y) return SQ_ERR_NULL_POINTER;
            if (!aligned16(d.x) || !aligned16(d.w) || !aligned16(d.zs) || !aligned16(d.y)) return SQ_ERR_MISALIGNED;
            if ((d.bias && (reinterpret_cast<uintptr_t>(d.bias) & 1u)) ||
                (d.residual && (reinterpret_cast<uintptr_t>(d.residual) & 1u)))
                return SQ_ERR_MISALIGNED;
        }
        probs[l] = sq::SeqProblem{d.x, d.w, d.zs, d.bias, d.residual, d.y, d.N, d.K, d.group_size, d.act, d.depends};
    }
    if (M == 0) return SQ_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (workspace && !aligned16(workspace)) workspace = nullptr;
    if (mode == SQ_SEQ_ONE_LAUNCH && workspace && M <= 4) {
        // everything in one persistent launch; outputs that later linears read travel as tagged words
        const size_t off = sequence_splitk_bytes(linears, count, M);
        const int rc = workspace_bytes > off ? sq::launch_gemv_seq(probs, count, M, static_cast<uint8_t*>(workspace) + off,
                                                                   workspace_bytes - off, g_seq_spin_limit, g_seq_lim, st)
                                             : 1;
        if (rc == 0) return SQ_OK;
        if (rc == 2) return SQ_ERR_LAUNCH;
    }
    // A linear that depends on an earlier one starts a new launch: the kernel boundary is the cheapest way to
    // honour a dependency on this part (about 2 us, against 5..9 us for a grid barrier inside a persistent
    // kernel).  Consecutive linears that do not depend on each other and share K and the group size (q, k and
    // v of a decoder layer) go out as ONE launch of the single-linear GEMV whose grid is the concatenation of
    // their row blocks.  Everything else (more than 4 tokens, K beyond 8192, a lone linear) is one launch per
    // linear through the automatic dispatch.
    int l0 = 0;
    while (l0 < count) {
        int l1 = l0 + 1;
        while (l1 < count && l1 - l0 < sq::GEMV_GROUP_MAX && !probs[l1].depends && probs[l1].K == probs[l0].K &&
               probs[l1].group_size == probs[l0].group_size)
            l1++;
        bool done = false;
        if (l1 - l0 > 1 && M <= 4 && probs[l0].K <= 8192) {
            const hipError_t e = sq::launch_gemv2_group(probs + l0, l1 - l0, M, st);
            if (e == hipSuccess)
                done = true;
            else if (e != hipErrorInvalidValue)
                return SQ_ERR_LAUNCH;
        } else if (l1 - l0 > 1 && M > 4 && M <= 16 && probs[l0].group_size == 128 && probs[l0].K % 128 == 0 &&
                   (probs[l0].K <= 4096 || workspace)) {
            // the streaming decode kernel on the concatenated row blocks (a K beyond 4096 needs the workspace)
            const hipError_t e = sq::launch_skinny3_group(probs + l0, l1 - l0, M, workspace, workspace_bytes, st);
            if (e == hipSuccess)
                done = true;
            else if (e != hipErrorInvalidValue)
                return SQ_ERR_LAUNCH;
        }
        if (!done && l1 - l0 > 1 && M > 16 && M <= 32 && probs[l0].group_size == 128 && probs[l0].K % 128 == 0 &&
            (probs[l0].K <= 4096 || workspace)) {
            const hipError_t e = sq::launch_skinny3_wide_group(probs + l0, l1 - l0, M, workspace, workspace_bytes, st);
            if (e == hipSuccess)
                done = true;
            else if (e != hipErrorInvalidValue)
                return SQ_ERR_LAUNCH;
        }
        if (!done && l1 - l0 > 1 && M > 4 && M <= 32 && workspace && aligned16(workspace)) {
            // the split-K decode kernel on the concatenated row blocks: large weights, more than 16 tokens, or long K
            // (17..32 tokens, the grouped launches against a launch of the ring kernel each, us at 32 tokens and group
            // size 128: q/k/v of 4096x4096 14.9 / 27.4, 5120 + 1024 + 1024 rows of 5120 16.5 / 27.7, three of 1024x1024
            // 7.3 / 23.8; two of 11008x4096 26.7 / 24.0.  One weight of their rows through the ring kernel: 12.1, 11.2,
            // 8.0, 18.7)
            long elems = 0;
            for (int l = l0; l < l1; l++) elems += (long)probs[l].N * probs[l].K;
            if (elems >= (1L << 25) || M > 16 || probs[l0].K > 8192) {
                const hipError_t e = sq::launch_skinny2_group(probs + l0, l1 - l0, M, workspace, workspace_bytes, st);
                if (e == hipSuccess)
                    done = true;
                else if (e != hipErrorInvalidValue)
                    return SQ_ERR_LAUNCH;
            }
        }
        if (!done) {
            for (int l = l0; l < l1; l++) {
                const sq::SeqProblem& q = probs[l];
                const sq::Epilogue epi{static_cast<const sq::half_t*>(q.bias), static_cast<const sq::half_t*>(q.residual),
                                       q.act};
                // no more than it needs: behind that may lie the one-launch mode's region (see sequence_splitk_bytes)
                size_t bytes = 0;
                if (M > 2 && workspace) {
                    bytes = sq_w4a16_workspace_bytes(M, q.N, q.K);
                    if (workspace_bytes < bytes) bytes = workspace_bytes;
                }
                const int rc = gemm_dispatch(q.x, q.w, q.zs, q.y, M, q.N, q.K, q.group_size, layout, SQ_ALGO_AUTO, epi,
                                             bytes ? workspace : nullptr, bytes, stream);
                if (rc != SQ_OK) return rc;
            }
        }
        l0 = l1;
    }
    return SQ_OK;
}

int sq_w4a16_gemm_fused(const void* x, const void* w, const void* zs, const void* bias, const void* residual, void* y,
                        int M, int N, int K, int group_size, int layout, int act, int algo, void* workspace,
                        size_t workspace_bytes, void* stream) {
    if (act != SQ_ACT_NONE && act != SQ_ACT_RELU && act != SQ_ACT_SILU) return SQ_ERR_BAD_ALGO;
    if (bias && (reinterpret_cast<uintptr_t>(bias) & 1u)) return SQ_ERR_MISALIGNED;
    if (residual && (reinterpret_cast<uintptr_t>(residual) & 1u)) return SQ_ERR_MISALIGNED;
    const sq::Epilogue epi{static_cast<const sq::half_t*>(bias), static_cast<const sq::half_t*>(residual), act};
    return gemm_dispatch(x, w, zs, y, M, N, K, group_size, layout, algo, epi, workspace, workspace_bytes, stream);
}

// Both products in one launch where the ring kernel is the choice for each, or pair_at_few_tokens says so, and no measured
// choice of the shape names a third kernel; SQ_ERR_BAD_ALGO, with nothing launched, where it is not.
static int silu_dot_one(const void* x, const void* w_gate, const void* zs_gate, const void* w_up, const void* zs_up, void* y,
                        void* up, int M, int N, int K, int group_size, int layout, int algo, void* workspace,
                        size_t workspace_bytes, void* stream) {
    if (M < 0) return SQ_ERR_BAD_SHAPE;
    const int rc = check_weight(N, K, group_size, layout);
    if (rc != SQ_OK) return rc;
    if (layout != SQ_LAYOUT_L1) return SQ_ERR_BAD_LAYOUT;
    if (M == 0) return SQ_OK;
    if (!x || !w_gate || !zs_gate || !w_up || !zs_up || !y) return SQ_ERR_NULL_POINTER;
    if (!aligned16(x) || !aligned16(w_gate) || !aligned16(zs_gate) || !aligned16(w_up) || !aligned16(zs_up) || !aligned16(y))
        return SQ_ERR_MISALIGNED;
    if (N > (1 << 29)) return SQ_ERR_BAD_ALGO;
    int tune = ring_tune(M, group_size);
    if (algo == SQ_ALGO_AUTO) {
        const bool ws_ok = decode_workspace(workspace, workspace_bytes, M, N, K);
        const int each = builtin_choice(M, N, K, group_size, ws_ok);
        if (M <= 16 ? !pair_at_few_tokens(M, N, K, group_size, each, ws_ok) : each != SQ_ALGO_RING) return SQ_ERR_BAD_ALGO;
        if (g_tuned_count.load(std::memory_order_relaxed) > 0) {
            // A measured choice is one linear's.  Another shape of the ring kernel, or another form of the kernel that the
            // one launch is ahead of, is no measurement against it; any other kernel is.
            const int measured = tuned_lookup(M, N, K, group_size, full_workspace(workspace, workspace_bytes, M, N, K)) & 0xFF;
            if (measured != SQ_ALGO_AUTO && measured != SQ_ALGO_RING && measured != each) return SQ_ERR_BAD_ALGO;
        }
    } else {
        if ((algo & 0xFF) != SQ_ALGO_RING) return SQ_ERR_BAD_ALGO;
        tune = (algo >> 8) & 0xFFFF;
    }
    const hipError_t e = sq::launch_gemm_ring_pair(x, w_gate, zs_gate, w_up, zs_up, y, up,
                                                   aligned16(workspace) ? workspace : nullptr, workspace_bytes, M, N, K,
                                                   group_size, tune, static_cast<hipStream_t>(stream));
    return e == hipErrorInvalidValue ? SQ_ERR_BAD_ALGO : launch_code(e);
}

int sq_w4a16_gemm_silu_dot_one(const void* x, const void* w_gate, const void* zs_gate, const void* w_up, const void* zs_up,
                               void* y, int M, int N, int K, int group_size, int layout, int algo, void* workspace,
                               size_t workspace_bytes, void* stream) {
    return silu_dot_one(x, w_gate, zs_gate, w_up, zs_up, y, nullptr, M, N, K, group_size, layout, algo, workspace,
                        workspace_bytes, stream);
}

int sq_w4a16_gemm_silu_dot(const void* x, const void* w_gate, const void* zs_gate, const void* w_up, const void* zs_up,
                           void* y, void* up_scratch, int M, int N, int K, int group_size, int layout, void* workspace,
                           size_t workspace_bytes, void* stream) {
    if (M > 0 && (!up_scratch || !w_up || !zs_up)) return SQ_ERR_NULL_POINTER;
    if (M > 0 && !aligned16(up_scratch)) return SQ_ERR_MISALIGNED;
    if (M > 0 && up_scratch == y) return SQ_ERR_BAD_SHAPE;
    {
        const int rc = silu_dot_one(x, w_gate, zs_gate, w_up, zs_up, y, up_scratch, M, N, K, group_size, layout, SQ_ALGO_AUTO,
                                    workspace, workspace_bytes, stream);
        if (rc != SQ_ERR_BAD_ALGO) return rc;
    }
    // the up projection first, rounded to fp16 once; the gate projection multiplies it into its store
    const int rc = gemm_dispatch(x, w_up, zs_up, up_scratch, M, N, K, group_size, layout, SQ_ALGO_AUTO,
                                 sq::Epilogue{nullptr, nullptr, SQ_ACT_NONE}, workspace, workspace_bytes, stream);
    if (rc != SQ_OK || M == 0) return rc;
    sq::Epilogue epi{nullptr, nullptr, SQ_ACT_SILU};
    epi.mul = static_cast<const sq::half_t*>(up_scratch);
    return gemm_dispatch(x, w_gate, zs_gate, y, M, N, K, group_size, layout, SQ_ALGO_AUTO, epi, workspace,
                         workspace_bytes, stream);
}

int sq_w4a16_gemm(const void* x, const void* w, const void* zs, void* y, int M, int N, int K, int group_size,
                  int layout, void* stream) {
    return sq_w4a16_gemm_ex(x, w, zs, y, M, N, K, group_size, layout, SQ_ALGO_AUTO, stream);
}

int sq_w4a16_dequant(const void* w, const void* zs, void* out, int N, int K, int group_size, int layout,
                     void* stream) {
    const int rc = check_weight(N, K, group_size, layout);
    if (rc != SQ_OK) return rc;
    if (!w || !zs || !out) return SQ_ERR_NULL_POINTER;
    if (!aligned16(w) || !aligned16(zs) || !aligned16(out)) return SQ_ERR_MISALIGNED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (layout == SQ_LAYOUT_L1) return launch_code(sq::launch_dequant_l1(w, zs, out, N, K, group_size, st));
    return launch_code(sq::launch_dequant_l2(w, zs, out, N, K, group_size, st));
}

int sq_w4a16_quantise(const void* w, void* q, void* zs, void* fake, int N, int K, int group_size, int n_bit, int layout,
                      void* stream) {
    if (layout != SQ_LAYOUT_L1 && layout != SQ_LAYOUT_L2) return SQ_ERR_BAD_LAYOUT;
    if (group_size != 32 && group_size != 64 && group_size != 128) return SQ_ERR_BAD_GROUP;
    if (N <= 0 || K <= 0 || K % group_size != 0 || (n_bit != 2 && n_bit != 4)) return SQ_ERR_BAD_SHAPE;
    if (layout == SQ_LAYOUT_L2 ? (N % 32 != 0 || K > (1 << 22)) : fake != nullptr) return SQ_ERR_BAD_SHAPE;
    if ((long)N * (long)K > (1L << 40)) return SQ_ERR_BAD_SHAPE;
    if (!w || !q || !zs) return SQ_ERR_NULL_POINTER;
    if (!aligned16(w) || !aligned16(q) || !aligned16(zs) || !aligned16(fake)) return SQ_ERR_MISALIGNED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (layout == SQ_LAYOUT_L1) return launch_code(sq::launch_quantise_l1(w, q, zs, N, K, group_size, n_bit, st));
    return launch_code(sq::launch_quantise_l2(w, q, zs, fake, N, K, group_size, n_bit, st));
}

int sq_transpose_merge_zeros_scales(const void* zeros, const void* scales, void* zs, int in_features,
                                    int out_features, int group_size, void* stream) {
    if (in_features <= 0 || out_features <= 0) return SQ_ERR_BAD_SHAPE;
    if (group_size <= 0 || in_features % group_size != 0) return SQ_ERR_BAD_GROUP;
    if (!zeros || !scales || !zs) return SQ_ERR_NULL_POINTER;
    return launch_code(sq::launch_transpose_merge_zeros_scales(zeros, scales, zs, in_features, out_features,
                                                               group_size, static_cast<hipStream_t>(stream)));
}

int sq_convert_ours_to_awq(const void* src, void* dst, int in_features, int out_features, void* stream) {
    if (in_features <= 0 || out_features <= 0 || in_features % 2 != 0 || out_features % 8 != 0)
        return SQ_ERR_BAD_SHAPE;
    if (!src || !dst) return SQ_ERR_NULL_POINTER;
    return launch_code(
        sq::launch_ours_to_awq(src, dst, in_features, out_features, static_cast<hipStream_t>(stream)));
}

int sq_convert_awq_to_lmdeploy(const void* src, void* dst, int in_features, int out_features, void* stream) {
    if (in_features <= 0 || out_features <= 0 || in_features % 32 != 0 || out_features % 32 != 0)
        return SQ_ERR_BAD_SHAPE;
    if (!src || !dst) return SQ_ERR_NULL_POINTER;
    if (src == dst) return SQ_ERR_BAD_SHAPE;
    return launch_code(
        sq::launch_awq_to_lmdeploy(src, dst, in_features, out_features, static_cast<hipStream_t>(stream)));
}

int sq_repack_l2_to_l1(const void* w_l2, const void* zs_l2, void* w_l1, void* zs_l1, int N, int K, int group_size,
                       void* stream) {
    const int rc = check_weight(N, K, group_size, SQ_LAYOUT_L2);
    if (rc != SQ_OK) return rc;
    if (!w_l2 || !zs_l2 || !w_l1 || !zs_l1) return SQ_ERR_NULL_POINTER;
    return launch_code(
        sq::launch_l2_to_l1(w_l2, zs_l2, w_l1, zs_l1, N, K, group_size, static_cast<hipStream_t>(stream)));
}

int sq_convert_2bit_to_4bit(const void* src, void* dst, int N, int K, void* stream) {
    if (N <= 0 || K <= 0 || K % 4 != 0) return SQ_ERR_BAD_SHAPE;
    if (!src || !dst) return SQ_ERR_NULL_POINTER;
    return launch_code(sq::launch_2bit_to_4bit(src, dst, N, K, static_cast<hipStream_t>(stream)));
}

int sq_l2_convert_4bit_to_2bit(const void* src, void* dst, int K, int N, void* stream) {
    if (N <= 0 || K <= 0 || N % 16 != 0) return SQ_ERR_BAD_SHAPE;
    if (!src || !dst) return SQ_ERR_NULL_POINTER;
    return launch_code(sq::launch_l2_4bit_to_2bit(src, dst, K, N, static_cast<hipStream_t>(stream)));
}

int sq_l2_convert_2bit_to_4bit(const void* src, void* dst, int K, int N, void* stream) {
    if (N <= 0 || K <= 0 || N % 16 != 0) return SQ_ERR_BAD_SHAPE;
    if (!src || !dst) return SQ_ERR_NULL_POINTER;
    return launch_code(sq::launch_l2_2bit_to_4bit(src, dst, K, N, static_cast<hipStream_t>(stream)));
}

int sq_lut_attention_fwd(const void* q, const void* k, const void* v, void* out, const void* lut, int lut_elem_bytes,
                         int Z, int H, int S, int D, int nnz, float sm_scale, int causal, void* stream) {
    if (Z <= 0 || H <= 0 || S <= 0 || nnz <= 0 || (D != 64 && D != 128)) return SQ_ERR_BAD_SHAPE;
    if ((long)Z * H > 65535) return SQ_ERR_BAD_SHAPE;
    if (lut_elem_bytes != 4 && lut_elem_bytes != 8) return SQ_ERR_BAD_LAYOUT;
    if (!q || !k || !v || !out || !lut) return SQ_ERR_NULL_POINTER;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out)) return SQ_ERR_MISALIGNED;
    const long hs = (long)S * D, zs = hs * H;
    const sq::LutAttnStrides st = {{zs, hs, D}, {zs, hs, D}, {zs, hs, D}, {0, 0, 0}};
    return launch_code(sq::launch_lut_attention(q, k, v, out, nullptr, nullptr, lut, lut_elem_bytes, Z, H, S, D, nnz, st,
                                                sm_scale, causal, static_cast<hipStream_t>(stream)));
}

int sq_lut_attention_strided(const void* q, const void* k, const void* v, void* out, void* k_cache, void* v_cache,
                             const void* lut, int lut_elem_bytes, int Z, int H, int S, int D, int nnz, const long* strides,
                             float sm_scale, int causal, void* stream) {
    if (Z <= 0 || H <= 0 || S <= 0 || (D != 64 && D != 128) || (lut && nnz <= 0)) return SQ_ERR_BAD_SHAPE;
    if ((long)Z * H > 65535) return SQ_ERR_BAD_SHAPE;
    if (lut && lut_elem_bytes != 4 && lut_elem_bytes != 8) return SQ_ERR_BAD_LAYOUT;
    if (!q || !k || !v || !out || !strides || !k_cache != !v_cache) return SQ_ERR_NULL_POINTER;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out)) return SQ_ERR_MISALIGNED;
    if (k_cache && (!aligned16(k_cache) || !aligned16(v_cache))) return SQ_ERR_MISALIGNED;
    sq::LutAttnStrides st;
    for (int i = 0; i < 3; i++) {
        st.q[i] = strides[i];
        st.kv[i] = strides[3 + i];
        st.o[i] = strides[6 + i];
        st.c[i] = k_cache ? strides[9 + i] : 0;
    }
    for (int i = 0; i < (k_cache ? 12 : 9); i++) {
        if (strides[i] < 0) return SQ_ERR_BAD_SHAPE;
        if (strides[i] % 8 != 0) return SQ_ERR_MISALIGNED;
    }
    if (st.kv[2] >= (1L << 24)) return SQ_ERR_BAD_SHAPE;  // 32-bit byte offsets inside a step of 32 rows
    return launch_code(sq::launch_lut_attention(q, k, v, out, k_cache, v_cache, lut, lut_elem_bytes, Z, H, S, D, nnz, st,
                                                sm_scale, causal, static_cast<hipStream_t>(stream)));
}

int sq_decode_attention(const void* q, const void* k_new, const void* v_new, void* k_cache, void* v_cache,
                        const void* mask, void* out, int B, int H, int D, int Lmax, long q_bstride, long q_hstride,
                        long new_bstride, long new_hstride, long cache_bstride, long cache_hstride, long mask_bstride,
                        int cache_len, const long long* cache_len_dev, float sm_scale, void* workspace,
                        size_t workspace_bytes, void* stream) {
    if (B <= 0 || H <= 0 || Lmax <= 0 || (D != 64 && D != 128)) return SQ_ERR_BAD_SHAPE;
    if ((long)B * H > (1L << 24)) return SQ_ERR_BAD_SHAPE;
    if (!q || !k_cache || !v_cache || !out) return SQ_ERR_NULL_POINTER;
    if ((k_new == nullptr) != (v_new == nullptr)) return SQ_ERR_NULL_POINTER;
    const bool append = k_new != nullptr;
    if (!cache_len_dev) {  // a length on the device is clamped to the cache by the kernel
        if (cache_len < 0 || cache_len + (append ? 1 : 0) > Lmax || cache_len + (append ? 1 : 0) < 1)
            return SQ_ERR_BAD_SHAPE;
    }
    if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || (append && (!aligned16(k_new) || !aligned16(v_new))))
        return SQ_ERR_MISALIGNED;
    if ((q_bstride | q_hstride | cache_bstride | cache_hstride) % 8 != 0) return SQ_ERR_MISALIGNED;
    if (append && (new_bstride | new_hstride) % 8 != 0) return SQ_ERR_MISALIGNED;
    if (q_bstride < 0 || q_hstride < 0 || cache_bstride < 0 || cache_hstride < (long)Lmax * D || mask_bstride < 0 ||
        (append && (new_bstride < 0 || new_hstride < 0)))
        return SQ_ERR_BAD_SHAPE;
    return launch_code(sq::launch_decode_attention(q, k_new, v_new, k_cache, v_cache, mask, out, B, H, D, Lmax,
                                                   q_bstride, q_hstride, new_bstride, new_hstride, cache_bstride,
                                                   cache_hstride, mask_bstride, cache_len, cache_len_dev, sm_scale,
                                                   aligned16(workspace) ? workspace : nullptr, workspace_bytes,
                                                   static_cast<hipStream_t>(stream)));
}

size_t sq_decode_attention_workspace_bytes(int B, int H, int D) {
    if (B <= 0 || H <= 0 || (D != 64 && D != 128)) return 0;
    return sq::decode_attention_workspace_bytes(B, H, D);
}

int sq_layernorm(const void* x, const void* gamma, const void* beta, void* y, int rows, int cols, float eps,
                 void* stream) {
    if (rows < 0 || cols <= 0 || cols % 8 != 0 || cols > 16384) return SQ_ERR_BAD_SHAPE;
    if (rows == 0) return SQ_OK;
    if (!x || !y) return SQ_ERR_NULL_POINTER;
    if (!aligned16(x) || !aligned16(y) || (gamma && !aligned16(gamma)) || (beta && !aligned16(beta)))
        return SQ_ERR_MISALIGNED;
    return launch_code(sq::launch_layernorm(x, gamma, beta, y, rows, cols, eps, static_cast<hipStream_t>(stream)));
}

int sq_w4a16_ln_fusable(int M, int N, int K, int group_size, int layout) {
    return layout == SQ_LAYOUT_L1 && M >= 1 && M <= 8 && N > 0 && group_size == 128 && K % 128 == 0 && K > 2048 &&
                   K <= 4096
               ? 1
               : 0;
}

int sq_w4a16_gemm_ln_fused(const void* x, const void* ln_gamma, const void* ln_beta, float ln_eps, void* x_norm,
                           const void* w, const void* zs, const void* bias, const void* residual, void* y, int M, int N,
                           int K, int group_size, int layout, int act, void* workspace, size_t workspace_bytes,
                           void* stream) {
    if (act != SQ_ACT_NONE && act != SQ_ACT_RELU && act != SQ_ACT_SILU) return SQ_ERR_BAD_ALGO;
    if (bias && (reinterpret_cast<uintptr_t>(bias) & 1u)) return SQ_ERR_MISALIGNED;
    if (residual && (reinterpret_cast<uintptr_t>(residual) & 1u)) return SQ_ERR_MISALIGNED;
    if ((ln_gamma && !aligned16(ln_gamma)) || (ln_beta && !aligned16(ln_beta))) return SQ_ERR_MISALIGNED;
    if (M < 0) return SQ_ERR_BAD_SHAPE;
    const int rc = check_weight(N, K, group_size, layout);
    if (rc != SQ_OK) return rc;
    if (layout != SQ_LAYOUT_L1) return SQ_ERR_BAD_LAYOUT;
    if (M == 0) return SQ_OK;
    const sq::Epilogue epi{static_cast<const sq::half_t*>(bias), static_cast<const sq::half_t*>(residual), act};
    if (sq_w4a16_ln_fusable(M, N, K, group_size, layout)) {
        if (!x || !w || !zs || !y) return SQ_ERR_NULL_POINTER;
        if (!aligned16(x) || !aligned16(w) || !aligned16(zs) || !aligned16(y)) return SQ_ERR_MISALIGNED;
        const sq::LnPre ln{static_cast<const sq::half_t*>(ln_gamma), static_cast<const sq::half_t*>(ln_beta), ln_eps};
        const hipError_t e = sq::launch_skinny3_tuned(x, w, zs, y, nullptr, M, N, K, group_size, 0, epi, &ln,
                                                      static_cast<hipStream_t>(stream));
        if (e != hipErrorInvalidValue) return launch_code(e);
    }
    // Not fusable: the LayerNorm kernel into the caller's scratch rows, then the linear on those.
    if (!x_norm) return SQ_ERR_NULL_POINTER;
    if (K > 16384) return SQ_ERR_BAD_SHAPE;
    const int rl = sq_layernorm(x, ln_gamma, ln_beta, x_norm, M, K, ln_eps, stream);
    if (rl != SQ_OK) return rl;
    return gemm_dispatch(x_norm, w, zs, y, M, N, K, group_size, layout, SQ_ALGO_AUTO, epi, workspace, workspace_bytes,
                         stream);
}

int sq_embed_rows(const void* embed, const void* pos_table, const void* tok, const void* pos, long long pos_offset,
                  void* out, int rows, int hidden, long long vocab, long long positions, void* stream) {
    if (rows < 0 || hidden <= 0 || hidden % 8 != 0 || vocab <= 0 || positions <= 0) return SQ_ERR_BAD_SHAPE;
    if (rows == 0) return SQ_OK;
    if (!embed || !pos_table || !tok || !pos || !out) return SQ_ERR_NULL_POINTER;
    if (!aligned16(embed) || !aligned16(pos_table) || !aligned16(out) || (reinterpret_cast<uintptr_t>(tok) & 7u) ||
        (reinterpret_cast<uintptr_t>(pos) & 7u))
        return SQ_ERR_MISALIGNED;
    return launch_code(sq::launch_embed_rows(embed, pos_table, tok, pos, pos_offset, out, rows, hidden, vocab, positions,
                                             static_cast<hipStream_t>(stream)));
}

int sq_f16_gemv_parts(int N) { return N > 0 ? sq::f16_gemv_parts(N) : 0; }

int sq_f16_gemv(const void* x, const void* w, void* y, void* part_val, void* part_idx, int M, int N, int K, void* stream) {
    if (M < 0 || M > 8 || N <= 0 || K < 512 || K % 512 != 0 || K > 8192) return SQ_ERR_BAD_SHAPE;
    if (M == 0) return SQ_OK;
    if (!x || !w || !y || ((part_val == nullptr) != (part_idx == nullptr))) return SQ_ERR_NULL_POINTER;
    if (!aligned16(x) || !aligned16(w) || (reinterpret_cast<uintptr_t>(y) & 1u) ||
        (reinterpret_cast<uintptr_t>(part_val) & 3u) || (reinterpret_cast<uintptr_t>(part_idx) & 3u))
        return SQ_ERR_MISALIGNED;
    return launch_code(sq::launch_f16_gemv(x, w, y, static_cast<float*>(part_val), static_cast<int*>(part_idx), M, N, K,
                                           static_cast<hipStream_t>(stream)));
}

int sq_greedy_feedback(const void* part_val, const void* part_idx, int parts, int M, void* tok, void* pos, void* history,
                       void* step, long long history_rows, void* stream) {
    if (M < 0 || M > 8 || parts <= 0 || history_rows < 0) return SQ_ERR_BAD_SHAPE;
    if (M == 0) return SQ_OK;
    if (!part_val || !part_idx || !tok) return SQ_ERR_NULL_POINTER;
    if ((reinterpret_cast<uintptr_t>(tok) & 7u) || (reinterpret_cast<uintptr_t>(pos) & 7u) ||
        (reinterpret_cast<uintptr_t>(history) & 7u) || (reinterpret_cast<uintptr_t>(step) & 7u))
        return SQ_ERR_MISALIGNED;
    return launch_code(sq::launch_greedy_feedback(static_cast<const float*>(part_val), static_cast<const int*>(part_idx),
                                                  parts, M, tok, pos, history, step, history_rows,
                                                  static_cast<hipStream_t>(stream)));
}

}  // extern "C"
