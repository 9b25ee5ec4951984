// llg_moe_split.hip -- MoE FFN of a batch of tokens at fp32 precision as
// grouped MFMA GEMMs (inference/moe_forward.go:32-150 for every token): the
// batches that the f16 GEMM (llg_moe_gemm.hip) does not take -- Q8_0 and F16
// experts, Q4_0 experts of other widths, and a few tokens.
//
//   1. k_moe_router (llg_moe.hip)
//   2. k_moe_group_split: the (token, slot) rows of each expert in tiles of at
//      most 16 * MS rows; x as three f16 pieces per element and a power of two
//      per row and 128 columns
//   3. k_moe_split_gemm: gate and up as one matrix of 2 * eff columns, K split
//      into slices
//   4. k_moe_act_split: h = silu(gate) * up from the slices' sums, in pieces
//   5. k_moe_split_gemm: down, K split into slices
//   6. k_moe_combine (llg_moe_gemm.hip)
//
// Precision.  A quantized element is a small integer q times its block's
// scale, and q is exact in f16, as is an F16 weight.  An fp32 value scaled by
// the power of two that puts its chunk's largest magnitude into [2^14, 2^15)
// is the exact sum of three f16 pieces (11 + 11 + 2 bits) down to 2^-16 of
// that magnitude, and within 2^-40 of it below.  One v_mfma_f32_16x16x32_f16
// takes the 32 elements of one block, so the three products of a block are
// summed in one fp32 accumulator, the block's scale multiplies that sum in
// fp32, and the chunk's power of two its four blocks: no operand loses a bit
// that its sum could hold and nothing is kept in less than 32 bits.  Relative
// error of a Mixtral layer's output against 64 bits (2-norm), per-token
// kernels -> these: Q8_0, 100 tokens 6.0e-7 -> 3.1e-7; Q4_0, 7 tokens
// 5.3e-6 -> 2.9e-7; F16, 100 tokens 2.5e-7 -> 2.3e-7.
//
// Measured (Mixtral layer, 4096 x 14336, 8 experts, top-2), per-token kernels
// -> these: Q8_0, 100 tokens 5025 -> 526 us (1.50 GB of weights, 2.9 TB/s) and
// 512 tokens 14.8 -> 1.78 ms; F16, 100 tokens 11.0 -> 0.72 ms (4.0 TB/s);
// Q4_0, 9 tokens 311 -> 225 us.  With 16 rows per tile the weight stream bounds
// it, together with the unpacking (17 instructions per 16 x 32 weights and 12
// MFMA cycles that overlap it in part: 105 us of the 236 us of a Q4_0 batch of
// 7 without any weight load); with more rows the MFMAs (three per product).
//
// MFMA operands: lane l holds 8 K elements of token row l % 16 (A) and of
// weight row l % 16 (B) for K group l / 16; C lane l holds weight row l % 16,
// token rows 4 * (l / 16) .. + 3.  The weights come straight from their rows:
// a lane loads 16 bytes per instruction (four lanes one row's 64), and where
// a 16-byte load is more than the lane's part of one block the words are
// exchanged between the four 16-lane groups (v_permlane32_swap /
// v_permlane16_swap), four swaps per four blocks.  Tokens go through LDS,
// double buffered in chunks of 4 blocks.  The unpacking uses full-rate
// instructions only: with conversions (v_cvt, a quarter of the rate) to bf16
// operands it cost as much as the products.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "llg_common.hpp"
#include "llg_internal.hpp"
#include "llg_moe_group.hpp"

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

#define MS_KB 4                    // 32-element blocks per K chunk
#define MS_BU 12                   // 16-byte units of a block's three pieces
#define MS_CU (MS_KB * MS_BU)      // units of a row's chunk
#define MS_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0)
#define MS_FILL 6                  // workgroups per CU that K is split for
#define MS_PAST 0x80000000u        // byte offset past any buffer (at most 2^31 bytes)
#define MS_RST (MS_CU * 16 + 16)   // LDS bytes per row: 4 words past a bank cycle

// Position of element e of an 8-element group in the pieces: the order in
// which a Q4_0 word gives its nibble pairs (0 4 1 5 2 6 3 7), else as stored.
__device__ __forceinline__ int piece_elem(int pos, bool q4) {
    return q4 ? (pos >> 1) + 4 * (pos & 1) : pos;
}

// v [rows x 32 nb] -> per row and chunk of 4 blocks the pieces
// [block][piece][32] (f16) and the chunk's power of two; one thread per 8
// elements, 16 per chunk (blocks past nb are written as zeros).  ACT: v holds
// ks slices (vstride floats apart) of gate and up rows side by side
// ([rows x 64 nb]), and the values are silu(gate) * up of the slices' sums in
// order (moe_forward.go:128-132).  Bound by its bytes (10 per element, 14 + 8
// per further slice with ACT).
template <bool ACT>
__device__ __forceinline__ void split_unit(long long t, const float *__restrict__ v, int nb, int nc,
                                           long long n_units, int ks, long long vstride, int q4,
                                           u32x4_t *__restrict__ out, float *__restrict__ scale) {
    if (t >= n_units) return;  // n_units is a multiple of 16: chunks stay whole
    const int u = (int)(t & 15);       // 8-element group of the chunk
    const long long rc = t >> 4;       // row * nc + chunk
    const int blk = (int)(rc % nc) * MS_KB + (u >> 2);
    const bool in = blk < nb;
    const int col = min(blk, nb - 1) * 32 + (u & 3) * 8;
    auto load8 = [](const float *p, float (&o)[8]) {
        const float4 a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1];
        o[0] = a.x, o[1] = a.y, o[2] = a.z, o[3] = a.w, o[4] = b.x, o[5] = b.y, o[6] = b.z, o[7] = b.w;
    };
    float x[8];
    if constexpr (ACT) {
        const float *p = v + (rc / nc) * nb * 64 + col;
        float g[8], w[8], y[8];
        load8(p, g);
        load8(p + nb * 32, w);
        for (int s = 1; s < ks; s++) {
            load8(p + s * vstride, x);
            load8(p + s * vstride + nb * 32, y);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                g[i] += x[i];
                w[i] += y[i];
            }
        }
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = g[i] / (1.0f + (float)exp(-(double)g[i])) * w[i];
    } else {
        load8(v + (rc / nc) * nb * 32 + col, x);
    }
    uint32_t m = 0;  // largest finite magnitude
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if (!in) x[i] = 0.0f;
        const uint32_t k = __float_as_uint(x[i]) & 0x7FFFFFFFu;
        m = max(m, k < 0x7F800000u ? k : 0u);
    }
#pragma unroll
    for (int i = 1; i < 16; i <<= 1) m = max(m, (uint32_t)__shfl_xor((int)m, i, 64));
    // m in [2^e, 2^(e+1)) -> values times 2^(14 - e), at most 2^126
    const int e = max((int)(m >> 23) - 127, -112);
    const float up = __uint_as_float((uint32_t)(127 + 14 - e) << 23);
    h8_t o[3];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float y = x[piece_elem(i, q4)] * up;
        const _Float16 hi = (_Float16)y;
        // infinities and NaN stay in piece 0 alone
        const float r = fabsf(y) < INFINITY ? y - (float)hi : 0.0f;
        const _Float16 mid = (_Float16)r;
        o[0][i] = hi;
        o[1][i] = mid;
        o[2][i] = (_Float16)(r - (float)mid);
    }
    u32x4_t *d = out + rc * MS_CU + (u >> 2) * MS_BU + (u & 3);
#pragma unroll
    for (int i = 0; i < 3; i++) d[4 * i] = __builtin_bit_cast(u32x4_t, o[i]);
    if (u == 0) scale[rc] = __uint_as_float((uint32_t)(127 - 14 + e) << 23);
}

// x in pieces; workgroup 0 groups the pairs meanwhile.
__global__ __launch_bounds__(MOE_GROUP_THREADS) void k_moe_group_split(
    MoeGroupArgs ga, const float *__restrict__ x, int nb, int nc, long long n_units, int q4,
    u32x4_t *__restrict__ out, float *__restrict__ scale) {
    if (blockIdx.x == 0)
        moe_group(ga);
    else
        split_unit<false>((blockIdx.x - 1LL) * blockDim.x + threadIdx.x, x, nb, nc, n_units, 0, 0, q4,
                          out, scale);
}

// h = silu(gate) * up in pieces.
__global__ __launch_bounds__(256) void k_moe_act_split(const float *__restrict__ v, int nb, int nc,
                                                       long long n_units, int ks, long long vstride,
                                                       int q4, u32x4_t *__restrict__ out,
                                                       float *__restrict__ scale) {
    split_unit<true>((long long)blockIdx.x * blockDim.x + threadIdx.x, v, nb, nc, n_units, ks, vstride,
                     q4, out, scale);
}

__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// The weights of one lane's row for a chunk (blocks 4c .. 4c + 3): loads, the
// exchange between the lane groups, and the f16 fragment of block j.  `row` is
// the row's byte offset in the buffer r, lg the lane group.  Blocks past the
// row's end read what follows it (zeros past the buffer); their tokens are
// zeros and the caller's mask drops their scales (or F16 values).
__device__ __forceinline__ u32x4_t buf16(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}
// scale of block j of a chunk's four; masked before the conversion
__device__ __forceinline__ float chunk_scale(const u32x2_t &d, int j, uint32_t mask) {
    const h2_t p = __builtin_bit_cast(h2_t, d[j >> 1] & mask);
    return (float)p[j & 1];
}

template <int T>
struct WChunk;

template <>
struct WChunk<LLG_TYPE_Q4_0> {
    u32x4_t q;  // block 4c + lane group; after arrange(): word j = this group's of block j
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int row, int c, int lg) {
        q = buf16(r, row + lg * 16, c * (MS_KB * 16));
    }
    __device__ __forceinline__ void arrange() {
        uint32_t w0 = q[0], w1 = q[1], w2 = q[2], w3 = q[3];
        swap32(w0, w2);
        swap32(w1, w3);
        swap16(w0, w1);
        swap16(w2, w3);
        q = {w0, w1, w2, w3};
    }
    // q - 8, exact: a nibble at bits 0-3 of an f16 under 0x6400 is 1024 + q,
    // one at bits 4-7 under 0x5400 is 64 + q
    __device__ __forceinline__ h8_t frag(int j, uint32_t) const {
        const uint32_t v = q[j], v8 = v >> 8;
        const h2_t lo = {(_Float16)1032.0f, (_Float16)1032.0f}, hi = {(_Float16)72.0f, (_Float16)72.0f};
        const h2_t a = __builtin_bit_cast(h2_t, llg_and_or(v, 0x000F000Fu, 0x64006400u)) - lo;
        const h2_t b = __builtin_bit_cast(h2_t, llg_and_or(v, 0x00F000F0u, 0x54005400u)) - hi;
        const h2_t c = __builtin_bit_cast(h2_t, llg_and_or(v8, 0x000F000Fu, 0x64006400u)) - lo;
        const h2_t e = __builtin_bit_cast(h2_t, llg_and_or(v8, 0x00F000F0u, 0x54005400u)) - hi;
        return h8_t{a[0], a[1], b[0], b[1], c[0], c[1], e[0], e[1]};
    }
    // K group of the lane's elements inside a block
    static __device__ __forceinline__ int group(int lg) { return lg; }
};

template <>
struct WChunk<LLG_TYPE_Q8_0> {
    u32x4_t q[2];  // 64 bytes (2 blocks) over the 4 lane groups, twice
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int row, int c, int lg) {
#pragma unroll
        for (int h = 0; h < 2; h++) q[h] = buf16(r, row + lg * 16 + h * 64, c * (MS_KB * 32));
    }
    // words 0, 1 of q[h] become block 2h's, words 2, 3 block 2h + 1's: groups
    // 0 .. 3 then hold its 8-element groups 0, 2, 1, 3
    __device__ __forceinline__ void arrange() {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t a = q[h][0], b = q[h][1], e = q[h][2], g = q[h][3];
            swap32(a, e);
            swap32(b, g);
            q[h] = {a, b, e, g};
        }
    }
    // q, exact: the byte q + 128 under 0x6400 is the f16 1152 + q
    __device__ __forceinline__ h8_t frag(int j, uint32_t) const {
        const h2_t off = {(_Float16)1152.0f, (_Float16)1152.0f};
        h2_t p[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t v = q[j >> 1][2 * (j & 1) + (i >> 1)] ^ 0x80808080u;
            p[i] = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, v, i & 1 ? 0x07030702u
                                                                                        : 0x07010700u)) - off;
        }
        return h8_t{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
    }
    static __device__ __forceinline__ int group(int lg) {
        return ((lg & 1) << 1) | (lg >> 1);
    }
};

template <>
struct WChunk<LLG_TYPE_F16> {
    u32x4_t q[MS_KB];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int row, int c, int lg) {
#pragma unroll
        for (int j = 0; j < MS_KB; j++) q[j] = buf16(r, row + lg * 16 + j * 64, c * (MS_KB * 64));
    }
    __device__ __forceinline__ void arrange() {}
    __device__ __forceinline__ h8_t frag(int j, uint32_t mask) const {
        return __builtin_bit_cast(h8_t, q[j] & mask);
    }
    static __device__ __forceinline__ int group(int lg) { return lg; }
};

// Slice ks of K of A_e . W_e^T to Y + ks * ystride ([row][N] fp32).  GATHER:
// A's row is the pair's token, and the N columns are those of W0 and then W1
// (gate and up); else A's row is the pair's own, of W0 (down).
// Workgroup: one tile of at most 16 * MS rows x 4 wavefronts of NF 16-column
// groups.  blockIdx = (N tile * n_mt + M tile) * ksplit + slice: the tiles of
// one expert that stream the same weights run side by side.
template <int T, bool GATHER, int MS, int NF>
__global__ __launch_bounds__(256, MS == 1 ? 3 : 2) void k_moe_split_gemm(
    const int4 *__restrict__ tiles, const int32_t *__restrict__ n_tiles_p, int n_mt,
    const int32_t *__restrict__ row_pair, int k_slots, const u32x4_t *__restrict__ A,
    uint32_t a_bytes, const float *__restrict__ a_scale, const uint8_t *__restrict__ W0,
    const uint8_t *__restrict__ W1, RowFmt f, int rows_per_expert, int N, float *__restrict__ Y,
    int ksplit, long long ystride) {
    __shared__ __attribute__((aligned(16))) uint8_t As[2][16 * MS * MS_RST];
    __shared__ __attribute__((aligned(16))) float Sc[2][16 * MS];
    const int ks = blockIdx.x % ksplit;
    const int mt = (blockIdx.x / ksplit) % n_mt;
    const int nt = blockIdx.x / ksplit / n_mt;
    if (mt >= *n_tiles_p) return;
    const int4 tile = tiles[mt];
    const int e = tile.x, row0 = tile.y, nrows = tile.z;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = (nt * 4 + wave) * NF * 16;
    const int li = lane & 15, lg = lane >> 4;

    // a body per count of 16-row groups, as in k_moe_gemm
    auto body = [&](auto nms_c) __attribute__((always_inline)) {
        constexpr int NMS = decltype(nms_c)::value;
        static_assert(NMS <= MS && MS <= 2, "tiles of 16 or 32 rows");
        constexpr int NA = 16 * NMS * MS_CU / 256;  // 16-byte units a thread stages per chunk
        const int nc = (f.nb + MS_KB - 1) / MS_KB;
        const int c0 = (int)((long long)nc * ks / ksplit), ce = (int)((long long)nc * (ks + 1) / ksplit);
        const int nbe = min(f.nb, ce * MS_KB);  // the slice's last block + 1
        auto arow = [&](int r) __attribute__((always_inline)) {
            const int rr = row0 + min(r, nrows - 1);
            return GATHER ? row_pair[rr] / k_slots : rr;
        };
        // Rows past the tile point past the buffer: such a load returns zeros
        // and moves nothing.
        int a_off[NA];
#pragma unroll
        for (int q = 0; q < NA; q++) {
            const int idx = tid + 256 * q, r = idx / MS_CU;
            a_off[q] = r < nrows ? (int)(((uint32_t)arow(r) * nc * MS_CU + idx % MS_CU) * 16u) : (int)MS_PAST;
        }
        // the rows' powers of two (a plain load was moved under the store's
        // condition, where it waited for every load in flight)
        const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(a_scale), 0, (int)(a_bytes / (MS_CU * 4)), 0x00027000);
        const int s_off = arow(tid & (16 * NMS - 1)) * nc * 4;
        // group i of the wavefront: 16 rows of the expert's matrix from ncol(i)
        // on (groups past N reload the last one and are dropped)
        const int w_bytes = (int)(f.stride * rows_per_expert);
        const long long w_off = (long long)e * w_bytes;
        __amdgpu_buffer_rsrc_t wr[NF];
        int brow[NF];
#pragma unroll
        for (int i = 0; i < NF; i++) {
            const int n = min(n0 + i * 16, N - 16);
            const bool second = GATHER && n >= rows_per_expert;
            wr[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>((second ? W1 : W0) + w_off), 0,
                                                      w_bytes, 0x00027000);
            brow[i] = (int)((n - (second ? rows_per_expert : 0) + li) * f.stride);
        }
        // Tokens and weights are requested one chunk ahead (three ahead, in
        // four slots, measured no gain: 239 -> 249 us for a Q4_0 batch of 7).
        u32x4_t ra[NA];
        float rs;
        WChunk<T> wb[2][NF];
        // Block scales of four chunks at a time: lane group g loads those of
        // chunk c + g, so a row's 32 bytes are one request.  Loaded per chunk
        // (8 bytes of a line each time) they took as many requests as the
        // quants: 286 -> 239 us for a Q4_0 batch of 7.
        u32x2_t dq[2][NF];
        auto load_d = [&](int c, int slot) __attribute__((always_inline)) {
            if constexpr (T != LLG_TYPE_F16)
#pragma unroll
                for (int i = 0; i < NF; i++)
                    dq[slot][i] = __builtin_amdgcn_raw_buffer_load_b64(
                        wr[i], brow[i] + f.d_off + lg * (MS_KB * 2), min(c, nc - 1) * (MS_KB * 2), 0);
        };
        auto load_a = [&](int c) __attribute__((always_inline)) {
            // a chunk past the slice: no buffer, zeros
            const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<u32x4_t *>(A), 0, c < ce ? (int)a_bytes : 0, 0x00027000);
#pragma unroll
            for (int q = 0; q < NA; q++) ra[q] = buf16(ar, a_off[q], c * (MS_CU * 16));
            rs = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(sr, s_off, min(c, nc - 1) * 4, 0));
        };
        auto load_b = [&](int c, int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NF; i++) wb[slot][i].load(wr[i], brow[i], min(c, nc - 1), lg);
        };
        auto store_a = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < NA; q++) {
                const int idx = tid + 256 * q;
                *reinterpret_cast<u32x4_t *>(&As[buf][(idx / MS_CU) * MS_RST + (idx % MS_CU) * 16]) = ra[q];
            }
            Sc[buf][tid & (16 * NMS - 1)] = rs;  // every copy is the same value
        };
        f32x4_t acc[NF][NMS];
#pragma unroll
        for (int i = 0; i < NF; i++)
#pragma unroll
            for (int m = 0; m < NMS; m++) acc[i][m] = {0.f, 0.f, 0.f, 0.f};

        load_d(c0, 0);
        load_a(c0);
        load_b(c0, 0);
        store_a(0);
        __syncthreads();
        const int ga = li * MS_RST + WChunk<T>::group(lg) * 16;
        // i: the chunk's place in the unrolled eight
        auto chunk = [&](int c, int i8) __attribute__((always_inline)) {
            const int g = i8 & 3, slot = i8 >> 2, buf = i8 & 1;
            load_a(c + 1);
            if (g == 0) load_d(c + 4, slot ^ 1);
            load_b(c + 1, buf ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            u32x2_t d[NF];
            if constexpr (T != LLG_TYPE_F16)
#pragma unroll
                for (int i = 0; i < NF; i++)
#pragma unroll
                    for (int h = 0; h < 2; h++)
                        d[i][h] = (uint32_t)__builtin_amdgcn_ds_bpermute(li * 4 + 64 * g, (int)dq[slot][i][h]);
            // the chunk's sums are formed first, then added to the running
            // sums: a short chain of additions each (F16: those of the
            // smaller pieces apart, so that they round at their own size)
            f32x4_t tc[NF][NMS], tl[NF][NMS];
#pragma unroll
            for (int i = 0; i < NF; i++)
#pragma unroll
                for (int m = 0; m < NMS; m++) {
                    tc[i][m] = {0.f, 0.f, 0.f, 0.f};
                    tl[i][m] = {0.f, 0.f, 0.f, 0.f};
                }
            h8_t a[2][NMS][3];
            auto read_a = [&](int j) __attribute__((always_inline)) {
#pragma unroll
                for (int m = 0; m < NMS; m++)
#pragma unroll
                    for (int p = 0; p < 3; p++)
                        a[j & 1][m][p] = *reinterpret_cast<const h8_t *>(
                            &As[buf][ga + m * 16 * MS_RST + j * (MS_BU * 16) + p * 64]);
            };
            if (NMS == 1) read_a(0);
#pragma unroll
            for (int i = 0; i < NF; i++) wb[buf][i].arrange();
#pragma unroll
            for (int j = 0; j < MS_KB; j++) {
                const uint32_t mask = MS_KB * c + j < nbe ? 0xFFFFFFFFu : 0u;
                // the next block's tokens early where the registers allow it
                if (NMS == 1) {
                    if (j + 1 < MS_KB) read_a(j + 1);
                } else {
                    read_a(j);
                }
                auto &aj = a[j & 1];
#pragma unroll
                for (int i = 0; i < NF; i++) {
                    const h8_t w = wb[buf][i].frag(j, mask);
                    if constexpr (T == LLG_TYPE_F16) {
                        // for the smaller pieces infinities and NaN are made
                        // finite (an infinity times a zero piece would be NaN)
                        const h8_t big = (_Float16)65504.0f;
                        const h8_t wc = __builtin_elementwise_max(__builtin_elementwise_min(w, big), -big);
#pragma unroll
                        for (int m = 0; m < NMS; m++) {
                            tl[i][m] = MS_MFMA(aj[m][2], wc, tl[i][m]);
                            tl[i][m] = MS_MFMA(aj[m][1], wc, tl[i][m]);
                            tc[i][m] = MS_MFMA(aj[m][0], w, tc[i][m]);
                        }
                    } else {
                        const float ds = chunk_scale(d[i], j, mask);
#pragma unroll
                        for (int m = 0; m < NMS; m++) {
                            f32x4_t t = {0.f, 0.f, 0.f, 0.f};
                            t = MS_MFMA(aj[m][2], w, t);
                            t = MS_MFMA(aj[m][1], w, t);
                            t = MS_MFMA(aj[m][0], w, t);
#pragma unroll
                            for (int v = 0; v < 4; v++) tc[i][m][v] = __builtin_fmaf(ds, t[v], tc[i][m][v]);
                        }
                    }
                }
                // one block at a time: moved across blocks, the products that
                // wait for their scale filled the registers and spilled
#pragma unroll
                for (int i = 0; i < NF; i++)
#pragma unroll
                    for (int m = 0; m < NMS; m++) asm volatile("" : "+v"(tc[i][m]));
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int m = 0; m < NMS; m++) {
                const f32x4_t sc = *reinterpret_cast<const f32x4_t *>(&Sc[buf][m * 16 + 4 * lg]);
#pragma unroll
                for (int i = 0; i < NF; i++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const float t = T == LLG_TYPE_F16 ? tc[i][m][v] + tl[i][m][v] : tc[i][m][v];
                        acc[i][m][v] = __builtin_fmaf(t, sc[v], acc[i][m][v]);
                    }
            }
            store_a(buf ^ 1);
            __syncthreads();
        };
        // F16: the running sums of eight chunks are added to the total (with
        // one chain, the error was 10-25% above the per-token kernels')
        f32x4_t tot[NF][NMS];
        if constexpr (T == LLG_TYPE_F16)
#pragma unroll
            for (int i = 0; i < NF; i++)
#pragma unroll
                for (int m = 0; m < NMS; m++) tot[i][m] = {0.f, 0.f, 0.f, 0.f};
        for (int c = c0;; c += 8) {
            bool more = true;
#pragma unroll
            for (int i = 0; i < 8 && more; i++) {
                chunk(c + i, i);
                more = c + i + 1 < ce;
            }
            if constexpr (T == LLG_TYPE_F16)
#pragma unroll
                for (int i = 0; i < NF; i++)
#pragma unroll
                    for (int m = 0; m < NMS; m++) {
                        tot[i][m] += acc[i][m];
                        acc[i][m] = {0.f, 0.f, 0.f, 0.f};
                    }
            if (!more) break;
        }

        float *y = Y + ks * ystride + (long long)row0 * N + n0 + li;
#pragma unroll
        for (int m = 0; m < NMS; m++)
#pragma unroll
            for (int i = 0; i < NF; i++) {
                if (n0 + i * 16 >= N) break;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int r = m * 16 + lg * 4 + v;
                    if (r < nrows) y[(long long)r * N + i * 16] = T == LLG_TYPE_F16 ? tot[i][m][v] : acc[i][m][v];
                }
            }
    };
    if constexpr (MS == 1) {
        body(std::integral_constant<int, 1>{});
    } else {
        if (nrows <= 16)
            body(std::integral_constant<int, 1>{});
        else
            body(std::integral_constant<int, 2>{});
    }
}

// ---------------------------------------------------------------------------
// Rows per tile: 16 while no expert can hold more (a token's slots are
// different experts), else 32.
static int split_ms(int n_tok) { return n_tok <= 16 ? 1 : 2; }

// K slices of a GEMM of n_tiles row tiles over `cols` output columns and a K of
// `kcols`: enough workgroups to fill the chip MS_FILL times, each slice at
// least 4 chunks.
static int split_ks(int cus, int n_tiles, int cols, int kcols) {
    const int nc = (kcols / 32 + MS_KB - 1) / MS_KB;
    const long long wgs = (long long)n_tiles * ((cols + 255) / 256);
    int ks = 1;
    while (ks < 8 && wgs * ks < (long long)MS_FILL * cus && nc / (ks * 2) >= 4) ks *= 2;
    return ks;
}

// Bytes of the pieces and of the scales of [rows x cols] values.
static long long split_chunks(int cols) { return (cols / 32 + MS_KB - 1) / MS_KB; }
static long long split_piece_bytes(long long rows, int cols) {
    return llg_align(rows * split_chunks(cols) * MS_CU * 16, 256);
}
static long long split_scale_bytes(long long rows, int cols) {
    return llg_align(rows * split_chunks(cols) * 4, 256);
}

// Upper bound of the tile count.
static long long split_nt_max(int n_tok, int k, int n_exp) {
    const long long np = (long long)n_tok * k;
    return std::min<long long>(np, np / (16 * split_ms(n_tok)) + n_exp);
}

size_t llg_moe_split_ws_bytes(int cus, int n_tok, int k, int n_exp, int hidden, int eff) {
    const long long np = (long long)n_tok * k, nt = split_nt_max(n_tok, k, n_exp);
    const int kg = split_ks(cus, (int)nt, 2 * eff, hidden), kd = split_ks(cus, (int)nt, hidden, eff);
    return (size_t)(llg_align(np * 4, 256) * 2 + llg_align(nt * 16, 256) + 256 +
                    split_piece_bytes(n_tok, hidden) + split_scale_bytes(n_tok, hidden) +
                    split_piece_bytes(np, eff) + split_scale_bytes(np, eff) +
                    std::max(kg * llg_align(np * eff * 8, 256), kd * llg_align(np * hidden * 4, 256)));
}

// Whether a batch takes this path.  The per-token kernels stream an expert's
// rows once per (token, slot) pair at up to 6 TB/s (the repeats come from the
// caches); this path once per hit expert at 3 - 5 TB/s, and has two launches
// more.  So it needs two pairs per expert that the batch is expected to hit
// (Mixtral layer, per-token -> here: Q4_0 5 tokens (1.6 pairs) 192 -> 232 us,
// 9 tokens (2.4) 311 -> 225 us; Q8_0 5 tokens 330 -> 327 us; F16 3 tokens
// (1.3) 392 -> 400 us), and enough weight bytes to pay for the launches
// (8 experts of 512 x 512, 8 tokens: 21 -> 30 us).
bool llg_moe_split_use(const LlgObject *gate, const LlgObject *down, int hidden, int eff, int n_tok,
                       int k, int n_exp) {
    if (gate->fmt.type == LLG_TYPE_F32) return false;
    const long long np = (long long)n_tok * k, nt = split_nt_max(n_tok, k, n_exp);
    const double hit = n_exp * (1.0 - pow(1.0 - (double)k / n_exp, n_tok));
    if ((double)np < 2.0 * hit) return false;
    const long long expert = 2 * gate->fmt.stride * eff + down->fmt.stride * hidden;
    if (n_tok < 16 && np * expert < (32LL << 20)) return false;
    // 31-bit byte offsets into the pieces and an expert's rows, and grid sizes
    const long long lim = 1LL << 31;
    return split_piece_bytes(np, eff) < lim && split_piece_bytes(n_tok, hidden) < lim &&
           gate->fmt.stride * eff < lim && down->fmt.stride * hidden < lim &&
           nt * ((2LL * eff + 31) / 32) * 8 < lim && nt * ((hidden + 31) / 32) * 8 < lim;
}

int llg_moe_split_enqueue(LlgDevice *d, const LlgObject *gate, const LlgObject *up,
                          const LlgObject *down, int n_exp, int k, int hidden, int eff,
                          const float *d_x, int n_tok, const int32_t *ids, const float *w,
                          float *d_out, uint8_t *ws) {
    hipStream_t st = llg_dev_stream(d);
    const long long np = (long long)n_tok * k;
    const int nt = (int)split_nt_max(n_tok, k, n_exp);
    const int cus = llg_cu_count(d);
    const int kg = split_ks(cus, nt, 2 * eff, hidden), kd = split_ks(cus, nt, hidden, eff);
    const int type = gate->fmt.type;
    uint8_t *p = ws;
    auto take = [&](long long bytes) {
        uint8_t *q = p;
        p += llg_align(bytes, 256);
        return q;
    };
    int32_t *row_pair = reinterpret_cast<int32_t *>(take(np * 4));
    int32_t *pair_row = reinterpret_cast<int32_t *>(take(np * 4));
    int4 *tiles = reinterpret_cast<int4 *>(take(nt * 16LL));
    int32_t *n_tiles = reinterpret_cast<int32_t *>(take(256));
    const long long xb = split_piece_bytes(n_tok, hidden), hb = split_piece_bytes(np, eff);
    u32x4_t *x3 = reinterpret_cast<u32x4_t *>(take(xb));
    float *xs = reinterpret_cast<float *>(take(split_scale_bytes(n_tok, hidden)));
    u32x4_t *h3 = reinterpret_cast<u32x4_t *>(take(hb));
    float *hs = reinterpret_cast<float *>(take(split_scale_bytes(np, eff)));
    float *Y = reinterpret_cast<float *>(p);  // the slices of gate and up, then of down
    const long long gstride = llg_align(np * eff * 8, 256) / 4, ystride = llg_align(np * hidden * 4, 256) / 4;

    const MoeGroupArgs ga = {ids, (int)np, n_exp, 16 * split_ms(n_tok), row_pair, pair_row, tiles, n_tiles};
    const int q4 = type == LLG_TYPE_Q4_0 ? 1 : 0;
    const int nbx = hidden / 32, ncx = (int)split_chunks(hidden), nbh = eff / 32, nch = (int)split_chunks(eff);
    const long long nx = (long long)n_tok * ncx * 16, nh = np * nch * 16;  // 8-element groups
    hipLaunchKernelGGL(k_moe_group_split,
                       dim3((unsigned)((nx + MOE_GROUP_THREADS - 1) / MOE_GROUP_THREADS + 1)),
                       dim3(MOE_GROUP_THREADS), 0, st, ga, d_x, nbx, ncx, nx, q4, x3, xs);
    auto launch = [&](auto t, auto ms, auto nf) {
        constexpr int T = decltype(t)::value, MS = decltype(ms)::value, NF = decltype(nf)::value;
        const int nw = 4 * NF * 16;  // columns of a workgroup
        hipLaunchKernelGGL((k_moe_split_gemm<T, true, MS, NF>),
                           dim3((unsigned)(nt * ((2 * eff + nw - 1) / nw) * kg)), dim3(256), 0, st, tiles,
                           n_tiles, nt, row_pair, k, x3, (uint32_t)xb, xs, gate->d, up->d, gate->fmt,
                           eff, 2 * eff, Y, kg, gstride);
        hipLaunchKernelGGL(k_moe_act_split, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, st, Y, nbh,
                           nch, nh, kg, gstride, q4, h3, hs);
        hipLaunchKernelGGL((k_moe_split_gemm<T, false, MS, NF>),
                           dim3((unsigned)(nt * ((hidden + nw - 1) / nw) * kd)), dim3(256), 0, st,
                           tiles, n_tiles, nt, row_pair, k, h3, (uint32_t)hb, hs, down->d,
                           (const uint8_t *)nullptr, down->fmt, hidden, hidden, Y, kd, ystride);
    };
    auto launch_t = [&](auto t) {
        constexpr int NF = decltype(t)::value == LLG_TYPE_F16 ? 2 : 4;
        if (split_ms(n_tok) == 1)
            launch(t, std::integral_constant<int, 1>{}, std::integral_constant<int, 2>{});
        else
            launch(t, std::integral_constant<int, 2>{}, std::integral_constant<int, NF>{});
    };
    if (type == LLG_TYPE_Q4_0)
        launch_t(std::integral_constant<int, LLG_TYPE_Q4_0>{});
    else if (type == LLG_TYPE_Q8_0)
        launch_t(std::integral_constant<int, LLG_TYPE_Q8_0>{});
    else
        launch_t(std::integral_constant<int, LLG_TYPE_F16>{});
    llg_moe_combine_launch(st, Y, pair_row, w, k, n_tok, hidden, kd, ystride, d_out);
    LLG_LAUNCH_CHECK(d, "moe split gemm");
    return 0;
}
