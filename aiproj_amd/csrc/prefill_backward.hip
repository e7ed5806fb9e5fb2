// Backward of the varlen causal prompt attention on the gfx950 matrix cores.
//
// Replaces the Triton backward of reference src/torch_llm/kernals/flash_attention.py:213
// onwards (dq, dk, dv of packed causal attention from the saved output and lse). With
// S = scale Q K^T, P = exp(S - lse), dP = dO V^T and delta = rowsum(dO O):
//   dV = P^T dO,   dS = P (dP - delta),   dQ = scale dS K,   dK = scale dS^T Q,
// dK and dV summed over the q heads of a KV head.
//
// Precision. Products are those of float32: the matrix cores multiply bf16 values exactly
// and add in float32, and a float32 factor enters as the sum of three bf16 values (`split3`:
// nothing is lost). bf16 inputs are one such plane, float16 inputs two, float32 inputs three
// (`split_planes_kernel`); P and dS, computed in float32, are always three. Products of planes
// i and j with i + j > 2 are left out: none for bf16 inputs, else two of at most 2^-25 of
// their product each (parts to nearest), of either sign.
// Measured against 64 bits, float32 inputs, 8q/2kv heads, D 64, sequences of 40 to 700 (dk and
// dv): PyTorch's float32 operations 4.5e-7 and 4.0e-7, this kernel 2.4e-7 and 2.2e-7; inputs
// of one sign 2.1e-7 and 1.2e-7, this kernel 1.1e-7 and 0.8e-7 (with truncated parts 1.4e-6
// and 4.1e-7: the products left out are then up to 2^-22, all of the sign of the product).
//
// Bound: instruction issue on the matrix cores and the vector ALU. Per pair of tiles with
// bf16 inputs: one product each for S and dP in either pass, three for each gradient; the
// vector ALU takes about as long (exponents and splits). By counters at 16 sequences of 1024
// tokens (16q/4kv heads, D 128) the matrix cores are busy half the time.
//
// Work split. All passes are one launch. An item is a block of "own" rows (64 keys for dK
// and dV, 16 queries of up to 4 heads for dQ) of one sequence and KV head; a wave keeps the
// operands and accumulators of 16 own rows in registers (161 VGPRs at D 128, so three
// workgroups of four waves share a CU and one's vector work overlaps another's products),
// and blocks of 32 streamed rows (keys for dQ; queries of the KV head's q heads for dK, dV)
// pass through LDS, triple buffered by direct global-to-LDS loads. The gradient is
// accumulated transposed, acc^T[d, own] += X^T[d, row] W[row, own], so P or dS is used as the
// B operand straight from the registers the score product left it in, and X^T comes from
// the transposing LDS read ds_read_b64_tr_b16. No pass needs atomics: results do not depend
// on timing. The heavy items (first key blocks, which every later query attends) are
// dispatched first and the dQ items fill in behind them.
//
// Measured (bf16, 16q/4kv heads, D 128; the launch alone unless stated): 16 ragged sequences
// of 64 to 1024 tokens, the whole backward 6.75 ms as float32 PyTorch operations per
// sequence -> 0.29 ms. 64 sequences of 1024 tokens, whole backward 2.0 ms (344 TFLOP/s of the
// five products). Other shapes of the same kernel at 16 sequences of 1024 (saturated) and at
// the ragged 16: 32 own rows per wave with two waves per SIMD 529 / 340 us; 16 own rows, dK
// and dV as separate passes, four waves per SIMD 521 / 330; dK and dV in different waves of a
// workgroup 543 / 351; fused with eight waves of one workgroup per CU 613 / 457; this one 503
// / 269.
#include "mfma_tiles.h"

namespace kvfp8 {

namespace {

// Workgroups go round-robin over the eight XCDs, so consecutive own blocks of one unit
// would all land on one XCD, and the XCD that got the longest sequences would end last. The
// units of every second block are turned by half a round (16 ragged sequences of 64 to 1024
// tokens, 16q/4kv heads, D 128, bf16: 347 -> 269 us in one order of the sequences, 264 ->
// 264 in sorted order).
constexpr int kRotate = 4;

struct BwdArgs {
    // bf16 planes of the inputs, each [plane][token][head][dp].
    const uint8_t* q;
    const uint8_t* k;
    const uint8_t* v;
    const uint8_t* dout;
    int64_t q_plane, kv_plane;     // bytes between planes
    const float* lse2;             // [Hq][T], log2 units (natural for float32 inputs)
    const float* delta;            // [Hq][T]
    void* dq;
    void* dk;
    void* dv;
    int32_t type;                  // of dq, dk, dv (kvfp8_dtype)
    const void* cu;
    int32_t cu64;
    int32_t batch, hq, hkv, d;     // d: the caller's head size (<= the kernel's)
    int32_t heads_per_block;       // dQ: q heads per workgroup (4, 2 or 1, dividing G)
    int32_t q_blocks;              // dQ: own blocks of a longest sequence
    int32_t max_len;
    int64_t total_tokens;
    int64_t key_items;             // items of the dK and dV pass
    float scale, scale_log2;
    int32_t splits;                // dK, dV: workgroups that share a KV head's q heads
    float* part;                   // their sums [dK, dV][split][T][Hkv][d] when splits > 1
};

// x as three bf16 values, hi + mid + lo = x exactly (|x| above some 1e-33, so that every part is
// a normal number); the parts of two floats share a dword. Truncated (kNearest false): the parts have x's sign and reach 2^-7 and 2^-15 of it,
// for one-plane inputs, where every product is added up. To nearest: 2^-8 and 2^-17, of either
// sign, for inputs of several planes, where some products are left out. Infinite x has itself
// as its first part and NaN as the others: gradients it enters are not finite in any form, and
// scores are read off the first parts.
template <bool kNearest>
__device__ __forceinline__ void split3(float x0, float x1, u32x4_t (&out)[3], int dword) {
    float r0 = x0, r1 = x1;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        const uint32_t b0 = f32_bits(r0), b1 = f32_bits(r1);
        const uint32_t two = kNearest ? pack2<false>(r0, r1) : __builtin_amdgcn_perm(b1, b0, 0x07060302u);
        out[p][dword] = two;
        if (p < 2) {
            r0 -= bits_f32(kNearest ? two << 16 : b0 & 0xFFFF0000u);
            r1 -= bits_f32((kNearest ? two : b1) & 0xFFFF0000u);
        }
    }
}

// D: head size of the planes (64, 96 or 128); NP: input planes.
template <int D, int NP>
struct BwdShape {
    static constexpr int kWaves = NP != 2 ? 4 : 8;
    static constexpr int kWavesPerSimd = NP == 3 ? 1 : (NP == 2 ? 2 : 3);
    static constexpr int kHalves = NP != 2 ? 1 : 2;             // dK, dV: waves that share keys
    static constexpr int kKeyGroups = kWaves / kHalves;
    static constexpr int kRows = 32 * kHalves;                  // streamed rows per block
    static constexpr int kBufs = NP == 2 ? 2 : 3;
    static constexpr int kChunks = D / 8;                       // 16-byte chunks of a row
    static constexpr int kPitch = D <= 64 ? 8 : 16;             // chunk slots of a row in LDS
    static constexpr int kTensorBytes = kRows * kPitch * 16;    // one plane of one streamed tensor
    static constexpr int kBufBytes = 2 * NP * kTensorBytes;
    static constexpr int kStatBytes = 2 * 64 * 4;               // lse and delta of a block's rows
    static constexpr int kLds = kBufs * (kBufBytes + kStatBytes);
};

template <int D, int NP, bool kDq>
__device__ __forceinline__ void bwd_item(const BwdArgs& a, int64_t item, uint8_t* lds) {
    using Sh = BwdShape<D, NP>;
    constexpr int OW = 16, SR = Sh::kRows, BUFS = Sh::kBufs;
    constexpr int KS = D / 32, NB = D / 16, CH = Sh::kChunks, PITCH = Sh::kPitch;
    constexpr int ROW = PITCH * 16, TB = Sh::kTensorBytes;
    constexpr int KG = Sh::kKeyGroups, WAVES = Sh::kWaves, THREADS = 64 * WAVES;
    constexpr int GRADS = kDq ? 1 : 2;                          // dQ, or dK and dV

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int m16 = lane & 15, j = lane >> 4;
    const int G = a.hq / a.hkv;

    // The item's own rows.
    int b, hk, own_wg, own0, own_head, split = 0;
    if constexpr (kDq) {
        const int gw = a.heads_per_block, bpk = G / gw;
        const int64_t units = (int64_t)a.batch * a.hkv * bpk;
        const int blk = a.q_blocks - 1 - (int)(item / units);  // longest first
        const int64_t unit = (item + kRotate * (blk & 1)) % units;
        b = (int)(unit / (a.hkv * bpk));
        const int rest = (int)(unit % (a.hkv * bpk));
        hk = rest / bpk;
        const int rows = OW * WAVES / gw;
        own_wg = blk * rows;
        own0 = own_wg + OW * (wave / gw);
        own_head = hk * G + (rest % bpk) * gw + wave % gw;
    } else {
        const int64_t units = (int64_t)a.batch * a.hkv * a.splits;
        const int blk = (int)(item / units);                    // longest first
        int64_t unit = (item + kRotate * (blk & 1)) % units;
        split = (int)(unit / ((int64_t)a.batch * a.hkv));
        unit -= (int64_t)split * a.batch * a.hkv;
        b = (int)(unit / a.hkv);
        hk = (int)(unit % a.hkv);
        own_wg = blk * OW * KG;
        own0 = own_wg + OW * (wave % KG);
        own_head = hk;
    }
    int64_t s0, s1;
    seq_bounds(a.cu, a.cu64, b, a.total_tokens, &s0, &s1);
    int64_t len64 = s1 > s0 ? s1 - s0 : 0;
    len64 = len64 < a.max_len ? len64 : a.max_len;
    const int L = (int)len64;
    if (own_wg >= L) return;                                    // whole workgroup

    const int64_t q_row = (int64_t)a.hq * D * 2, kv_row = (int64_t)a.hkv * D * 2;
    const int64_t str_row = kDq ? kv_row : q_row, own_row = kDq ? q_row : kv_row;
    const int64_t str_plane = kDq ? a.kv_plane : a.q_plane, own_plane = kDq ? a.q_plane : a.kv_plane;
    const uint8_t* const str1 = kDq ? a.k : a.q;
    const uint8_t* const str2 = kDq ? a.v : a.dout;
    const uint8_t* const own1p = kDq ? a.q : a.k;
    const uint8_t* const own2p = kDq ? a.dout : a.v;

    // Streamed blocks: first .. first + blocks - 1, of each of `heads` heads.
    int first, blocks, heads;
    if constexpr (kDq) {
        first = 0;
        blocks = (min(L, own_wg + OW * WAVES / a.heads_per_block) + SR - 1) / SR;
        heads = 1;
    } else {
        first = own_wg / SR;
        blocks = (L + SR - 1) / SR - first;
        heads = G / a.splits;
    }
    const int steps = blocks * heads;

    typedef __attribute__((address_space(3))) void* lds_ptr;
    typedef __attribute__((address_space(3))) const uint8_t lds_u8;
    typedef __attribute__((address_space(3))) const u32x4_t lds_u32x4;
    typedef __attribute__((address_space(3))) const f32x4_t lds_f32x4;
    typedef short s16x4_t __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)lds;
    const uint32_t stat0 = lds0 + BUFS * Sh::kBufBytes;

    // Loads of a streamed block into buffer `buf`, the same number by every wave. Chunk slot
    // c = thread + THREADS i of the buffer ([tensor][plane][row][slot]) holds chunk
    // slot ^ (row % PITCH) of its row: the xor spreads the 16 rows that an operand read
    // touches over the bank groups. Rows past the sequence read its last row (masked
    // below). They are inline assembly because the compiler would otherwise wait for every
    // load in flight before any LDS read; the waits at the end of each step cover them. m0
    // is written in the same statement.
    constexpr int CPT = 2 * NP * SR * PITCH / THREADS;
    constexpr int LOADS = CPT + (kDq ? 0 : 1);                  // vector-memory instructions per block
    const int c_row = threadIdx.x / PITCH;
    const int c_chunk = (threadIdx.x % PITCH) ^ (c_row % PITCH);
    static_assert((THREADS / PITCH) % PITCH == 0 && CPT > 0, "one chunk index for all of a thread's rows");
    auto load_block = [&](int head, int blk, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            // Rows of both tensors' planes, numbered through: 32 per plane, wave-uniform plane.
            const int part_row = c_row + (THREADS / PITCH) * i;
            const int part = __builtin_amdgcn_readfirstlane(part_row / SR);
            const int row = min(blk * SR + part_row % SR, L - 1);
            const uint8_t* base = (part < NP ? str1 : str2) + (part < NP ? part : part - NP) * str_plane;
            const uint8_t* g = base + (s0 + row) * str_row + (int64_t)head * D * 2 + 16 * c_chunk;
            const uint32_t at = lds0 + (uint32_t)buf * Sh::kBufBytes + 16u * (uint32_t)(THREADS * i + 64 * wave);
            if (CH == PITCH || c_chunk < CH)
                __asm__ volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off"
                                 :: "s"(__builtin_amdgcn_readfirstlane(at)), "v"(g) : "memory");
        }
        if constexpr (!kDq) {
            // Row statistics of the block: even waves the lse, odd waves delta (each wave
            // writes the same 64 values; those past the block's rows are not read).
            const int row = min(blk * SR + lane, L - 1);
            const float* g = (wave & 1 ? a.delta : a.lse2) + (int64_t)head * a.total_tokens + s0 + row;
            const uint32_t at = stat0 + (uint32_t)buf * Sh::kStatBytes + 256u * (uint32_t)(wave & 1);
            __asm__ volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off"
                             :: "s"(__builtin_amdgcn_readfirstlane(at)), "v"(g) : "memory");
        }
    };

    // Own operands: lane (row m16, j) holds dims 32 s + 8 j .. + 7; rows past the
    // sequence read its last row (their results are not stored).
    u32x4_t own1[KS][NP], own2[KS][NP];
    float own_lse = 0.0f, own_delta = 0.0f;
    {
        const int row = min(own0 + m16, L - 1);
        const int64_t off = (s0 + row) * own_row + (int64_t)own_head * D * 2 + 16 * j;
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                own1[s][p] = *reinterpret_cast<const u32x4_t*>(own1p + off + p * own_plane + 64 * s);
                own2[s][p] = *reinterpret_cast<const u32x4_t*>(own2p + off + p * own_plane + 64 * s);
            }
        if constexpr (kDq) {
            const int64_t at = (int64_t)own_head * a.total_tokens + s0 + row;
            own_lse = a.lse2[at];
            own_delta = a.delta[at];
        }
    }

    // Operand addresses within a buffer (see the forward kernel for the transposing read).
    uint32_t row_off[KS], tr_off[NB];
#pragma unroll
    for (int s = 0; s < KS; ++s) row_off[s] = lds0 + (uint32_t)(m16 * ROW + 16 * ((4 * s + j) ^ (m16 % PITCH)));
    {
        const int r = 4 * j + (m16 >> 2);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
            tr_off[nb] = lds0 + (uint32_t)(r * ROW + 16 * ((2 * nb + ((m16 >> 1) & 1)) ^ (r % PITCH)) + 8 * (m16 & 1));
    }

    // acc[0]: dQ or dK, acc[1]: dV. float32 inputs keep the products of lower planes in a
    // sum of their own: the large sum is then rounded no more often than in a float32 product.
    f32x4_t acc[GRADS][NB], acc_lo[GRADS][NP == 3 ? NB : 1];
#pragma unroll
    for (int x = 0; x < GRADS; ++x)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            acc[x][nb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (NP == 3) acc_lo[x][nb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }

    // acc[x] += X^T W over the 32 rows of sub-block pp, X the streamed tensor `tensor`.
    // Operand element i of lane (own m16, j) is streamed row 16 (i / 4) + 4 j + i % 4.
    auto gradient = [&](int x, int tensor, const u32x4_t (&w)[3], int pp, uint32_t buf_off) __attribute__((always_inline)) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int pa = 0; pa < NP; ++pa) {
                u32x4_t xt;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const s16x4_t t = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (lds_s16x4*)((lds_u8*)(uintptr_t)(tr_off[nb] + buf_off) + (32 * pp + 16 * h) * ROW +
                                     (tensor * NP + pa) * TB));
                    const uint2 t2 = __builtin_bit_cast(uint2, t);
                    xt[2 * h] = t2.x;
                    xt[2 * h + 1] = t2.y;
                }
#pragma unroll
                for (int pb = 0; pa + pb < 3; ++pb) {
                    f32x4_t& sum = NP == 3 && pa + pb > 0 ? acc_lo[x][nb] : acc[x][nb];
                    sum = mma16<false>(xt, w[pb], sum);
                }
            }
    };

    // One sub-block of 32 streamed rows, row0 .. row0 + 31, in rows 32 pp of the buffer.
    auto sub_block = [&](int pp, int row0, uint32_t buf_off, uint32_t stat) __attribute__((always_inline)) {
        // dP - delta starts from -delta. [1]: the products of lower planes, for the scores of
        // several planes (see below) and dP of float32 inputs.
        constexpr int SC = NP > 1 ? 2 : 1, DP = NP == 3 ? 2 : 1;
        f32x4_t sc[SC][2], dp[DP][2], lse4[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (kDq) {
                dp[0][h] = f32x4_t{-own_delta, -own_delta, -own_delta, -own_delta};
            } else {
                lds_u8* const at = (lds_u8*)(uintptr_t)(stat + (uint32_t)(32 * pp + 16 * h + 4 * j) * 4u);
                lse4[h] = *(lds_f32x4*)at;
                dp[0][h] = -*(lds_f32x4*)(at + 256);
            }
            if constexpr (SC == 2) sc[1][h] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (DP == 2) dp[1][h] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int s = 0; s < KS; ++s)
#pragma unroll
                for (int pa = 0; pa < NP; ++pa) {
                    lds_u8* const at = (lds_u8*)(uintptr_t)(row_off[s] + buf_off) + (32 * pp + 16 * h) * ROW + pa * TB;
                    const u32x4_t x1 = *(lds_u32x4*)at, x2 = *(lds_u32x4*)(at + NP * TB);
#pragma unroll
                    for (int pb = 0; pb < NP && pa + pb < 3; ++pb) {
                        const int x = pa + pb > 0 ? SC - 1 : 0, y = pa + pb > 0 ? DP - 1 : 0;
                        const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
                        sc[x][h] = mma16<false>(x1, own1[s][pb], s == 0 && pa + pb == 0 ? zero : sc[x][h]);
                        dp[y][h] = mma16<false>(x2, own2[s][pb], dp[y][h]);
                    }
                }
        const bool full = kDq ? row0 + 31 <= own0 : (row0 >= own0 + OW - 1 && row0 + 32 <= L);   // wave-uniform
        float pr[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (SC == 2) {
                // An infinite q or k has NaN in its lower planes, but its score is that of the first
                // planes: -inf is a weight of zero.
#pragma unroll
                for (int jj = 0; jj < 4; ++jj)
                    sc[0][h][jj] = __builtin_isinf(sc[0][h][jj]) ? sc[0][h][jj] : sc[0][h][jj] + sc[1][h][jj];
            }
            if constexpr (DP == 2) dp[0][h] += dp[1][h];
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                const float lse = kDq ? own_lse : lse4[h][jj];
                // float32 inputs: expf, since rounding the exponent in log2 units is an error of
                // some 3e-7 of P, which the 16-bit types' own rounding hides.
                if constexpr (NP == 3) pr[h][jj] = expf(__builtin_fmaf(sc[0][h][jj], a.scale, -lse));
                else pr[h][jj] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[0][h][jj], a.scale_log2, -lse));
            }
            if (!full) {
                const int row = row0 + 16 * h + 4 * j, own = own0 + m16;
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    const bool valid = kDq ? row + jj <= own : (row + jj >= own && row + jj < L);
                    pr[h][jj] = valid ? pr[h][jj] : 0.0f;
                    dp[0][h][jj] = valid ? dp[0][h][jj] : 0.0f;
                }
            }
        }
        u32x4_t w[3];
        if constexpr (!kDq) {
#pragma unroll
            for (int u = 0; u < 4; ++u) split3<(NP > 1)>(pr[u / 2][2 * (u % 2)], pr[u / 2][2 * (u % 2) + 1], w, u);
            gradient(1, 1, w, pp, buf_off);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int h = u / 2, jj = 2 * (u % 2);
            split3<(NP > 1)>(pr[h][jj] * dp[0][h][jj], pr[h][jj + 1] * dp[0][h][jj + 1], w, u);
        }
        gradient(0, 0, w, pp, buf_off);
    };

    // End of a step: this wave's loads of the next block have arrived (with BUFS 3 one
    // younger block may still be in flight, `ahead` 1) and its LDS reads are done; after the
    // barrier that holds for every wave.
    auto end_step = [&](int ahead) __attribute__((always_inline)) {
        constexpr int kLgkm0 = 7 << 4;
        constexpr auto imm = [](int n) { return (n & 15) | kLgkm0 | (((n >> 4) & 3) << 14); };
        if (BUFS > 2 && ahead >= 1) __builtin_amdgcn_s_waitcnt(imm(LOADS));
        else __builtin_amdgcn_s_waitcnt(imm(0));
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __asm__ volatile("" ::: "memory");
    };

    // Step t computes block t from buffer t % BUFS; block t + BUFS - 1 is loaded meanwhile
    // into the buffer of block t - 1, whose last reads ended before the previous barrier.
    int head = kDq ? hk : hk * G + split * heads, blk = first, loaded = 0;       // the load cursor
    auto load_next = [&](int buf) __attribute__((always_inline)) {
        if (loaded == steps) return;
        load_block(head, blk, buf);
        ++loaded;
        if (++blk == first + blocks) {
            blk = first;
            ++head;
        }
    };
#pragma unroll
    for (int i = 0; i < BUFS - 1; ++i) load_next(i);
    end_step(loaded - 1);
    int buf = 0, this_blk = first;
    for (int t = 0; t < steps; ++t) {
        load_next(buf == 0 ? BUFS - 1 : buf - 1);
#pragma unroll
        for (int pp = 0; pp < SR / 32; ++pp) {
            const int row0 = this_blk * SR + 32 * pp;
            // dK, dV: the waves of a key group share the block's rows.
            if (!kDq && pp != wave / KG) continue;
            // Wave-uniform: some pair of the sub-block is attended.
            const bool some = own0 < L && row0 < L && (kDq ? row0 <= own0 + OW - 1 : row0 + 31 >= own0);
            if (some) sub_block(pp, row0, (uint32_t)buf * Sh::kBufBytes, stat0 + (uint32_t)buf * Sh::kStatBytes);
        }
        end_step(loaded - t - 2);
        if (++this_blk == first + blocks) this_blk = first;
        buf = buf == BUFS - 1 ? 0 : buf + 1;
    }

    if constexpr (NP == 3) {
#pragma unroll
        for (int x = 0; x < GRADS; ++x)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[x][nb] += acc_lo[x][nb];
    }
    if constexpr (!kDq && Sh::kHalves == 2) {
        // Waves w and w + KG hold the two halves of the streamed rows' sums for the same keys
        // (the last step's barrier ended every read of the buffers).
        f32x4_t* const half = reinterpret_cast<f32x4_t*>(lds) + (wave % KG) * (GRADS * NB * 64) + lane;
        static_assert(KG * GRADS * NB * 64 * 16 <= BUFS * Sh::kBufBytes, "the sums fit the buffers");
        if (wave >= KG) {
#pragma unroll
            for (int i = 0; i < GRADS * NB; ++i) half[i * 64] = acc[i / NB][i % NB];
        }
        __syncthreads();
        if (wave >= KG) return;
#pragma unroll
        for (int i = 0; i < GRADS * NB; ++i) acc[i / NB][i % NB] += half[i * 64];
    }

    // Lane (own row m16, j) holds dims 16 nb + 4 j .. + 3.
    const int row = own0 + m16;
    if (row >= L) return;
    const int heads_out = kDq ? a.hq : a.hkv;
    const int es = a.type == KVFP8_F32 ? 4 : 2;
#pragma unroll
    for (int x = 0; x < GRADS; ++x) {
        const int64_t at = ((s0 + row) * heads_out + own_head) * (int64_t)a.d;
        if (!kDq && a.splits > 1) {
            float* const prow = a.part + (int64_t)(x * a.splits + split) * a.total_tokens * a.hkv * a.d + at;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const int d0 = 16 * nb + 4 * j;
                if ((a.d & 3) == 0) {
                    if (d0 < a.d) *reinterpret_cast<f32x4_t*>(prow + d0) = acc[x][nb];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (d0 + i < a.d) prow[d0 + i] = acc[x][nb][i];
                }
            }
            continue;
        }
        const float factor = x == 0 ? a.scale : 1.0f;
        uint8_t* const orow = reinterpret_cast<uint8_t*>(x == 1 ? a.dv : (kDq ? a.dq : a.dk)) + at * es;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int d0 = 16 * nb + 4 * j;
            const f32x4_t y = acc[x][nb] * factor;
            if ((a.d & 3) == 0) {
                if (d0 >= a.d) continue;
                if (a.type == KVFP8_F32) *reinterpret_cast<f32x4_t*>(orow + d0 * 4) = y;
                else if (a.type == KVFP8_F16)
                    *reinterpret_cast<uint2*>(orow + d0 * 2) = make_uint2(pack2<true>(y[0], y[1]), pack2<true>(y[2], y[3]));
                else
                    *reinterpret_cast<uint2*>(orow + d0 * 2) = make_uint2(pack2<false>(y[0], y[1]), pack2<false>(y[2], y[3]));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (d0 + i >= a.d) continue;
                    if (a.type == KVFP8_F32) reinterpret_cast<float*>(orow)[d0 + i] = y[i];
                    else
                        reinterpret_cast<uint16_t*>(orow)[d0 + i] =
                            a.type == KVFP8_F16 ? f32_to_f16(y[i]) : f32_to_bf16(y[i]);
                }
            }
        }
    }
}

template <int D, int NP>
__global__ void __launch_bounds__((64 * BwdShape<D, NP>::kWaves), (BwdShape<D, NP>::kWavesPerSimd))
prefill_backward_kernel(BwdArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[BwdShape<D, NP>::kLds];
    const int64_t item = blockIdx.x;
    if (item < a.key_items) bwd_item<D, NP, false>(a, item, lds);
    else bwd_item<D, NP, true>(a, item - a.key_items, lds);
}

// Row statistics: lse (in log2 units for 16-bit inputs) and delta = sum(dO O), both [Hq][T], sixteen lanes
// per (token, q head). Tokens of no sequence (or past max_len of theirs) get zero gradients
// here, since no item covers them. Bound: HBM (O and dO read once).
struct StatArgs {
    const void* out;
    const void* dout;
    const float* lse;
    float* lse2;
    float* delta;
    void* dq;
    void* dk;
    void* dv;
    const void* cu;
    int32_t cu64, batch, hq, hkv, d, max_len;
    int64_t total_tokens;
    int32_t splits;
    float* part;
};

__device__ __forceinline__ int64_t load_cu(const StatArgs& a, int i) {
    return a.cu64 ? reinterpret_cast<const int64_t*>(a.cu)[i] : (int64_t)reinterpret_cast<const int32_t*>(a.cu)[i];
}

template <int IT>
__global__ void __launch_bounds__(256)
bwd_stats_kernel(StatArgs a, int32_t vec) {
    using T = typename Elem<IT>::T;
    // Sixteen lanes per row; four rows of one wave need not be of one token.
    const int lane = threadIdx.x & 15;
    const int64_t row = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    if (row >= a.total_tokens * a.hq) return;
    const int64_t token = row / a.hq;
    const int h = (int)(row - token * a.hq);
    const T* o = reinterpret_cast<const T*>(a.out) + row * a.d;
    const T* g = reinterpret_cast<const T*>(a.dout) + row * a.d;
    float sum = 0.0f;
    if (vec) {
        // 16-byte loads: d is a multiple of the elements in one, the rows are aligned.
        constexpr int N = 16 / sizeof(T);
        for (int i = N * lane; i < a.d; i += N * 16) {
            T x[N], y[N];
            *reinterpret_cast<u32x4_t*>(x) = *reinterpret_cast<const u32x4_t*>(o + i);
            *reinterpret_cast<u32x4_t*>(y) = *reinterpret_cast<const u32x4_t*>(g + i);
#pragma unroll
            for (int e = 0; e < N; ++e) sum = __builtin_fmaf(Elem<IT>::load(x[e]), Elem<IT>::load(y[e]), sum);
        }
    } else {
        for (int i = lane; i < a.d; i += 16) sum = __builtin_fmaf(Elem<IT>::load(o[i]), Elem<IT>::load(g[i]), sum);
    }
    int covered = 0;
    for (int b = lane; b < a.batch; b += 16) {
        const int64_t s0 = load_cu(a, b), s1 = load_cu(a, b + 1), lo = s0 < 0 ? 0 : s0;
        covered |= token >= lo && token < s1 && token - lo < a.max_len;
    }
#pragma unroll
    for (int x = 1; x < 16; x <<= 1) {
        sum += __shfl_xor(sum, x);
        covered |= __shfl_xor(covered, x);
    }
    if (covered) {
        if (lane == 0) {
            a.lse2[(int64_t)h * a.total_tokens + token] =
                a.lse[row] * (IT == KVFP8_F32 ? 1.0f : 1.44269504088896340736f);
            a.delta[(int64_t)h * a.total_tokens + token] = sum;
        }
        return;
    }
    for (int i = lane; i < a.d; i += 16) {
        reinterpret_cast<T*>(a.dq)[row * a.d + i] = (T)0;
        if (h < a.hkv) {
            const int64_t at = (token * a.hkv + h) * a.d + i;
            reinterpret_cast<T*>(a.dk)[at] = (T)0;
            reinterpret_cast<T*>(a.dv)[at] = (T)0;
            if (a.splits > 1)
                for (int x = 0; x < 2 * a.splits; ++x) a.part[x * a.total_tokens * a.hkv * a.d + at] = 0.0f;
        }
    }
}

// dK and dV from the sums of the workgroups that shared a KV head's q heads, in split order.
// Bound: memory (each sum read once).
template <int IT>
__global__ void __launch_bounds__(256)
bwd_reduce_kernel(const float* part, int64_t count, int32_t splits, float scale, void* dk, void* dv) {
    using T = typename Elem<IT>::T;
    T* const out = reinterpret_cast<T*>(blockIdx.y == 0 ? dk : dv);
    const float factor = blockIdx.y == 0 ? scale : 1.0f;
    const float* const in = part + (int64_t)blockIdx.y * splits * count;
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= count) return;
    if (i + 4 <= count && (count & 3) == 0) {
        f32x4_t sum = *reinterpret_cast<const f32x4_t*>(in + i);
        for (int x = 1; x < splits; ++x) sum += *reinterpret_cast<const f32x4_t*>(in + x * count + i);
        sum *= factor;
        if constexpr (IT == KVFP8_F32)
            *reinterpret_cast<f32x4_t*>(out + i) = sum;
        else
            *reinterpret_cast<uint2*>(out + i) =
                make_uint2(pack2<IT == KVFP8_F16>(sum[0], sum[1]), pack2<IT == KVFP8_F16>(sum[2], sum[3]));
        return;
    }
    for (int64_t e = i; e < i + 4 && e < count; ++e) {
        float sum = in[e];
        for (int x = 1; x < splits; ++x) sum += in[x * count + e];
        out[e] = Elem<IT>::store(sum * factor);
    }
}

// Inputs as bf16 planes of head size dp (zero-padded from d), for the input types and
// head sizes the kernel does not read in place. Four tensors in one launch; a thread
// takes two consecutive dims.
struct PlaneArgs {
    const void* in[4];
    uint32_t* out[4];          // two bf16 per dword, [plane][rows][dp]
    int64_t end[4];            // running ends of the tensors' rows
    int32_t d, dp, planes;
};

template <int IT>
__global__ void __launch_bounds__(256)
split_planes_kernel(PlaneArgs a) {
    using T = typename Elem<IT>::T;
    const int pairs = a.dp / 2;
    const int64_t total = a.end[3] * pairs;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        int64_t row = i / pairs;
        const int c = (int)(i - row * pairs), d0 = 2 * c;
        int t = 0;
        while (row >= a.end[t]) ++t;
        const int64_t begin = t == 0 ? 0 : a.end[t - 1], rows = a.end[t] - begin;
        row -= begin;
        const T* in = reinterpret_cast<const T*>(a.in[t]) + row * a.d + d0;
        const float x0 = d0 < a.d ? Elem<IT>::load(in[0]) : 0.0f;
        const float x1 = d0 + 1 < a.d ? Elem<IT>::load(in[1]) : 0.0f;
        u32x4_t planes[3];
        // (Finite values above the largest bf16 would round to infinity.)
        if (fmaxf(__builtin_fabsf(x0), __builtin_fabsf(x1)) > 3.3895313e38f) split3<false>(x0, x1, planes, 0);
        else split3<true>(x0, x1, planes, 0);
        for (int p = 0; p < a.planes; ++p) a.out[t][(p * rows + row) * pairs + c] = planes[p][0];
    }
}

// The launches, and the layout of the workspace: the two statistics, the sums of split dK and
// dV, then the planes of q, dO, k, v where the inputs are not read in place.
struct BwdPlan {
    int planes, dp, splits, waves, heads_per_block;
    bool in_place;
    int64_t key_items, items, stat_blocks, reduce_blocks;
    int64_t stat, part, q_plane, kv_plane, bytes;
};

// Workgroups per KV head and key block for dK and dV. One workgroup for all G q heads needs
// no second pass, but its chain of G * len / 32 steps then bounds the launch unless the
// batch keeps every CU busy for longer; a split writes float32 sums (up to four times q's bytes)
// that a second pass adds in order. The smallest split is taken whose chain fits under the rest,
// in steps of a CU (64 keys x 32 rows; dQ adds about 0.6):
// - the pairs at the mean length, or those of the longest sequence where they are more (lengths
//   are not known on the host, only their sum and their limit);
// - the dispatch of `items` workgroups, of which most are empty where lengths are uneven: 1.4 to
//   4 ns each, about 400 a step.
// A chain's step takes 1.75 times a CU's where three workgroups share one (bf16), else as long.
// Measured with 1, 2 and 4 workgroups (us; * taken). 16q/4kv heads, D 128, bf16: 4 sequences of
// 1024 tokens 257, 154, 138*; 8: 289, 245*, 270; 16: 455*, 504, 554; 16 of 64 to 1024: 292, 277*,
// 297; 300 of 64 with a limit of 4096 675*, 828, 1060; 60 of 128 and one of 4096 1001, 860*, 931.
// float16, 4 of 1024 287, 292*, 308; 8 574*, 601, 648; float32, 8 1091*, 1116, 1160. 8q/2kv, D 64,
// bf16: 16 of 1024 184, 142*, 152; 300 of 64 and one of 1024 194, 153, 181*. Over 123 batches of
// five head layouts the choice costs 2.1% more than the best one, at most 30%; at the mean length
// alone and 1.75 for every type it cost 8.8%, at most 85%.
int dkv_splits(int64_t tokens, int32_t batch, int64_t longest, int32_t hq, int32_t hkv, int planes, int64_t items) {
    const int G = hq / hkv;
    double squares = batch > 0 ? (double)tokens * (double)tokens / batch : 0.0;
    squares = squares > (double)longest * longest ? squares : (double)longest * longest;
    const double busy = 1.6 * hq * squares / 2 / (64 * 32) / device_cus() + (double)items / 400;
    const double step = planes == 1 ? 1.75 : 1.0;
    for (int n = 1; n < G; ++n)
        if (G % n == 0 && (double)(G / n) * (double)longest / 32 * step <= busy) return n;
    return G;
}

int check_backward(int dtype, int64_t tokens, int32_t hq, int32_t hkv, int32_t batch, int32_t max_len) {
    if (dtype != KVFP8_F32 && dtype != KVFP8_F16 && dtype != KVFP8_BF16) return KVFP8_EDTYPE;
    return tokens < 0 || batch < 0 || max_len < 0 || hq <= 0 || hkv <= 0 || hq % hkv != 0 ? KVFP8_ESHAPE : KVFP8_OK;
}

// KVFP8_ELIMIT where a launch would take 2^32 threads or more, which the runtime refuses.
int plan_backward(int dtype, int64_t tokens, int32_t hq, int32_t hkv, int32_t d, int32_t batch, int32_t max_len,
                  bool aligned, BwdPlan* p) {
    if (d < 1 || d > 128) return KVFP8_ESHAPE;
    if (tokens >= ((int64_t)1 << 31)) return KVFP8_ELIMIT;
    const int64_t longest = max_len < tokens ? max_len : tokens;
    const int G = hq / hkv;
    p->planes = dtype == KVFP8_BF16 ? 1 : (dtype == KVFP8_F16 ? 2 : 3);
    p->dp = d <= 64 ? 64 : (d <= 96 ? 96 : 128);
    p->waves = p->planes != 2 ? 4 : 8;
    p->heads_per_block = G % 4 == 0 ? 4 : (G % 2 == 0 ? 2 : 1);
    const int64_t key_rows = 64;                   // four waves' keys
    const int64_t q_rows = 16 * p->waves / p->heads_per_block;
    const int64_t key_items = (longest + key_rows - 1) / key_rows * batch * hkv;
    const int64_t q_items = (longest + q_rows - 1) / q_rows * batch * hkv * (G / p->heads_per_block);
    p->splits = dkv_splits(tokens, batch, longest, hq, hkv, p->planes, key_items + q_items);
    p->key_items = key_items * p->splits;
    p->items = p->key_items + q_items;
    p->stat_blocks = (tokens * hq + 15) / 16;
    p->reduce_blocks = (tokens * hkv * d + 1023) / 1024;
    const int64_t threads = (int64_t)1 << 32;
    if (p->items >= threads / (64 * p->waves) || p->stat_blocks >= threads / 256 ||
        (p->splits > 1 && p->reduce_blocks >= threads / 256))
        return KVFP8_ELIMIT;
    p->in_place = dtype == KVFP8_BF16 && d == p->dp && aligned;
    p->stat = (tokens * hq * 4 + 255) / 256 * 256;
    p->part = p->splits > 1 ? (2 * p->splits * tokens * hkv * d * 4 + 255) / 256 * 256 : 0;
    p->q_plane = tokens * hq * p->dp * 2;
    p->kv_plane = tokens * hkv * p->dp * 2;
    p->bytes = 2 * p->stat + p->part + (p->in_place ? 0 : 2 * p->planes * (p->q_plane + p->kv_plane));
    return KVFP8_OK;
}

template <int D>
hipError_t launch_backward(const BwdArgs& a, int planes, int64_t items, hipStream_t s) {
    const dim3 grid((unsigned)items), block(planes != 2 ? 256 : 512);
    if (planes == 1) hipLaunchKernelGGL((prefill_backward_kernel<D, 1>), grid, block, 0, s, a);
    else if (planes == 2) hipLaunchKernelGGL((prefill_backward_kernel<D, 2>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((prefill_backward_kernel<D, 3>), grid, block, 0, s, a);
    return hipGetLastError();
}

}  // namespace

}  // namespace kvfp8

using namespace kvfp8;

extern "C" int64_t kvfp8_prefill_backward_workspace_bytes(int dtype, int64_t total_tokens, int32_t num_q_heads,
                                                          int32_t num_kv_heads, int32_t head_dim, int32_t batch,
                                                          int32_t max_seq_len, int aligned) {
    int rc = check_backward(dtype, total_tokens, num_q_heads, num_kv_heads, batch, max_seq_len);
    if (rc != KVFP8_OK) return rc;
    BwdPlan p;
    rc = plan_backward(dtype, total_tokens, num_q_heads, num_kv_heads, head_dim, batch, max_seq_len, aligned != 0, &p);
    return rc == KVFP8_OK ? p.bytes : rc;
}

extern "C" int kvfp8_prefill_attention_backward(
    const void* q, const void* k, const void* v, const void* out, const float* lse, const void* grad_out, int dtype,
    int64_t total_tokens, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, const void* cu_seqlens,
    int cu_dtype, int32_t batch, int32_t max_seq_len, float scale, void* dq, void* dk, void* dv, void* workspace,
    int64_t workspace_bytes, void* stream) {
    int rc = check_backward(dtype, total_tokens, num_q_heads, num_kv_heads, batch, max_seq_len);
    if (rc != KVFP8_OK) return rc;
    if (cu_dtype != KVFP8_I32 && cu_dtype != KVFP8_I64) return KVFP8_EDTYPE;
    if (total_tokens == 0) return KVFP8_OK;
    if (!q || !k || !v || !out || !lse || !grad_out || !dq || !dk || !dv || !workspace || (batch > 0 && !cu_seqlens))
        return KVFP8_ENULL;
    const uintptr_t inputs = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)grad_out;
    const uintptr_t element = dtype == KVFP8_F32 ? 3 : 1;
    if (((inputs | (uintptr_t)out) & element) != 0) return KVFP8_ESTRIDE;
    if ((((uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv | (uintptr_t)workspace) & 15) != 0) return KVFP8_ESTRIDE;
    BwdPlan plan;
    rc = plan_backward(dtype, total_tokens, num_q_heads, num_kv_heads, head_dim, batch, max_seq_len, (inputs & 15) == 0,
                       &plan);
    if (rc != KVFP8_OK) return rc;
    if (workspace_bytes < plan.bytes) return KVFP8_EWORKSPACE;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);

    BwdArgs a;
    a.heads_per_block = plan.heads_per_block;
    a.splits = plan.splits;
    a.key_items = plan.key_items;

    StatArgs st;
    st.out = out;
    st.dout = grad_out;
    st.lse = lse;
    st.lse2 = reinterpret_cast<float*>(ws);
    st.delta = reinterpret_cast<float*>(ws + plan.stat);
    st.dq = dq;
    st.dk = dk;
    st.dv = dv;
    st.cu = cu_seqlens;
    st.cu64 = cu_dtype == KVFP8_I64;
    st.batch = batch;
    st.hq = num_q_heads;
    st.hkv = num_kv_heads;
    st.d = head_dim;
    st.max_len = max_seq_len;
    st.total_tokens = total_tokens;
    st.splits = plan.splits;
    st.part = a.part = reinterpret_cast<float*>(ws + 2 * plan.stat);
    const dim3 stat_grid((unsigned)plan.stat_blocks), block(256);
    const int32_t vec = (head_dim * (dtype == KVFP8_F32 ? 4 : 2)) % 16 == 0 && (((uintptr_t)out | (uintptr_t)grad_out) & 15) == 0;
    switch (dtype) {
        case KVFP8_F32: hipLaunchKernelGGL((bwd_stats_kernel<KVFP8_F32>), stat_grid, block, 0, s, st, vec); break;
        case KVFP8_F16: hipLaunchKernelGGL((bwd_stats_kernel<KVFP8_F16>), stat_grid, block, 0, s, st, vec); break;
        default: hipLaunchKernelGGL((bwd_stats_kernel<KVFP8_BF16>), stat_grid, block, 0, s, st, vec); break;
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess || plan.items == 0) return (int)err;

    a.q = reinterpret_cast<const uint8_t*>(q);
    a.k = reinterpret_cast<const uint8_t*>(k);
    a.v = reinterpret_cast<const uint8_t*>(v);
    a.dout = reinterpret_cast<const uint8_t*>(grad_out);
    a.q_plane = plan.q_plane;
    a.kv_plane = plan.kv_plane;
    if (!plan.in_place) {
        uint8_t* at = ws + 2 * plan.stat + plan.part;
        PlaneArgs pa;
        const void* in[4] = {q, grad_out, k, v};
        const uint8_t** to[4] = {&a.q, &a.dout, &a.k, &a.v};
        int64_t end = 0;
        for (int t = 0; t < 4; ++t) {
            pa.in[t] = in[t];
            pa.out[t] = reinterpret_cast<uint32_t*>(at);
            *to[t] = at;
            end += total_tokens * (t < 2 ? num_q_heads : num_kv_heads);
            pa.end[t] = end;
            at += plan.planes * (t < 2 ? plan.q_plane : plan.kv_plane);
        }
        pa.d = head_dim;
        pa.dp = plan.dp;
        pa.planes = plan.planes;
        int64_t blocks = (end * (plan.dp / 2) + 255) / 256;
        blocks = blocks < 16384 ? blocks : 16384;
        const dim3 grid((unsigned)blocks);
        switch (dtype) {
            case KVFP8_F32: hipLaunchKernelGGL((split_planes_kernel<KVFP8_F32>), grid, block, 0, s, pa); break;
            case KVFP8_F16: hipLaunchKernelGGL((split_planes_kernel<KVFP8_F16>), grid, block, 0, s, pa); break;
            default: hipLaunchKernelGGL((split_planes_kernel<KVFP8_BF16>), grid, block, 0, s, pa); break;
        }
        err = hipGetLastError();
        if (err != hipSuccess) return (int)err;
    }
    a.lse2 = st.lse2;
    a.delta = st.delta;
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    a.type = dtype;
    a.cu = cu_seqlens;
    a.cu64 = st.cu64;
    a.batch = batch;
    a.hq = num_q_heads;
    a.hkv = num_kv_heads;
    a.d = head_dim;
    const int64_t longest = max_seq_len < total_tokens ? max_seq_len : total_tokens;
    const int64_t q_rows = 16 * plan.waves / plan.heads_per_block;
    a.q_blocks = (int32_t)((longest + q_rows - 1) / q_rows);
    a.max_len = max_seq_len;
    a.total_tokens = total_tokens;
    a.scale = scale;
    a.scale_log2 = scale * 1.44269504088896340736f;
    switch (plan.dp) {
        case 64: err = launch_backward<64>(a, plan.planes, plan.items, s); break;
        case 96: err = launch_backward<96>(a, plan.planes, plan.items, s); break;
        default: err = launch_backward<128>(a, plan.planes, plan.items, s); break;
    }
    if (err != hipSuccess || plan.splits == 1) return (int)err;
    const int64_t count = total_tokens * num_kv_heads * head_dim;
    const dim3 grid((unsigned)plan.reduce_blocks, 2);
    switch (dtype) {
        case KVFP8_F32: hipLaunchKernelGGL((bwd_reduce_kernel<KVFP8_F32>), grid, block, 0, s, a.part, count, plan.splits, scale, dk, dv); break;
        case KVFP8_F16: hipLaunchKernelGGL((bwd_reduce_kernel<KVFP8_F16>), grid, block, 0, s, a.part, count, plan.splits, scale, dk, dv); break;
        default: hipLaunchKernelGGL((bwd_reduce_kernel<KVFP8_BF16>), grid, block, 0, s, a.part, count, plan.splits, scale, dk, dv); break;
    }
    return (int)hipGetLastError();
}
