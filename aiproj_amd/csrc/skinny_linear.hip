// y = x W^T for the few rows of a decode step: x [M, K] with M <= 64, W [N, K] row-major (a
// Linear layer's weight), bf16 or f16, float32 sums, one rounding.
//
// Bound: HBM, the weight read once (a decode step's weights exceed the last-level cache).
//
// Work split. A workgroup's eight waves divide K: wave w owns STEPS steps of 32 and the
// workgroup walks over tiles of 16 weight rows. Everything a wave reads is a stream of
// blocks of 16 rows of its K slice: first x (16 MT rows, kept in registers as MFMA operands:
// 32 MT VGPRs at 8 steps), then its slice of tile after tile. Blocks go straight from global
// memory into the wave's own two LDS slots, whole 512-byte row pieces per instruction (an
// operand-shaped load of 64 bytes from each of 16 rows moved 25 bytes/ns per CU, from L2 as
// from HBM: 64 rows through a 3072 x 2048 weight 12.4 us), one block in flight while the
// other is used, with no barrier. The eight partial tiles meet in LDS and are added in
// wave order. K beyond 2048 goes in groups, x read again. With fewer tiles than CUs the rows
// of x are divided over workgroups instead (their second read of a tile hits L2).
//
// Measured (us, bf16, weights from HBM; 64 rows, then 1 row; in brackets torch's GEMM):
//   3072 x 2048    8.0 [11.9]   5.4 [11.3]      2048 x 5632   12.0 [18.7]    9.2 [11.7]
//   2048 x 2048    6.0 [11.6]   4.9 [11.0]     32000 x 2048   34.2 [36.0]   27.4 [34.9]
//  11264 x 2048   16.5 [18.1]  12.2 [16.4]      8192 x 4096   26.7 [20.2]   16.0 [17.1]
// The last one reads x twice per tile and has more tiles than workgroups: callers leave
// such shapes (K above 2048 and more than 256 tiles) to the GEMM.
//
// kGated: W is a feed-forward block's fused projection [gate rows | up rows] and the output
// silu(gate) * up. A tile is then 8 gate rows and the 8 up rows beside them, so the activation
// needs no launch and no pass of its own; gate and up are rounded to the output's type first,
// as the projection's store rounds them: the same bits as the two launches.
// Measured (us, bf16, the two launches -> this one; the projection alone costs the same within
// 0.6): 2 x 5632 x 2048, 64 rows 18.6 -> 15.6, 1 row 14.3 -> 11.1; 2 x 512 x 256, 64 rows 5.0 -> 2.7.
//
// kRotates: W is the fused q, k and v projection of a decode step and the q and k columns are
// rotated by their row's position, in the epilogue's pairs; the projection's rounding is kept
// here too. A thread's row is the same for every tile: its position is read once, the tile's
// angles while the tile streams in.
// Measured (us, bf16, the two launches -> this one, in brackets the projection alone): 3072 x
// 2048, 64 rows 11.4 -> 8.4 [7.8], 1 row 8.4 -> 6.2 [5.4]; 768 x 256, 64 rows 5.4 -> 3.1 [2.4].
#include "mfma_tiles.h"

namespace kvfp8 {

namespace {

constexpr int kLinWaves = 8;
constexpr int kLinSteps = 8;                 // K steps of 32 per wave and group
constexpr int kLinRows = 16;                 // weight rows per tile

struct LinArgs {
    const uint8_t* x;
    const uint8_t* w;
    uint8_t* y;
    int64_t x_row, y_row, w_row;             // bytes between rows
    int32_t rows, tiles, steps;              // rows of x, tiles of N, K / 32
    int32_t groups;                          // ceil(steps / (8 waves x steps per wave))
    int32_t walkers;                         // workgroups that walk the tiles side by side
    int32_t half;                            // kGated: rows of gate, and of up
    // kRotates: columns before `rotated` turn by the angles of positions[row] in the tables
    // [table_rows][head_dim / 2] (rows of positions outside them stay).
    const void* positions;
    const void* cos_table;
    const void* sin_table;
    int64_t table_rows;
    int32_t pos64, table_dtype, rotated, head_dim;
};

enum { kPlain, kGate, kRotate };             // what the epilogue does

__device__ __forceinline__ float table_value(const void* table, int dtype, int64_t at) {
    if (dtype == KVFP8_F32) return reinterpret_cast<const float*>(table)[at];
    const uint16_t x = reinterpret_cast<const uint16_t*>(table)[at];
    return dtype == KVFP8_F16 ? Elem<KVFP8_F16>::load(x) : Elem<KVFP8_BF16>::load(x);
}

// Barrier over LDS accesses only: __syncthreads would also wait for the block in flight.
__device__ __forceinline__ void lds_barrier() {
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

template <int MT, int STEPS, bool kF16, int kEpi>
__global__ void __launch_bounds__(64 * kLinWaves, 2)
skinny_linear_kernel(LinArgs a) {
    constexpr bool kGated = kEpi == kGate, kRotates = kEpi == kRotate;
    constexpr int ROW = STEPS * 64;                  // bytes of a row's slice
    constexpr int CPR = ROW / 16;                    // 16-byte chunks of it
    constexpr int MASK = CPR < 16 ? CPR - 1 : 15;    // chunk c of row r sits in slot c ^ (r & MASK)
    constexpr int BLOCK = 16 * ROW;
    constexpr int LOADS = BLOCK / 1024;              // instructions per block
    __shared__ __attribute__((aligned(16))) uint8_t ring[kLinWaves][2][BLOCK];
    __shared__ __attribute__((aligned(16))) float sums[kLinWaves][MT * 16 * kLinRows];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int m16 = lane & 15, j = lane >> 4;
    const int part = blockIdx.x / a.walkers, first = blockIdx.x % a.walkers;
    const int m0 = part * 16 * MT;                   // this workgroup's rows of x
    if (first >= a.tiles) return;

    typedef __attribute__((address_space(3))) void* lds_ptr;
    typedef __attribute__((address_space(3))) const uint8_t lds_u8;
    typedef __attribute__((address_space(3))) const u32x4_t lds_u32x4;
    const uint32_t ring0 = (uint32_t)(uintptr_t)(lds_ptr)&ring[wave][0][0];

    // One block: rows row0 .. row0 + 15 (at most last_row) of a matrix, this wave's slice of
    // group `group`; chunks past K repeat its last one (and are not multiplied). Rows 8 .. 15
    // are taken from `up` rows further on.
    // Instruction i fills 1 KB: slot lane of it is row (64 i + lane) / CPR. Inline assembly,
    // waited for by hand, as in the prompt-attention kernel.
    auto load = [&](const uint8_t* base, int64_t stride, int row0, int last_row, int group, int slot, int up)
        __attribute__((always_inline)) {
        const int chunk0 = (group * kLinWaves + wave) * CPR;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int r = (64 * i + lane) / CPR, c = (lane % CPR) ^ (r & MASK);
            const int row = min(row0 + r, last_row) + (kGated && r >= 8 ? up : 0);
            const uint8_t* p = base + row * stride + 16 * (int64_t)min(chunk0 + c, 4 * a.steps - 1);
            __asm__ volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off"
                             :: "s"(__builtin_amdgcn_readfirstlane(ring0 + slot * BLOCK + 1024 * i)), "v"(p) : "memory");
        }
    };
    // Operand of step s from a slot: row m16, chunk 4 s + j.
    auto operand = [&](int slot, int s) __attribute__((always_inline)) -> u32x4_t {
        return *(lds_u32x4*)(lds_u8*)(uintptr_t)(ring0 + slot * BLOCK + m16 * ROW + 16 * ((4 * s + j) ^ (m16 & MASK)));
    };

    // The stream: for each tile and group, the MT blocks of x (once when there is one
    // group), then the tile's. The load cursor runs one block ahead.
    int l_tile = first, l_group = 0, l_block = 0, l_slot = 0;
    bool l_more = true;
    auto load_next = [&]() __attribute__((always_inline)) -> bool {
        if (!l_more) return false;
        if (l_block < MT) load(a.x, a.x_row, m0 + 16 * l_block, a.rows - 1, l_group, l_slot, 0);
        else if constexpr (kGated) load(a.w, a.w_row, 8 * l_tile, 2 * a.half - 1, l_group, l_slot, a.half - 8);
        else load(a.w, a.w_row, kLinRows * l_tile, kLinRows * a.tiles - 1, l_group, l_slot, 0);
        l_slot ^= 1;
        if (++l_block <= MT) return true;
        l_block = a.groups > 1 ? 0 : MT;
        if (++l_group == a.groups) {
            l_group = 0;
            l_tile += a.walkers;
            l_more = l_tile < a.tiles;
        }
        return true;
    };
    // The oldest block has arrived (`younger`: one more was issued after it); its slot may be
    // filled again once its reads are done.
    auto arrived = [&](bool younger) __attribute__((always_inline)) {
        if (younger) __builtin_amdgcn_s_waitcnt((LOADS & 15) | (7 << 4) | (15 << 8));
        else __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));
        __asm__ volatile("" ::: "memory");
    };
    auto reads_done = [&]() __attribute__((always_inline)) {
        __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };

    // The epilogue's thread: two neighbouring outputs (col, col + 1 of the tile) of one row of x.
    using E = Elem<kF16 ? KVFP8_F16 : KVFP8_BF16>;
    constexpr int kCols = kGated ? kLinRows / 2 : kLinRows;
    constexpr int kPairs = MT * 16 * kCols / 2;
    const int local = 2 * (int)threadIdx.x / kCols, col = 2 * (int)threadIdx.x % kCols, row = m0 + local;
    const bool stores = (int)threadIdx.x < kPairs && row < a.rows;

    u32x4_t x[MT][STEPS];
    f32x4_t acc[MT];
    int slot = 0;
    load_next();
    int64_t pos = -1;
    if constexpr (kRotates) {
        if (stores)
            pos = a.pos64 ? reinterpret_cast<const int64_t*>(a.positions)[row]
                          : (int64_t)reinterpret_cast<const int32_t*>(a.positions)[row];
        // Arrived before the loop, where a wait for it would wait for the block in flight too.
        __asm__ volatile("" : "+v"(pos));
    }
    for (int tile = first; tile < a.tiles; tile += a.walkers) {
        float cs = 1.0f, sn = 0.0f;
        bool turn = false;
        if constexpr (kRotates) {
            const int at = tile * kLinRows + col;
            turn = at < a.rotated && pos >= 0 && pos < a.table_rows;
            if (turn) {
                const int64_t angle = pos * (a.head_dim / 2) + (at % a.head_dim) / 2;
                cs = table_value(a.cos_table, a.table_dtype, angle);
                sn = table_value(a.sin_table, a.table_dtype, angle);
            }
        }
        for (int group = 0; group < a.groups; ++group) {
            if (a.groups > 1 || tile == first) {
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    arrived(load_next());
#pragma unroll
                    for (int s = 0; s < STEPS; ++s) x[t][s] = operand(slot, s);
                    reads_done();
                    slot ^= 1;
                }
            }
            arrived(load_next());
            if (group == 0) {
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
            const int valid = a.steps - (group * kLinWaves + wave) * STEPS;
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                if (s >= valid) break;       // wave-uniform
                const u32x4_t w = operand(slot, s);
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t] = mma16<kF16>(w, x[t][s], acc[t]);
            }
            reads_done();
            slot ^= 1;
        }
        // acc[t]: lane holds weight rows 4 j .. + 3 of x row 16 t + m16.
#pragma unroll
        for (int t = 0; t < MT; ++t)
            *reinterpret_cast<f32x4_t*>(&sums[wave][(16 * t + m16) * kLinRows + 4 * j]) = acc[t];
        lds_barrier();
        auto sum2 = [&](int at) __attribute__((always_inline)) -> float2 {
            float2 sum = *reinterpret_cast<const float2*>(&sums[0][at]);
#pragma unroll
            for (int v = 1; v < kLinWaves; ++v) {
                const float2 y = *reinterpret_cast<const float2*>(&sums[v][at]);
                sum.x += y.x;
                sum.y += y.y;
            }
            return sum;
        };
        if (stores) {
            uint32_t out;
            if constexpr (kGated) {
                const float2 gate = sum2(local * kLinRows + col), up = sum2(local * kLinRows + 8 + col);
                const uint32_t g = pack2<kF16>(gate.x, gate.y), u = pack2<kF16>(up.x, up.y);
                out = pack2<kF16>(swiglu(E::load((uint16_t)g), E::load((uint16_t)u)),
                                  swiglu(E::load((uint16_t)(g >> 16)), E::load((uint16_t)(u >> 16))));
            } else {
                const float2 sum = sum2(local * kLinRows + col);
                out = pack2<kF16>(sum.x, sum.y);
                if constexpr (kRotates) {
                    constexpr int DT = kF16 ? KVFP8_F16 : KVFP8_BF16;
                    if (turn) {
                        float x0 = E::load((uint16_t)out), x1 = E::load((uint16_t)(out >> 16));
                        rotate_pair<DT>(rnd<DT>(cs), rnd<DT>(sn), x0, x1);
                        out = pack2<kF16>(x0, x1);
                    }
                }
            }
            *reinterpret_cast<uint32_t*>(a.y + row * a.y_row + (int64_t)(tile * kCols + col) * 2) = out;
        }
        lds_barrier();
    }
}

template <int MT, int STEPS>
hipError_t launch_linear(const LinArgs& a, bool f16, int grid, hipStream_t s) {
    const dim3 g(grid), b(64 * kLinWaves);
    if (a.half > 0) {
        if (f16) hipLaunchKernelGGL((skinny_linear_kernel<MT, STEPS, true, kGate>), g, b, 0, s, a);
        else hipLaunchKernelGGL((skinny_linear_kernel<MT, STEPS, false, kGate>), g, b, 0, s, a);
    } else if (a.rotated > 0) {
        if (f16) hipLaunchKernelGGL((skinny_linear_kernel<MT, STEPS, true, kRotate>), g, b, 0, s, a);
        else hipLaunchKernelGGL((skinny_linear_kernel<MT, STEPS, false, kRotate>), g, b, 0, s, a);
    } else {
        if (f16) hipLaunchKernelGGL((skinny_linear_kernel<MT, STEPS, true, kPlain>), g, b, 0, s, a);
        else hipLaunchKernelGGL((skinny_linear_kernel<MT, STEPS, false, kPlain>), g, b, 0, s, a);
    }
    return hipGetLastError();
}

template <int MT>
hipError_t launch_linear_steps(const LinArgs& a, int per_wave, bool f16, int grid, hipStream_t s) {
    switch (per_wave) {
        case 2: return launch_linear<MT, 2>(a, f16, grid, s);
        case 4: return launch_linear<MT, 4>(a, f16, grid, s);
        default: return launch_linear<MT, 8>(a, f16, grid, s);
    }
}

}  // namespace

}  // namespace kvfp8

using namespace kvfp8;

namespace {

// n: weight rows; a: what the epilogue needs (zeros for plain).
int skinny_linear(LinArgs a, const void* x, int dtype, int64_t x_stride, int32_t rows, int32_t k, const void* weight,
                  int64_t w_stride, int32_t n, void* out, int64_t out_stride, void* stream) {
    if (dtype != KVFP8_BF16 && dtype != KVFP8_F16) return KVFP8_EDTYPE;
    if (rows < 0 || rows > 64 || k <= 0 || k % 32 != 0 || n <= 0 || n % kLinRows != 0) return KVFP8_ESHAPE;
    if (rows == 0) return KVFP8_OK;
    if (!x || !weight || !out) return KVFP8_ENULL;
    if ((((uintptr_t)x | (uintptr_t)weight) & 15) != 0 || ((uintptr_t)out & 3) != 0 || x_stride % 8 != 0 ||
        w_stride % 8 != 0 || out_stride % 2 != 0 || w_stride < k)
        return KVFP8_ESTRIDE;
    a.x = reinterpret_cast<const uint8_t*>(x);
    a.w = reinterpret_cast<const uint8_t*>(weight);
    a.y = reinterpret_cast<uint8_t*>(out);
    a.x_row = x_stride * 2;
    a.w_row = w_stride * 2;
    a.y_row = out_stride * 2;
    a.rows = rows;
    a.tiles = n / kLinRows;
    a.steps = k / 32;
    int per_wave = 2;
    while (per_wave < kLinSteps && kLinWaves * per_wave < a.steps) per_wave *= 2;
    a.groups = (a.steps + kLinWaves * per_wave - 1) / (kLinWaves * per_wave);
    const int cus = device_cus();
    // Row tiles per workgroup: all of them, or fewer while that puts idle CUs to work.
    int mt = (rows + 15) / 16;
    const int row_tiles = mt;
    while (mt > 1 && (int64_t)a.tiles * ((row_tiles + mt / 2 - 1) / (mt / 2)) <= cus) mt /= 2;
    const int parts = (row_tiles + mt - 1) / mt;
    a.walkers = cus / parts < 1 ? 1 : cus / parts;
    if (a.walkers > a.tiles) a.walkers = a.tiles;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const bool f16 = dtype == KVFP8_F16;
    const int grid = a.walkers * parts;
    switch (mt) {
        case 1: return (int)launch_linear_steps<1>(a, per_wave, f16, grid, s);
        case 2: return (int)launch_linear_steps<2>(a, per_wave, f16, grid, s);
        case 3: return (int)launch_linear_steps<3>(a, per_wave, f16, grid, s);
        default: return (int)launch_linear_steps<4>(a, per_wave, f16, grid, s);
    }
}

}  // namespace

extern "C" int kvfp8_skinny_linear(const void* x, int dtype, int64_t x_stride, int32_t rows, int32_t k,
                                   const void* weight, int64_t w_stride, int32_t n, void* out, int64_t out_stride,
                                   void* stream) {
    return skinny_linear(LinArgs{}, x, dtype, x_stride, rows, k, weight, w_stride, n, out, out_stride, stream);
}

extern "C" int kvfp8_skinny_linear_swiglu(const void* x, int dtype, int64_t x_stride, int32_t rows, int32_t k,
                                          const void* weight, int64_t w_stride, int32_t n, void* out,
                                          int64_t out_stride, void* stream) {
    if (n <= 0 || n % (kLinRows / 2) != 0 || n > (1 << 30)) return KVFP8_ESHAPE;
    LinArgs a{};
    a.half = n;
    return skinny_linear(a, x, dtype, x_stride, rows, k, weight, w_stride, 2 * n, out, out_stride, stream);
}

extern "C" int kvfp8_skinny_linear_rope(const void* x, int dtype, int64_t x_stride, int32_t rows, int32_t k,
                                        const void* weight, int64_t w_stride, int32_t n, int32_t heads,
                                        int32_t head_dim, const void* positions, int pos_dtype, const void* cos_table,
                                        const void* sin_table, int table_dtype, int64_t table_rows, void* out,
                                        int64_t out_stride, void* stream) {
    if (table_dtype != KVFP8_F32 && table_dtype != KVFP8_F16 && table_dtype != KVFP8_BF16) return KVFP8_EDTYPE;
    if (pos_dtype != KVFP8_I32 && pos_dtype != KVFP8_I64) return KVFP8_EDTYPE;
    if (heads <= 0 || head_dim <= 0 || head_dim % 2 != 0 || table_rows <= 0 || (int64_t)heads * head_dim > n)
        return KVFP8_ESHAPE;
    if (rows > 0 && (!positions || !cos_table || !sin_table)) return KVFP8_ENULL;
    LinArgs a{};
    a.positions = positions;
    a.pos64 = pos_dtype == KVFP8_I64;
    a.cos_table = cos_table;
    a.sin_table = sin_table;
    a.table_dtype = table_dtype;
    a.table_rows = table_rows;
    a.rotated = heads * head_dim;
    a.head_dim = head_dim;
    return skinny_linear(a, x, dtype, x_stride, rows, k, weight, w_stride, n, out, out_stride, stream);
}
