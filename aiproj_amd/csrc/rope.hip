// Interleaved-pair rotary embedding applied in place to the q and k heads of a
// packed projection output (gfx950).
//
// Replaces the PyTorch op sequence of reference src/torch_llm/model/rope.py:46-55
// with one kernel. For every row t, head h < heads and pair i < head_dim / 2:
//   c = cos_table[pos[t], i], s = sin_table[pos[t], i]     (cast to the dtype)
//   x0' = c x0 - s x1,  x1' = s x0 + c x1
// Each multiply, add and subtract is rounded to the tensor dtype, as the
// reference's elementwise operations on a bf16/f16 tensor are, so the result is
// bit-identical to that sequence. Rows whose position lies outside the tables are
// left unrotated (the reference's table lookup would fault on them).
#include "kvfp8_common.h"

namespace kvfp8 {

constexpr int kRopeThreads = 256;

struct RopeArgs {
    void* x;
    int64_t rows;
    int32_t heads, head_dim;
    int64_t row_stride, head_stride;     // elements
    const void* positions;
    int32_t pos64;
    const void* cos_table;
    const void* sin_table;
    int64_t table_rows;
};

template <int DT, int TT>
__global__ void __launch_bounds__(kRopeThreads)
rope_kernel(RopeArgs a) {
    using T = typename Elem<DT>::T;
    const int half = a.head_dim / 2;
    const int64_t pairs_per_row = (int64_t)a.heads * half;
    const int64_t total = a.rows * pairs_per_row;
    for (int64_t p = (int64_t)blockIdx.x * kRopeThreads + threadIdx.x; p < total;
         p += (int64_t)gridDim.x * kRopeThreads) {
        const int64_t r = p / pairs_per_row;
        const int64_t rem = p - r * pairs_per_row;
        const int h = (int)(rem / half);
        const int i = (int)(rem - (int64_t)h * half);
        const int64_t pos = a.pos64 ? reinterpret_cast<const int64_t*>(a.positions)[r]
                                    : (int64_t)reinterpret_cast<const int32_t*>(a.positions)[r];
        if (pos < 0 || pos >= a.table_rows) continue;
        using TabT = typename Elem<TT>::T;
        const float c = rnd<DT>(Elem<TT>::load(reinterpret_cast<const TabT*>(a.cos_table)[pos * half + i]));
        const float s = rnd<DT>(Elem<TT>::load(reinterpret_cast<const TabT*>(a.sin_table)[pos * half + i]));
        T* e = reinterpret_cast<T*>(a.x) + r * a.row_stride + (int64_t)h * a.head_stride + 2 * i;
        float x0 = Elem<DT>::load(e[0]), x1 = Elem<DT>::load(e[1]);
        rotate_pair<DT>(c, s, x0, x1);
        e[0] = Elem<DT>::store(x0);
        e[1] = Elem<DT>::store(x1);
    }
}

// Eight consecutive elements (four pairs) per thread, for head sizes that are a multiple of 8
// and aligned rows; the same rounding sequence. kSplit: the rows are a fused projection
// [q heads | k heads | v heads]; q, k (rotated) and v go to packed tensors, so that a prompt's
// attention needs no copies. Bound: HBM, rows read and written once.
// Measured (4224 rows of 16q/4kv heads, D 128, bf16): one pair per thread with 64-bit index
// divisions 30 us in place, and 20 us more for the three copies -> 19 us split.
// In place, few rows are launch and latency: one pair per thread then ends sooner. Measured (us,
// bf16, one pair | eight elements): 20 heads of 128, 65 rows 2.3 | 2.8, 128 rows (164 thousand
// pairs) 2.6 | 2.9, 256 rows 3.3 | 3.2; 40 heads of 80, 128 rows (205 thousand) 3.0 | 2.9.
constexpr int64_t kRopeVecPairs = 200000;
struct RopeOut {
    void* q;
    void* k;
    void* v;
    int32_t num_q_heads, num_kv_heads;
};

template <int DT, int TT, bool kSplit>
__global__ void __launch_bounds__(kRopeThreads)
rope_vec_kernel(RopeArgs a, RopeOut out) {
    using T = typename Elem<DT>::T;
    using TabT = typename Elem<TT>::T;
    struct alignas(16) Vec { T e[8]; };
    struct alignas(4 * sizeof(TabT)) Tab { TabT e[4]; };
    const uint32_t per_head = (uint32_t)a.head_dim / 8;
    const uint32_t heads = kSplit ? (uint32_t)(out.num_q_heads + 2 * out.num_kv_heads) : (uint32_t)a.heads;
    const uint32_t per_row = heads * per_head;
    const uint32_t total = (uint32_t)a.rows * per_row;              // below 2^31, checked by the host
    for (uint32_t p = blockIdx.x * kRopeThreads + threadIdx.x; p < total; p += gridDim.x * kRopeThreads) {
        const uint32_t r = p / per_row, rem = p - r * per_row;
        const uint32_t h = rem / per_head, c = rem - h * per_head;
        T* const src = reinterpret_cast<T*>(a.x) + (int64_t)r * a.row_stride + (int64_t)h * a.head_stride + 8 * c;
        Vec v = *reinterpret_cast<const Vec*>(src);
        const int64_t pos = a.pos64 ? reinterpret_cast<const int64_t*>(a.positions)[r]
                                    : (int64_t)reinterpret_cast<const int32_t*>(a.positions)[r];
        const bool rotate = (!kSplit || h < (uint32_t)(out.num_q_heads + out.num_kv_heads)) && pos >= 0 &&
                            pos < a.table_rows;
        if (rotate) {
            const int64_t at = pos * (a.head_dim / 2) + 4 * c;
            const Tab ct = *reinterpret_cast<const Tab*>(reinterpret_cast<const TabT*>(a.cos_table) + at);
            const Tab st = *reinterpret_cast<const Tab*>(reinterpret_cast<const TabT*>(a.sin_table) + at);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float cs = rnd<DT>(Elem<TT>::load(ct.e[i])), sn = rnd<DT>(Elem<TT>::load(st.e[i]));
                float x0 = Elem<DT>::load(v.e[2 * i]), x1 = Elem<DT>::load(v.e[2 * i + 1]);
                rotate_pair<DT>(cs, sn, x0, x1);
                v.e[2 * i] = Elem<DT>::store(x0);
                v.e[2 * i + 1] = Elem<DT>::store(x1);
            }
        }
        T* dst = src;
        if constexpr (kSplit) {
            const uint32_t nq = (uint32_t)out.num_q_heads, nkv = (uint32_t)out.num_kv_heads;
            const uint32_t first = h < nq ? 0 : (h < nq + nkv ? nq : nq + nkv), n = h < nq ? nq : nkv;
            T* const base = reinterpret_cast<T*>(h < nq ? out.q : (h < nq + nkv ? out.k : out.v));
            dst = base + ((int64_t)r * n + (h - first)) * a.head_dim + 8 * c;
        } else if (!rotate) {
            continue;
        }
        *reinterpret_cast<Vec*>(dst) = v;
    }
}

}  // namespace kvfp8

using namespace kvfp8;

namespace {

template <int DT>
hipError_t launch_rope(const RopeArgs& a, int table_dtype, dim3 grid, hipStream_t s) {
    switch (table_dtype) {
        case KVFP8_F32: hipLaunchKernelGGL((rope_kernel<DT, KVFP8_F32>), grid, dim3(kRopeThreads), 0, s, a); break;
        case KVFP8_F16: hipLaunchKernelGGL((rope_kernel<DT, KVFP8_F16>), grid, dim3(kRopeThreads), 0, s, a); break;
        default: hipLaunchKernelGGL((rope_kernel<DT, KVFP8_BF16>), grid, dim3(kRopeThreads), 0, s, a); break;
    }
    return hipGetLastError();
}

template <int DT, bool kSplit>
hipError_t launch_rope_vec(const RopeArgs& a, const RopeOut& out, int table_dtype, dim3 grid, hipStream_t s) {
    switch (table_dtype) {
        case KVFP8_F32: hipLaunchKernelGGL((rope_vec_kernel<DT, KVFP8_F32, kSplit>), grid, dim3(kRopeThreads), 0, s, a, out); break;
        case KVFP8_F16: hipLaunchKernelGGL((rope_vec_kernel<DT, KVFP8_F16, kSplit>), grid, dim3(kRopeThreads), 0, s, a, out); break;
        default: hipLaunchKernelGGL((rope_vec_kernel<DT, KVFP8_BF16, kSplit>), grid, dim3(kRopeThreads), 0, s, a, out); break;
    }
    return hipGetLastError();
}

template <bool kSplit>
hipError_t launch_rope_vec(const RopeArgs& a, const RopeOut& out, int dtype, int table_dtype, int64_t vectors,
                           hipStream_t s) {
    int64_t blocks = (vectors + kRopeThreads - 1) / kRopeThreads;
    const dim3 grid((unsigned)(blocks > 65536 ? 65536 : blocks));
    switch (dtype) {
        case KVFP8_F32: return launch_rope_vec<KVFP8_F32, kSplit>(a, out, table_dtype, grid, s);
        case KVFP8_F16: return launch_rope_vec<KVFP8_F16, kSplit>(a, out, table_dtype, grid, s);
        default: return launch_rope_vec<KVFP8_BF16, kSplit>(a, out, table_dtype, grid, s);
    }
}

// Rows, heads and tables that eight-element accesses fit, and indices below 2^31.
bool rope_vec_ok(const RopeArgs& a, int dtype, int table_dtype, int64_t heads) {
    const int64_t es = dtype == KVFP8_F32 ? 4 : 2, ts = table_dtype == KVFP8_F32 ? 4 : 2;
    return a.head_dim % 8 == 0 && ((uintptr_t)a.x & 15) == 0 && (a.row_stride * es) % 16 == 0 &&
           (a.head_stride * es) % 16 == 0 && (((uintptr_t)a.cos_table | (uintptr_t)a.sin_table) & (4 * ts - 1)) == 0 &&
           a.rows * heads * (a.head_dim / 8) < ((int64_t)1 << 31) - 65536 * kRopeThreads;
}

}  // namespace

extern "C" int kvfp8_rope_split(const void* x, int dtype, int64_t rows, int32_t num_q_heads, int32_t num_kv_heads,
                                int32_t head_dim, int64_t row_stride, const void* positions, int pos_dtype,
                                const void* cos_table, const void* sin_table, int table_dtype, int64_t table_rows,
                                void* q_out, void* k_out, void* v_out, void* stream) {
    auto is_float = [](int d) { return d == KVFP8_F32 || d == KVFP8_F16 || d == KVFP8_BF16; };
    if (!is_float(dtype) || !is_float(table_dtype)) return KVFP8_EDTYPE;
    if (pos_dtype != KVFP8_I32 && pos_dtype != KVFP8_I64) return KVFP8_EDTYPE;
    if (rows < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || head_dim % 2 != 0 || table_rows <= 0)
        return KVFP8_ESHAPE;
    if (rows == 0) return KVFP8_OK;
    if (!x || !positions || !cos_table || !sin_table || !q_out || !k_out || !v_out) return KVFP8_ENULL;
    const RopeArgs a{const_cast<void*>(x), rows, num_q_heads + num_kv_heads, head_dim, row_stride, head_dim, positions,
                     pos_dtype == KVFP8_I64, cos_table, sin_table, table_rows};
    const int64_t heads = (int64_t)num_q_heads + 2 * (int64_t)num_kv_heads;
    if (!rope_vec_ok(a, dtype, table_dtype, heads) ||
        (((uintptr_t)q_out | (uintptr_t)k_out | (uintptr_t)v_out) & 15) != 0)
        return KVFP8_ESTRIDE;
    const RopeOut out{q_out, k_out, v_out, num_q_heads, num_kv_heads};
    return (int)launch_rope_vec<true>(a, out, dtype, table_dtype, rows * heads * (head_dim / 8),
                                      reinterpret_cast<hipStream_t>(stream));
}

extern "C" int kvfp8_rope_inplace(void* x, int dtype, int64_t rows, int32_t heads, int32_t head_dim,
                                  int64_t row_stride, int64_t head_stride, const void* positions, int pos_dtype,
                                  const void* cos_table, const void* sin_table, int table_dtype,
                                  int64_t table_rows, void* stream) {
    auto is_float = [](int d) { return d == KVFP8_F32 || d == KVFP8_F16 || d == KVFP8_BF16; };
    if (!is_float(dtype) || !is_float(table_dtype)) return KVFP8_EDTYPE;
    if (pos_dtype != KVFP8_I32 && pos_dtype != KVFP8_I64) return KVFP8_EDTYPE;
    if (rows < 0 || heads <= 0 || head_dim <= 0 || head_dim % 2 != 0 || table_rows <= 0) return KVFP8_ESHAPE;
    if (rows == 0) return KVFP8_OK;
    if (!x || !positions || !cos_table || !sin_table) return KVFP8_ENULL;
    RopeArgs a{x, rows, heads, head_dim, row_stride, head_stride, positions, pos_dtype == KVFP8_I64,
               cos_table, sin_table, table_rows};
    if (rows * heads * (head_dim / 2) >= kRopeVecPairs && rope_vec_ok(a, dtype, table_dtype, heads))
        return (int)launch_rope_vec<false>(a, RopeOut{}, dtype, table_dtype, rows * heads * (head_dim / 8),
                                           reinterpret_cast<hipStream_t>(stream));
    const int64_t total = rows * heads * (head_dim / 2);
    int64_t blocks = (total + kRopeThreads - 1) / kRopeThreads;
    blocks = blocks > 65536 ? 65536 : blocks;
    const dim3 grid((unsigned)blocks);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    switch (dtype) {
        case KVFP8_F32: return (int)launch_rope<KVFP8_F32>(a, table_dtype, grid, s);
        case KVFP8_F16: return (int)launch_rope<KVFP8_F16>(a, table_dtype, grid, s);
        default: return (int)launch_rope<KVFP8_BF16>(a, table_dtype, grid, s);
    }
}
