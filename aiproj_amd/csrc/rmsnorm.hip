// RMSNorm forward for the decode and prefill steps (gfx950), optionally fused with
// the residual add that precedes it, and its backward.
//
// Replaces the Triton `rmsnorm_kernal` of reference
// src/torch_llm/model/rmsnorm.py:60-113 (its backward
// is further below):
//   inv_rms = 1 / sqrt(mean(x^2) + eps)        (float32)
//   out     = (x * inv_rms) * weight           (float32, stored in x's dtype)
// The fused form first forms the residual sum s = x + update in float32, rounds
// it to the state dtype (what `state + update` stores, reference
// model/residual.py:33-35) and normalizes that rounded value.
//
// One wave per row, rows grid-strided over the launch. A lane holds 8 elements
// (one 16-byte vector of a 16-bit dtype) per 512-element chunk of the row, so a
// row of up to 4096 elements stays in registers between the reduction and the
// scaling; longer rows are read twice.
#include "kvfp8_common.h"

namespace kvfp8 {

constexpr int kNormThreads = 256;
constexpr int kNormVec = 8;          // elements per lane per chunk
constexpr int kNormChunks = 8;       // chunks kept in registers (4096 elements)

struct NormArgs {
    const void* x;
    const void* update;     // null: plain RMSNorm
    const void* weight;
    void* out;
    void* state_out;        // fused form: x + update in x's dtype
    float* inv_rms;         // may be null
    int64_t rows;
    int32_t d_model;
    int64_t x_stride, update_stride, out_stride, state_stride;   // elements
    float eps;
};

template <int DT>
__device__ __forceinline__ void load8(const typename Elem<DT>::T* p, bool vec, int n, float (&v)[kNormVec]) {
    using T = typename Elem<DT>::T;
    if (vec && n == kNormVec) {
        if constexpr (sizeof(T) == 2) {
            const uint4 raw = *reinterpret_cast<const uint4*>(p);
            const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
            for (int i = 0; i < kNormVec; ++i) v[i] = Elem<DT>::load(e[i]);
        } else {
            const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
            v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < kNormVec; ++i) v[i] = i < n ? Elem<DT>::load(p[i]) : 0.0f;
    }
}

template <int DT>
__device__ __forceinline__ void store8(typename Elem<DT>::T* p, bool vec, int n, const float (&v)[kNormVec]) {
    using T = typename Elem<DT>::T;
    if (vec && n == kNormVec) {
        if constexpr (sizeof(T) == 2) {
            T e[kNormVec];
#pragma unroll
            for (int i = 0; i < kNormVec; ++i) e[i] = Elem<DT>::store(v[i]);
            *reinterpret_cast<uint4*>(p) = *reinterpret_cast<const uint4*>(e);
        } else {
            reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
            reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < kNormVec; ++i)
            if (i < n) p[i] = Elem<DT>::store(v[i]);
    }
}

// Row element of the (possibly fused) input: x, or round(x + update) to x's dtype.
template <int DT, bool kFused>
__device__ __forceinline__ void row_chunk(const NormArgs& a, int64_t r, int d0, int n, bool vec, float (&v)[kNormVec]) {
    using T = typename Elem<DT>::T;
    load8<DT>(reinterpret_cast<const T*>(a.x) + r * a.x_stride + d0, vec, n, v);
    if constexpr (kFused) {
        float u[kNormVec];
        load8<DT>(reinterpret_cast<const T*>(a.update) + r * a.update_stride + d0, vec, n, u);
#pragma unroll
        for (int i = 0; i < kNormVec; ++i) v[i] = Elem<DT>::load(Elem<DT>::store(v[i] + u[i]));
    }
}

template <int DT, int WT, bool kFused>
__global__ void __launch_bounds__(kNormThreads)
rmsnorm_kernel(NormArgs a, int vec_ok) {
    using T = typename Elem<DT>::T;
    using W = typename Elem<WT>::T;
    const int lane = threadIdx.x & 63;
    const int64_t wave0 = ((int64_t)blockIdx.x * kNormThreads + threadIdx.x) >> 6;
    const int64_t waves = ((int64_t)gridDim.x * kNormThreads) >> 6;
    const int D = a.d_model;
    const int chunk = 64 * kNormVec;
    const int nchunks = (D + chunk - 1) / chunk;
    const bool cached = nchunks <= kNormChunks;
    const bool vec = vec_ok != 0;

    for (int64_t r = wave0; r < a.rows; r += waves) {
        float ss = 0.0f;
        if (cached) {
            // Every load of the row (x, update, weight) is issued before the first
            // store, so no store can order the loads behind it (outputs may alias).
            float v[kNormChunks][kNormVec], w[kNormChunks][kNormVec];
#pragma unroll
            for (int c = 0; c < kNormChunks; ++c) {
                const int d0 = c * chunk + lane * kNormVec;
                const int n = c < nchunks ? max(0, min(kNormVec, D - d0)) : 0;
                if (n > 0) {
                    row_chunk<DT, kFused>(a, r, d0, n, vec, v[c]);
                    load8<WT>(reinterpret_cast<const W*>(a.weight) + d0, vec, n, w[c]);
                } else {
#pragma unroll
                    for (int i = 0; i < kNormVec; ++i) v[c][i] = w[c][i] = 0.0f;
                }
            }
#pragma unroll
            for (int c = 0; c < kNormChunks; ++c) {
#pragma unroll
                for (int i = 0; i < kNormVec; ++i) ss += v[c][i] * v[c][i];
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
            const float inv = 1.0f / sqrtf(ss / (float)D + a.eps);
            if (lane == 0 && a.inv_rms) a.inv_rms[r] = inv;
#pragma unroll
            for (int c = 0; c < kNormChunks; ++c) {
                const int d0 = c * chunk + lane * kNormVec;
                const int n = c < nchunks ? max(0, min(kNormVec, D - d0)) : 0;
                if (n <= 0) continue;
                if constexpr (kFused) store8<DT>(reinterpret_cast<T*>(a.state_out) + r * a.state_stride + d0, vec, n, v[c]);
                float o[kNormVec];
#pragma unroll
                for (int i = 0; i < kNormVec; ++i) o[i] = (v[c][i] * inv) * w[c][i];
                store8<DT>(reinterpret_cast<T*>(a.out) + r * a.out_stride + d0, vec, n, o);
            }
        } else {
            for (int c = 0; c < nchunks; ++c) {
                const int d0 = c * chunk + lane * kNormVec;
                const int n = max(0, min(kNormVec, D - d0));
                float t[kNormVec];
                row_chunk<DT, kFused>(a, r, d0, n, vec, t);
                if constexpr (kFused) {
                    if (n > 0) store8<DT>(reinterpret_cast<T*>(a.state_out) + r * a.state_stride + d0, vec, n, t);
                }
#pragma unroll
                for (int i = 0; i < kNormVec; ++i) ss += t[i] * t[i];
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
            const float inv = 1.0f / sqrtf(ss / (float)D + a.eps);
            if (lane == 0 && a.inv_rms) a.inv_rms[r] = inv;
            for (int c = 0; c < nchunks; ++c) {
                const int d0 = c * chunk + lane * kNormVec;
                const int n = max(0, min(kNormVec, D - d0));
                if (n <= 0) continue;
                float t[kNormVec], w[kNormVec];
                // The fused form re-reads the rounded sum it stored above.
                if constexpr (kFused)
                    load8<DT>(reinterpret_cast<const T*>(a.state_out) + r * a.state_stride + d0, vec, n, t);
                else
                    row_chunk<DT, false>(a, r, d0, n, vec, t);
                load8<WT>(reinterpret_cast<const W*>(a.weight) + d0, vec, n, w);
#pragma unroll
                for (int i = 0; i < kNormVec; ++i) t[i] = (t[i] * inv) * w[i];
                store8<DT>(reinterpret_cast<T*>(a.out) + r * a.out_stride + d0, vec, n, t);
            }
        }
    }
}

// One workgroup per row (grid-strided over the rows) for aligned rows of up to
// 256 x 8 x VPT elements: thread t owns the 16-byte vectors t, t + 256, ... of the
// row in every tensor, so the row is read once, with 256 independent loads in
// flight per tensor. The sum of squares is reduced across the wave (shuffles)
// and then across the four waves through LDS, with one barrier per row (the LDS
// slot alternates by row parity, so a fast wave writing row r + 2 cannot overwrite
// values a slow wave still reads for row r: the barrier of row r + 1 lies between).
// A decode step's 64 rows then run as 64 workgroups instead of 64 waves.
template <int DT, int WT, bool kFused, int VPT>
__global__ void __launch_bounds__(kNormThreads)
rmsnorm_row_kernel(NormArgs a) {
    using T = typename Elem<DT>::T;
    using W = typename Elem<WT>::T;
    __shared__ float partial[2][kNormThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int D = a.d_model;
    float w[VPT][kNormVec];
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int d0 = (tid + kNormThreads * k) * kNormVec;
        load8<WT>(reinterpret_cast<const W*>(a.weight) + d0, true, d0 < D ? kNormVec : 0, w[k]);
    }
    int parity = 0;
    for (int64_t r = blockIdx.x; r < a.rows; r += gridDim.x, parity ^= 1) {
        float v[VPT][kNormVec];
        float ss = 0.0f;
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            const int d0 = (tid + kNormThreads * k) * kNormVec;
            if (d0 < D) {
                row_chunk<DT, kFused>(a, r, d0, kNormVec, true, v[k]);
            } else {
#pragma unroll
                for (int i = 0; i < kNormVec; ++i) v[k][i] = 0.0f;
            }
#pragma unroll
            for (int i = 0; i < kNormVec; ++i) ss += v[k][i] * v[k][i];
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
        if (lane == 0) partial[parity][wave] = ss;
        __syncthreads();
        float total = 0.0f;
#pragma unroll
        for (int i = 0; i < kNormThreads / 64; ++i) total += partial[parity][i];
        const float inv = 1.0f / sqrtf(total / (float)D + a.eps);
        if (tid == 0 && a.inv_rms) a.inv_rms[r] = inv;
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            const int d0 = (tid + kNormThreads * k) * kNormVec;
            if (d0 >= D) continue;
            if constexpr (kFused) store8<DT>(reinterpret_cast<T*>(a.state_out) + r * a.state_stride + d0, true, kNormVec, v[k]);
            float o[kNormVec];
#pragma unroll
            for (int i = 0; i < kNormVec; ++i) o[i] = (v[k][i] * inv) * w[k][i];
            store8<DT>(reinterpret_cast<T*>(a.out) + r * a.out_stride + d0, true, kNormVec, o);
        }
    }
}

// ---------------------------------------------------------------------------
// Backward of one norm (reference model/rmsnorm.py: training), float32 throughout:
//   xhat = x inv_rms, gw = grad weight
//   dx = inv_rms (gw - xhat mean(gw xhat)),  dw = sum over rows of grad xhat
// Bound: HBM, x and grad read once and dx written once. The rows' parts of dw stay in
// registers; a workgroup writes one row of partial sums, which norm_weight_grad_kernel adds
// in a fixed order. Rows of up to 1024 elements take one wave each and no barrier: a lane
// holds the row's vectors of 8 elements l, l + 64 (CH of them). Longer rows take a workgroup
// each: with four vectors per lane and tensor a wave would spill (2048 elements: 67 us for
// the kernel). Every workgroup gets the same number of rows (the last one excepted): with
// 1024 workgroups at most, no round of rows is nearly empty.
// Measured (8704 x 2048 bf16): 20.6 us for this kernel (5.2 TB/s) and 5 us for the sums,
// against 266 us as PyTorch's float32 operations; forward and backward 313 -> 108 us, which
// is the host's time (forward kernel 16 us).
// ---------------------------------------------------------------------------
constexpr int kNormBwdBlocks = 1024;

struct NormBwdArgs {
    const void* x;
    const void* grad;
    const void* weight;
    const float* inv_rms;
    void* dx;
    float* part;            // [workgroup][d_model]
    int64_t rows;
    int32_t d_model, w_dtype;
    int64_t x_stride, grad_stride, dx_stride;    // elements
};

template <typename T>
struct alignas(16) RawRow {
    T e[kNormVec];
};

// Eight weights from d0 (zeros past the row).
__device__ __forceinline__ void load_weight(const NormBwdArgs& a, int d0, float (&w)[kNormVec]) {
    const int n = d0 < a.d_model ? kNormVec : 0;
    if (a.w_dtype == KVFP8_F32) load8<KVFP8_F32>(reinterpret_cast<const float*>(a.weight) + d0, true, n, w);
    else if (a.w_dtype == KVFP8_F16) load8<KVFP8_F16>(reinterpret_cast<const uint16_t*>(a.weight) + d0, true, n, w);
    else load8<KVFP8_BF16>(reinterpret_cast<const uint16_t*>(a.weight) + d0, true, n, w);
}

template <int DT, int CH>
__global__ void __launch_bounds__(kNormThreads)
rmsnorm_backward_kernel(NormBwdArgs a) {
    using T = typename Elem<DT>::T;
    __shared__ float sums[kNormThreads / 64][64 * kNormVec];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int D = a.d_model;
    float dw[CH][kNormVec];
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int i = 0; i < kNormVec; ++i) dw[c][i] = 0.0f;

    for (int64_t r = (int64_t)blockIdx.x * 4 + wave; r < a.rows; r += (int64_t)gridDim.x * 4) {
        const T* const x = reinterpret_cast<const T*>(a.x) + r * a.x_stride;
        const T* const g = reinterpret_cast<const T*>(a.grad) + r * a.grad_stride;
        const float inv = a.inv_rms[r];
        RawRow<T> xr[CH], gr[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int d0 = (64 * c + lane) * kNormVec;
            if (d0 < D) {
                xr[c] = *reinterpret_cast<const RawRow<T>*>(x + d0);
                gr[c] = *reinterpret_cast<const RawRow<T>*>(g + d0);
            } else {
                xr[c] = gr[c] = RawRow<T>{};
            }
        }
        float dot = 0.0f;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            float w[kNormVec];
            load_weight(a, (64 * c + lane) * kNormVec, w);
#pragma unroll
            for (int i = 0; i < kNormVec; ++i) {
                const float xh = Elem<DT>::load(xr[c].e[i]) * inv, gi = Elem<DT>::load(gr[c].e[i]);
                dw[c][i] += gi * xh;
                dot += (gi * w[i]) * xh;
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off);
        const float mean = dot / (float)D;
        T* const dx = reinterpret_cast<T*>(a.dx) + r * a.dx_stride;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int d0 = (64 * c + lane) * kNormVec;
            if (d0 >= D) continue;
            float w[kNormVec], o[kNormVec];
            load_weight(a, d0, w);
#pragma unroll
            for (int i = 0; i < kNormVec; ++i) {
                const float xh = Elem<DT>::load(xr[c].e[i]) * inv;
                o[i] = inv * (Elem<DT>::load(gr[c].e[i]) * w[i] - xh * mean);
            }
            store8<DT>(dx + d0, true, kNormVec, o);
        }
    }

    float* const part = a.part + (int64_t)blockIdx.x * D;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        if (c > 0) __syncthreads();
        float4* const mine = reinterpret_cast<float4*>(&sums[wave][lane * kNormVec]);
        mine[0] = make_float4(dw[c][0], dw[c][1], dw[c][2], dw[c][3]);
        mine[1] = make_float4(dw[c][4], dw[c][5], dw[c][6], dw[c][7]);
        __syncthreads();
        const int e = threadIdx.x * 2, d0 = 64 * kNormVec * c + e;
        if (d0 < D) {
            float2 sum = *reinterpret_cast<const float2*>(&sums[0][e]);
#pragma unroll
            for (int w = 1; w < kNormThreads / 64; ++w) {
                const float2 y = *reinterpret_cast<const float2*>(&sums[w][e]);
                sum.x += y.x;
                sum.y += y.y;
            }
            *reinterpret_cast<float2*>(part + d0) = sum;
        }
    }
}

// Rows of up to 2048 VPT elements, one workgroup each: thread t owns vectors t, t + 256, ...
// The next row's vectors load while this row is reduced; the LDS slot of the row sum
// alternates by row parity, as in rmsnorm_row_kernel.
template <int DT, int VPT>
__global__ void __launch_bounds__(kNormThreads)
rmsnorm_backward_row_kernel(NormBwdArgs a) {
    using T = typename Elem<DT>::T;
    __shared__ float partial[2][kNormThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int D = a.d_model;
    float w[VPT][kNormVec], dw[VPT][kNormVec];
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        load_weight(a, (tid + kNormThreads * k) * kNormVec, w[k]);
#pragma unroll
        for (int i = 0; i < kNormVec; ++i) dw[k][i] = 0.0f;
    }
    RawRow<T> xr[VPT], gr[VPT];
    float inv = 0.0f;
    auto load_row = [&](int64_t r) __attribute__((always_inline)) {
        const T* const x = reinterpret_cast<const T*>(a.x) + r * a.x_stride;
        const T* const g = reinterpret_cast<const T*>(a.grad) + r * a.grad_stride;
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            const int d0 = (tid + kNormThreads * k) * kNormVec;
            if (d0 < D) {
                xr[k] = *reinterpret_cast<const RawRow<T>*>(x + d0);
                gr[k] = *reinterpret_cast<const RawRow<T>*>(g + d0);
            } else {
                xr[k] = gr[k] = RawRow<T>{};
            }
        }
        inv = a.inv_rms[r];
    };
    load_row(blockIdx.x);                       // the grid is no larger than the rows
    int parity = 0;
    for (int64_t r = blockIdx.x; r < a.rows; r += gridDim.x, parity ^= 1) {
        float xh[VPT][kNormVec], gw[VPT][kNormVec], dot = 0.0f;
        const float row_inv = inv;
#pragma unroll
        for (int k = 0; k < VPT; ++k)
#pragma unroll
            for (int i = 0; i < kNormVec; ++i) {
                xh[k][i] = Elem<DT>::load(xr[k].e[i]) * inv;
                const float g = Elem<DT>::load(gr[k].e[i]);
                dw[k][i] += g * xh[k][i];
                gw[k][i] = g * w[k][i];
                dot += gw[k][i] * xh[k][i];
            }
        if (r + gridDim.x < a.rows) load_row(r + gridDim.x);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off);
        if (lane == 0) partial[parity][wave] = dot;
        __syncthreads();
        float total = 0.0f;
#pragma unroll
        for (int i = 0; i < kNormThreads / 64; ++i) total += partial[parity][i];
        const float mean = total / (float)D;
        T* const dx = reinterpret_cast<T*>(a.dx) + r * a.dx_stride;
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            const int d0 = (tid + kNormThreads * k) * kNormVec;
            if (d0 >= D) continue;
            float o[kNormVec];
#pragma unroll
            for (int i = 0; i < kNormVec; ++i) o[i] = row_inv * (gw[k][i] - xh[k][i] * mean);
            store8<DT>(dx + d0, true, kNormVec, o);
        }
    }
    float* const part = a.part + (int64_t)blockIdx.x * D;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int d0 = (tid + kNormThreads * k) * kNormVec;
        if (d0 < D) store8<KVFP8_F32>(part + d0, true, kNormVec, dw[k]);
    }
}

// dw[d] = sum over workgroups of their partial sums: 32 columns per workgroup, 32 groups of
// eight lanes down the rows, joined through LDS.
__global__ void __launch_bounds__(kNormThreads)
norm_weight_grad_kernel(const float* part, int32_t blocks, int32_t D, int32_t w_dtype, void* dw) {
    __shared__ float4 sums[32][8];
    const int col = threadIdx.x & 7, group = threadIdx.x >> 3;
    const int d0 = blockIdx.x * 32 + 4 * col;
    float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (d0 < D) {
#pragma unroll 4
        for (int b = group; b < blocks; b += 32) {
            const float4 y = *reinterpret_cast<const float4*>(part + (int64_t)b * D + d0);
            sum.x += y.x;
            sum.y += y.y;
            sum.z += y.z;
            sum.w += y.w;
        }
    }
    sums[group][col] = sum;
    __syncthreads();
    if (threadIdx.x < 32) {
        const int d = blockIdx.x * 32 + threadIdx.x;
        float total = 0.0f;
        for (int g = 0; g < 32; ++g) total += reinterpret_cast<const float*>(&sums[g][0])[threadIdx.x];
        if (d < D) {
            if (w_dtype == KVFP8_F32) reinterpret_cast<float*>(dw)[d] = total;
            else reinterpret_cast<uint16_t*>(dw)[d] = w_dtype == KVFP8_F16 ? f32_to_f16(total) : f32_to_bf16(total);
        }
    }
}

}  // namespace kvfp8

using namespace kvfp8;

namespace {

int esize(int dt) { return dt == KVFP8_F32 ? 4 : 2; }

bool is_float(int dt) { return dt == KVFP8_F32 || dt == KVFP8_F16 || dt == KVFP8_BF16; }

bool aligned(const void* p, int64_t stride_elems, int es) {
    return p == nullptr || (((uintptr_t)p % 16) == 0 && (stride_elems * es) % 16 == 0);
}

template <int DT, int WT, bool F>
hipError_t launch_norm(const NormArgs& a, hipStream_t s) {
    const int es = esize(DT);
    const bool vec = a.d_model % kNormVec == 0 && aligned(a.x, a.x_stride, es) && aligned(a.out, a.out_stride, es) &&
                     aligned(a.update, a.update_stride, es) && aligned(a.state_out, a.state_stride, es) &&
                     aligned(a.weight, 0, esize(WT));
    // Aligned rows of up to 8192 elements: a workgroup per row (at most 4096
    // workgroups in flight, each then loops over rows).
    const int vectors = (a.d_model + kNormVec - 1) / kNormVec;
    if (vec && vectors <= 4 * kNormThreads) {
        const int vpt = (vectors + kNormThreads - 1) / kNormThreads;
        const dim3 grid((unsigned)(a.rows < 4096 ? a.rows : 4096)), block(kNormThreads);
        if (vpt == 1) hipLaunchKernelGGL((rmsnorm_row_kernel<DT, WT, F, 1>), grid, block, 0, s, a);
        else if (vpt == 2) hipLaunchKernelGGL((rmsnorm_row_kernel<DT, WT, F, 2>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((rmsnorm_row_kernel<DT, WT, F, 4>), grid, block, 0, s, a);
        return hipGetLastError();
    }
    int64_t blocks = (a.rows + 3) / 4;
    blocks = blocks < 1 ? 1 : (blocks > 65536 ? 65536 : blocks);
    hipLaunchKernelGGL((rmsnorm_kernel<DT, WT, F>), dim3((unsigned)blocks), dim3(kNormThreads), 0, s, a, (int)vec);
    return hipGetLastError();
}

template <int DT, bool F>
hipError_t dispatch_weight(const NormArgs& a, int w_dtype, hipStream_t s) {
    switch (w_dtype) {
        case KVFP8_F32: return launch_norm<DT, KVFP8_F32, F>(a, s);
        case KVFP8_F16: return launch_norm<DT, KVFP8_F16, F>(a, s);
        default: return launch_norm<DT, KVFP8_BF16, F>(a, s);
    }
}

template <bool F>
hipError_t dispatch_norm(const NormArgs& a, int dtype, int w_dtype, hipStream_t s) {
    switch (dtype) {
        case KVFP8_F32: return dispatch_weight<KVFP8_F32, F>(a, w_dtype, s);
        case KVFP8_F16: return dispatch_weight<KVFP8_F16, F>(a, w_dtype, s);
        default: return dispatch_weight<KVFP8_BF16, F>(a, w_dtype, s);
    }
}

int check_norm(const void* x, int dtype, int64_t rows, int32_t d_model, const void* weight, int w_dtype,
               const void* out) {
    if (!is_float(dtype) || !is_float(w_dtype)) return KVFP8_EDTYPE;
    if (rows < 0 || d_model <= 0) return KVFP8_ESHAPE;
    if (rows > 0 && (!x || !weight || !out)) return KVFP8_ENULL;
    return KVFP8_OK;
}

// Workgroups of the backward: all take the same number of rows (four at a time up to 1024
// elements, where a wave takes a row).
int64_t norm_backward_blocks(int64_t rows, int32_t d_model) {
    const int64_t at_once = d_model <= 2 * 64 * kNormVec ? 4 : 1;
    const int64_t rounds = (rows + at_once * kNormBwdBlocks - 1) / (at_once * kNormBwdBlocks);
    return rounds == 0 ? 0 : (rows + at_once * rounds - 1) / (at_once * rounds);
}

template <int DT>
hipError_t launch_norm_backward(const NormBwdArgs& a, int64_t blocks, hipStream_t s) {
    const dim3 grid((unsigned)blocks), block(kNormThreads);
    const int chunks = (a.d_model + 64 * kNormVec - 1) / (64 * kNormVec);
    if (chunks == 1) hipLaunchKernelGGL((rmsnorm_backward_kernel<DT, 1>), grid, block, 0, s, a);
    else if (chunks == 2) hipLaunchKernelGGL((rmsnorm_backward_kernel<DT, 2>), grid, block, 0, s, a);
    else if (chunks <= 4) hipLaunchKernelGGL((rmsnorm_backward_row_kernel<DT, 1>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((rmsnorm_backward_row_kernel<DT, 2>), grid, block, 0, s, a);
    return hipGetLastError();
}

}  // namespace

extern "C" int kvfp8_rmsnorm_forward(const void* x, int dtype, int64_t x_stride, int64_t rows, int32_t d_model,
                                     const void* weight, int w_dtype, float eps, void* out, int64_t out_stride,
                                     float* inv_rms, void* stream) {
    const int rc = check_norm(x, dtype, rows, d_model, weight, w_dtype, out);
    if (rc != KVFP8_OK || rows == 0) return rc;
    NormArgs a{x, nullptr, weight, out, nullptr, inv_rms, rows, d_model, x_stride, 0, out_stride, 0, eps};
    return (int)dispatch_norm<false>(a, dtype, w_dtype, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int kvfp8_add_rmsnorm_forward(const void* x, const void* update, int dtype, int64_t x_stride,
                                         int64_t update_stride, int64_t rows, int32_t d_model, const void* weight,
                                         int w_dtype, float eps, void* state_out, int64_t state_stride, void* out,
                                         int64_t out_stride, float* inv_rms, void* stream) {
    int rc = check_norm(x, dtype, rows, d_model, weight, w_dtype, out);
    if (rc != KVFP8_OK || rows == 0) return rc;
    if (!update || !state_out) return KVFP8_ENULL;
    NormArgs a{x, update, weight, out, state_out, inv_rms, rows, d_model, x_stride, update_stride, out_stride,
               state_stride, eps};
    return (int)dispatch_norm<true>(a, dtype, w_dtype, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int64_t kvfp8_rmsnorm_backward_workspace_bytes(int64_t rows, int32_t d_model) {
    if (rows < 0 || d_model <= 0) return KVFP8_ESHAPE;
    if (d_model % kNormVec != 0 || d_model > 64 * kNormVec * kNormChunks) return KVFP8_ELIMIT;
    return norm_backward_blocks(rows, d_model) * d_model * 4;
}

extern "C" int kvfp8_rmsnorm_backward(const void* x, const void* grad, int dtype, int64_t x_stride,
                                      int64_t grad_stride, int64_t rows, int32_t d_model, const void* weight,
                                      int w_dtype, const float* inv_rms, void* dx, int64_t dx_stride, void* dw,
                                      void* workspace, int64_t workspace_bytes, void* stream) {
    const int rc = check_norm(x, dtype, rows, d_model, weight, w_dtype, dx);
    if (rc != KVFP8_OK) return rc;
    const int64_t need = kvfp8_rmsnorm_backward_workspace_bytes(rows, d_model);
    if (need < 0) return (int)need;
    if (!weight || !dw || (rows > 0 && (!grad || !inv_rms || !workspace))) return KVFP8_ENULL;
    const int es = esize(dtype);
    if (!aligned(x, x_stride, es) || !aligned(grad, grad_stride, es) || !aligned(dx, dx_stride, es) ||
        !aligned(weight, 0, esize(w_dtype)) || !aligned(workspace, 0, 4))
        return KVFP8_ESTRIDE;
    if (workspace_bytes < need) return KVFP8_EWORKSPACE;
    NormBwdArgs a{x, grad, weight, inv_rms, dx, reinterpret_cast<float*>(workspace), rows, d_model, w_dtype,
                  x_stride, grad_stride, dx_stride};
    const int64_t blocks = norm_backward_blocks(rows, d_model);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (rows > 0) {
        hipError_t err;
        switch (dtype) {
            case KVFP8_F32: err = launch_norm_backward<KVFP8_F32>(a, blocks, s); break;
            case KVFP8_F16: err = launch_norm_backward<KVFP8_F16>(a, blocks, s); break;
            default: err = launch_norm_backward<KVFP8_BF16>(a, blocks, s); break;
        }
        if (err != hipSuccess) return (int)err;
    }
    hipLaunchKernelGGL(norm_weight_grad_kernel, dim3((unsigned)((d_model + 31) / 32)), dim3(kNormThreads), 0, s, a.part,
                       (int32_t)blocks, d_model, w_dtype, dw);
    return (int)hipGetLastError();
}
