// Causal depthwise conv1d (+ SiLU) on gfx950, forward and backward.
//
// The reference runs this step in PyTorch as nn.Conv1d(groups=dim,
// padding=width - 1) cut to the first seqlen outputs, followed by SiLU
// (modules/mamba_simple.py:40-47,100-101):
//
//   pre[b, d, t] = bias[d] + sum_k w[d, k] * x[b, d, t - (width - 1) + k]   (x = 0 before t = 0)
//   out = silu(pre) or pre
//
// Layout: a workgroup of 256 threads covers 256 VW consecutive steps of one
// (batch, channel) row (grid x: rows, grid y: segments); each thread VW
// consecutive steps, one 16-byte vector: VW = 4 for fp32, 8 for 16-bit
// types.  The vectors need only element alignment (this target accesses
// memory in its unaligned mode: 16-byte loads and stores at any element
// offset), so rows at any offset and of any length keep them; the one
// vector that straddles a row's end is read and written element by element.
// The 3-step halo before a thread's steps comes from the previous vector (an
// L1 / L2 hit).
// The op is HBM-bound: one read of x, one write of out (forward); reads of
// x and dout, one write of dx, and per-workgroup sums of dweight / dbias
// (backward).  The backward's arithmetic is close behind: the SiLU derivative
// of 11 steps for 8 (of 16, every step of the following vector, it took 52
// us at batch 8 x 1536 x 2047 bf16; now 49.5), and its sums over the wave are
// DPP moves, not LDS permutes.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/mamba_ss.h"
#include "row_vec.hpp"
#include "ss_device.hpp"

namespace ss {

namespace {

constexpr int kCT = 256;            // threads per workgroup

// weight and bias come in fp32 or in the rows' type: casting them, and casting
// and clearing their gradients, took eight small launches beside the two; now
// there is one, the fixed-order sum of the gradients (batch 8 x 1536 x 2047 bf16
// forward + backward 118 us with the eight, 109 with the one, its 4 us included)
struct ConvParams {
    int64_t batch, dim, seqlen;
    int32_t width, has_bias, silu;
    int64_t x_bs, x_ds, o_bs, o_ds, w_ds, w_ks;
    int64_t do_bs, do_ds, dx_bs, dx_ds;
    int32_t w_io;                                // weight, bias (and dw, dbias) in the rows' type, not fp32
    int32_t overwrite;                           // dw, dbias: stored, not added to (fixed-order sums)
    const void* x; const void* w; const void* bias; void* out;
    const void* dout; void* dx; void* dw; void* dbias;
    float* part;                                 // fixed-order sums: (row, tile, 5) partials; null: atomics
};

template <typename IT>
__device__ __forceinline__ float ld(const IT* p, int64_t i, int64_t n) {
    // element i of a row of n elements; 0 outside [0, n)
    const float v = io<IT>::load(p + row_elem(i, n));
    return row_in(i, n) ? v : 0.f;
}

// The taps of channel d aligned to the right (w[4 - width .. 3], zeros before)
// and its bias, of type WT.  Every load is unconditional, at a clamped tap: a
// runtime loop or type switch here waits for memory once per tap.
template <typename WT>
__device__ __forceinline__ void load_taps(const ConvParams& p, int64_t d, float (&w)[4], float& bias) {
    const WT* row = static_cast<const WT*>(p.w) + d * p.w_ds;
    const WT* bp = p.has_bias ? static_cast<const WT*>(p.bias) + d : row;
    const WT bv = *bp;
    WT raw[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int tap = k - (4 - p.width);
        raw[k] = row[(tap >= 0 ? tap : 0) * p.w_ks];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = k >= 4 - p.width ? io<WT>::load(&raw[k]) : 0.f;
    bias = p.has_bias ? io<WT>::load(&bv) : 0.f;
}

// 16-byte vectors with element alignment only
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(2)));

// VW consecutive elements starting at i (a multiple of VW; 16 bytes: VW = 4
// fp32, 8 16-bit; any element offset); zeros outside [0, n).  One load where
// row_vec_ok, else element by element.
template <typename IT, int VW, Rows kRows>
__device__ __forceinline__ void ldv(const IT* p, int64_t i, int64_t n, float (&o)[VW]) {
    static_assert(VW * sizeof(IT) == 16, "16-byte vectors");
    const bool in = row_in(i, n);
    if constexpr (kRows != Rows::kWhole) {
        if (!row_vec_ok(kRows, i, n, VW)) {
#pragma unroll
            for (int k = 0; k < VW; ++k) o[k] = ld<IT>(p, i + k, n);
            return;
        }
    }
    const int64_t c = row_vec_at(i, n);
    if constexpr (sizeof(IT) == 4) {
        const f32x4_u v = *reinterpret_cast<const f32x4_u*>(p + c);
        o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    } else {
        const u32x4_u v = *reinterpret_cast<const u32x4_u*>(p + c);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if constexpr (__is_same(IT, bf16_t)) {
                o[2 * k] = __uint_as_float(w[k] << 16);
                o[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
            } else {
                o[2 * k] = float(__builtin_bit_cast(_Float16, uint16_t(w[k] & 0xffffu)));
                o[2 * k + 1] = float(__builtin_bit_cast(_Float16, uint16_t(w[k] >> 16)));
            }
        }
    }
    if (!in) {
#pragma unroll
        for (int k = 0; k < VW; ++k) o[k] = 0.f;
    }
}

// v into elements i .. i + VW - 1 of a row of n (0 <= i < n): one 16-byte
// store, or (not kWhole) element stores of those below n when the vector
// straddles the row's end
template <typename IT, int VW, Rows kRows>
__device__ __forceinline__ void stv(IT* p, int64_t i, int64_t n, const float (&v)[VW]) {
    static_assert(VW * sizeof(IT) == 16, "16-byte vectors");
    if (kRows != Rows::kWhole && i + VW > n) {
#pragma unroll
        for (int k = 0; k < VW; ++k)
            if (i + k < n) io<IT>::store(p + i + k, v[k]);
        return;
    }
    if constexpr (sizeof(IT) == 4) {
        *reinterpret_cast<f32x4_u*>(p + i) = f32x4_u{v[0], v[1], v[2], v[3]};
    } else {
        uint32_t o[VW / 2];
#pragma unroll
        for (int k = 0; k < VW / 2; ++k) {
            if constexpr (__is_same(IT, bf16_t)) {
                o[k] = io<bf16_t>::pack2(v[2 * k], v[2 * k + 1]);
            } else {
                o[k] = uint32_t(__builtin_bit_cast(uint16_t, _Float16(v[2 * k]))) |
                       (uint32_t(__builtin_bit_cast(uint16_t, _Float16(v[2 * k + 1]))) << 16);
            }
        }
        *reinterpret_cast<u32x4_u*>(p + i) = u32x4_u{o[0], o[1], o[2], o[3]};
    }
}

// x[t0 - VW .. t0 + VW * (1 + extra) - 1] into xs
template <typename IT, int VW, Rows kRows, int kExtra>
__device__ __forceinline__ void load_window(const IT* row, int64_t t0, int64_t L, float (&xs)[VW * (2 + kExtra)]) {
#pragma unroll
    for (int q = 0; q < 2 + kExtra; ++q) {
        float v[VW];
        ldv<IT, VW, kRows>(row, t0 - VW + VW * q, L, v);
#pragma unroll
        for (int k = 0; k < VW; ++k) xs[VW * q + k] = v[k];
    }
}

template <typename IT, typename WT, int VW, Rows kRows>
__global__ __launch_bounds__(kCT) void conv1d_fwd_kernel(const ConvParams p) {
    constexpr int V = VW;                               // steps per thread
    const int64_t row_id = blockIdx.x;                  // b * dim + d
    const int64_t b = row_id / p.dim, d = row_id % p.dim;
    const int64_t t0 = int64_t(blockIdx.y) * (kCT * V) + threadIdx.x * V;
    if (t0 >= p.seqlen) return;                         // no barrier in this kernel
    const IT* xr = static_cast<const IT*>(p.x) + b * p.x_bs + d * p.x_ds;
    IT* orow = static_cast<IT*>(p.out) + b * p.o_bs + d * p.o_ds;

    float w[4], bias;
    load_taps<WT>(p, d, w, bias);
    float xs[2 * V];                                    // x[t0 - V .. t0 + V - 1]
    load_window<IT, VW, kRows, 0>(xr, t0, p.seqlen, xs);
    float o[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        float acc = bias;
#pragma unroll
        for (int k = 0; k < 4; ++k) acc = __builtin_fmaf(w[k], xs[V + i - 3 + k], acc);
        o[i] = p.silu ? acc * sigmoidf_(acc) : acc;
    }
    stv<IT, VW, kRows>(orow, t0, p.seqlen, o);
}

template <typename IT, typename WT, int VW, Rows kRows>
__global__ __launch_bounds__(kCT) void conv1d_bwd_kernel(const ConvParams p) {
    constexpr int V = VW;                               // steps per thread
    __shared__ float red[kCT / 64][5];
    const int64_t row_id = blockIdx.x;
    const int64_t b = row_id / p.dim, d = row_id % p.dim;
    const int64_t t0 = int64_t(blockIdx.y) * (kCT * V) + threadIdx.x * V;
    const bool live = t0 < p.seqlen;
    const int64_t tl = live ? t0 : 0;                   // dead threads still join the reduction
    const IT* xr = static_cast<const IT*>(p.x) + b * p.x_bs + d * p.x_ds;
    const IT* gr = static_cast<const IT*>(p.dout) + b * p.do_bs + d * p.do_ds;
    IT* dxr = static_cast<IT*>(p.dx) + b * p.dx_bs + d * p.dx_ds;

    float w[4], bias;
    load_taps<WT>(p, d, w, bias);
    // x[t0 - V .. t0 + 2 V - 1], dout[t0 .. t0 + 2 V - 1]
    float xs[3 * V];
    load_window<IT, VW, kRows, 1>(xr, tl, p.seqlen, xs);
    float gs[2 * V];
    {
        float v[VW];
        ldv<IT, VW, kRows>(gr, tl, p.seqlen, v);
#pragma unroll
        for (int k = 0; k < VW; ++k) gs[k] = v[k];
        ldv<IT, VW, kRows>(gr, tl + VW, p.seqlen, v);
#pragma unroll
        for (int k = 0; k < VW; ++k) gs[VW + k] = v[k];
    }
    // dpre at t0 .. t0 + V + 2, the steps dx reaches (zero beyond seqlen: gs is
    // zero there)
    float dp[V + 3];
#pragma unroll
    for (int i = 0; i < V + 3; ++i) {
        float pre = bias;
#pragma unroll
        for (int k = 0; k < 4; ++k) pre = __builtin_fmaf(w[k], xs[V + i - 3 + k], pre);
        float g = gs[i];
        if (p.silu) {
            const float s = sigmoidf_(pre);
            g *= s * (1.f + pre * (1.f - s));
        }
        dp[i] = g;
    }
    // dx[t] = sum_k w[k] * dpre[t + 3 - k] (taps right-aligned)
    float dxo[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        float acc = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) acc = __builtin_fmaf(w[k], dp[i + 3 - k], acc);
        dxo[i] = acc;
    }
    if (live) stv<IT, VW, kRows>(dxr, t0, p.seqlen, dxo);
    // dw[k] += sum_t dpre[t] * x[t - 3 + k], dbias += sum_t dpre[t], over this thread's V steps
    float part[5];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < V; ++i) acc = __builtin_fmaf(dp[i], xs[V + i - 3 + k], acc);
        part[k] = live ? acc : 0.f;
    }
    {
        float sb = 0.f;
#pragma unroll
        for (int i = 0; i < V; ++i) sb += dp[i];
        part[4] = live ? sb : 0.f;
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) part[k] = wave_allsum(part[k]);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < 5; ++k) red[wv][k] = part[k];
    }
    __syncthreads();
    if (threadIdx.x < 5) {
        const int k = threadIdx.x;
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < kCT / 64; ++i) s += red[i][k];
        if (p.part) {                                   // summed later in a fixed order
            p.part[(row_id * int64_t(gridDim.y) + blockIdx.y) * 5 + k] = s;
            return;
        }
        if (k < 4) {
            const int tap = k - (4 - p.width);          // right-aligned slot k is tap k - (4 - width)
            if (tap >= 0) atomicAdd(static_cast<float*>(p.dw) + d * p.width + tap, s);
        } else if (p.dbias) {
            atomicAdd(static_cast<float*>(p.dbias) + d, s);
        }
    }
}

// dweight / dbias += the backward's partials, a wave per channel: lane l sums
// the (batch row, sequence tile) pairs l, l + 64, ... of each slot (0..3 the
// right-aligned taps, 4 the bias) and the lanes are added as a butterfly, a
// fixed order.  With overwrite, the sums are stored in place of what dweight /
// dbias held, rounded to the weight's type.
template <typename WT>
__global__ __launch_bounds__(64) void conv1d_bwd_reduce(const ConvParams p, int64_t ntiles) {
    const int64_t d = blockIdx.x;
    float s[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    for (int64_t i = threadIdx.x; i < p.batch * ntiles; i += 64) {
        const int64_t b = i / ntiles;
        const float* q = p.part + ((b * p.dim + d) * ntiles + (i - b * ntiles)) * 5;
#pragma unroll
        for (int k = 0; k < 5; ++k) s[k] += q[k];
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] = wave_allsum(s[k]);
    const int k = threadIdx.x, tap = k - (4 - p.width);
    if (k > 4 || (k < 4 && tap < 0) || (k == 4 && !p.dbias)) return;
    const float v = k == 0 ? s[0] : k == 1 ? s[1] : k == 2 ? s[2] : k == 3 ? s[3] : s[4];
    void* out = k < 4 ? p.dw : p.dbias;
    const int64_t o = k < 4 ? d * p.width + tap : d;
    WT* q = static_cast<WT*>(out) + o;
    io<WT>::store(q, p.overwrite ? v : io<WT>::load(q) + v);
}

template <typename IT, typename WT, int VW, Rows kRows>
void launch_vw(const ConvParams& p, bool bwd, hipStream_t stream) {
    constexpr int V = VW;
    const dim3 grid(unsigned(p.batch * p.dim), unsigned((p.seqlen + kCT * V - 1) / (kCT * V)));
    if (bwd) {
        hipLaunchKernelGGL((conv1d_bwd_kernel<IT, WT, VW, kRows>), grid, dim3(kCT), 0, stream, p);
        if (p.part)
            hipLaunchKernelGGL((conv1d_bwd_reduce<WT>), dim3(unsigned(p.dim)), dim3(64), 0, stream, p,
                               int64_t(grid.y));
    } else {
        hipLaunchKernelGGL((conv1d_fwd_kernel<IT, WT, VW, kRows>), grid, dim3(kCT), 0, stream, p);
    }
}

template <typename IT, typename WT>
void launch_w(const ConvParams& p, bool bwd, hipStream_t stream) {
    // 16-byte vectors; rows of whole vectors take the branch-free loads
    constexpr int VW = 16 / sizeof(IT);
    switch (rows_of(p.seqlen, VW)) {
        case Rows::kWhole: return launch_vw<IT, WT, VW, Rows::kWhole>(p, bwd, stream);
        case Rows::kRagged: return launch_vw<IT, WT, VW, Rows::kRagged>(p, bwd, stream);
        case Rows::kShort: return launch_vw<IT, WT, VW, Rows::kShort>(p, bwd, stream);
    }
}

template <typename IT>
hipError_t launch_t(const ConvParams& p, bool bwd, hipStream_t stream) {
    if (p.w_io) launch_w<IT, IT>(p, bwd, stream);
    else launch_w<IT, float>(p, bwd, stream);
    return hipGetLastError();
}

hipError_t launch_conv(const ConvParams& p, int itype, bool bwd, hipStream_t stream) {
    switch (itype) {
        case SS_F32: return launch_t<float>(p, bwd, stream);
        case SS_BF16: return launch_t<bf16_t>(p, bwd, stream);
        case SS_F16: return launch_t<_Float16>(p, bwd, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

int64_t conv1d_bwd_workspace_bytes(int64_t batch, int64_t dim, int64_t seqlen) {
    // the most sequence tiles a launch can have (4 steps per thread)
    const int64_t ntiles = (seqlen + kCT * 4 - 1) / (kCT * 4);
    return batch * dim * ntiles * 5 * int64_t(sizeof(float));
}

hipError_t conv1d_launch(const ss_conv1d_args* a, const ss_conv1d_bwd_args* g, int w_dtype, bool overwrite,
                         hipStream_t stream) {
    ConvParams p{};
    p.batch = a->batch; p.dim = a->dim; p.seqlen = a->seqlen; p.width = int32_t(a->width);
    p.has_bias = a->has_bias; p.silu = a->silu;
    p.x_bs = a->x_batch_stride; p.x_ds = a->x_dim_stride;
    p.o_bs = a->out_batch_stride; p.o_ds = a->out_dim_stride;
    p.w_ds = a->w_dim_stride; p.w_ks = a->w_width_stride;
    p.x = a->x; p.w = a->weight; p.bias = a->has_bias ? a->bias : nullptr; p.out = a->out;
    if (g) {
        p.do_bs = g->dout_batch_stride; p.do_ds = g->dout_dim_stride;
        p.dx_bs = g->dx_batch_stride; p.dx_ds = g->dx_dim_stride;
        p.dout = g->dout; p.dx = g->dx; p.dw = g->dweight; p.dbias = a->has_bias ? g->dbias : nullptr;
        p.part = g->workspace;
    }
    p.w_io = w_dtype != SS_F32;
    p.overwrite = overwrite;
    return launch_conv(p, a->itype, g != nullptr, stream);
}

}  // namespace ss
