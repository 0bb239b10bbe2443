// Decode-size linear layer on gfx950's matrix cores:
//
//   Y[b, n] = sum_k X[b, k] * W[n, k] (+ bias[n])      (nn.Linear's layout)
//
// for the few rows b of a single-token step (the block's in-, x-, delta- and
// out-projections at batch <= 64).  Such a product streams the weight once
// and does little arithmetic per byte; the library GEMMs choose large tiles
// for it and take several times the weight's streaming time.
//
// A workgroup computes a 16 (n) x 16 (b) tile of Y, or one slice of K of
// it, with NW waves that take every NW-th K step; each K step is one MFMA
// with the W tile (16 n x KS k) as A and the X tile (KS k x 16 b) as B.
// With 16-byte aligned rows and k_in a multiple of 32 a K step covers 32 k
// on gfx950's v_mfma_f32_16x16x32_bf16 (or f16):
//   A: lane l holds W[n0 + (l & 15)][8 (l >> 4) .. + 7] (one 16-byte load)
//   B: lane l holds X[b0 + (l & 15)][the same 8 k]
//   D: lane l holds Y[b0 + (l & 15)][n0 + 4 (l >> 4) + v], v = 0..3
// otherwise 16 k on v_mfma_f32_16x16x16_bf16 (or f16), with lane l holding
// W[n0 + (l & 15)][4 (l >> 4) .. + 3] and the same k of its X row (an
// 8-byte load each).  The
// wave count grows with the steps a workgroup has (4, 8 or 16) so that a
// wave requests all its steps before it uses any.  The partial tiles of the
// waves are summed through LDS.
//
// Split K: a workgroup's time grows with the K it covers (measured on a
// 16 x 16 tile: 3.1 us at K = 48, 5.7 at 768, 9.0 at 1536, whatever the
// wave count), and a decode product can have very few tiles (5 for the
// x-projection of a 1536-wide block).  For such shapes (fewer than
// kLinSplitMaxTiles tiles) and a workspace, the K range of a tile is cut
// into slices, one workgroup each; each puts its fp32 partial tile into a
// slot, and the last of a tile's workgroups to arrive (a per-tile counter)
// sums the slots in slice order, so the result does not depend on which
// one finishes last, and puts the counter back to zero for the next call.
// The exchange costs about three dependent atomic round trips and grows
// with the atomics it issues, so it pays only where the tiles are few
// (x-projection, 5 tiles: 9.0 -> 5.25 us with 4 slices, 5.8 with 16; output
// projection, 48 tiles: 9.06 -> 6.04 us with 4; the 192-tile input
// projection loses with 2), and each slot moves as 64-bit swaps of two
// outputs.  It uses atomics only: an agent-scope fence writes back and
// invalidates the
// whole L2 of its XCD, which made every workgroup's weight reads miss (53 us
// instead of 5.7 for the 768 x 3072 input projection).  The counters have a
// fixed region ahead of the partials, so calls of different shapes can
// share a workspace.
//
// Epilogue: the bias is added in fp32 and the result rounded once; with a
// conv update the rounded product of an output n < conv.dim is the input of
// that channel's causal conv step (state shifted in place, conv output
// written to Y).  Rows n >= N and b >= B read as zero (clamped addresses)
// and are not stored, so every access stays in bounds.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/mamba_ss.h"
#include "ss_device.hpp"
#include "ss_kernels.hpp"

namespace ss {

namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ f32x4 mfma16(s16x4 a, s16x4 b, f32x4 c) {
    if constexpr (__is_same(T, bf16_t)) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h16x4, a), __builtin_bit_cast(h16x4, b), c,
                                                     0, 0, 0);
    }
}

// 16 x 16 x 32 product (gfx950): 8 k per lane
template <typename T>
__device__ __forceinline__ f32x4 mfma32(s16x8 a, s16x8 b, f32x4 c) {
    if constexpr (__is_same(T, bf16_t)) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b16x8, a), __builtin_bit_cast(b16x8, b), c,
                                                       0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h16x8, a), __builtin_bit_cast(h16x8, b), c,
                                                      0, 0, 0);
    }
}

// KV elements of a row (KV = 4: 8 bytes, KV = 8: 16 bytes)
template <int KV>
using rowvec = short __attribute__((ext_vector_type(KV)));

// v rounded to T and back to float (round to nearest even)
template <typename T>
__device__ __forceinline__ float round_io(float v) {
    if constexpr (__is_same(T, bf16_t)) return __uint_as_float(uint32_t(io<bf16_t>::round(v)) << 16);
    else return float(_Float16(v));
}

// What a launch reads, packed: the kernel asks for all of it at its start, in
// a few scalar loads that it waits for once.  (Taken from the C ABI's structs
// where they were used, the arguments came in five dependent waits, each a
// miss of the scalar cache, and with 64-bit index divisions and loads
// converted inside branches the input projection took 10.0 us, its 24 KB of
// weights per workgroup cached or not; this form takes 7.2 us, and the two
// split projections 5.0 us instead of 6.4.  s_memtime stamps of the former:
// 2.3 us to the last load's issue, 0.8 us waiting for it, 2.2 us normalising,
// 0.4 us for the products, 0.7 us to the end, most of it instruction fetch.)
struct LinArgs {
    const void* weight;
    const void* x;
    void* y;
    int64_t w_ld, x_ld, y_ld;          // row strides, elements
    int64_t n_out, k_in, kslice, conv_dim;   // kslice: K elements per workgroup of a tile
    int32_t batch, ksplit, has_conv, bias_f32;
    const void* bias;
    int* counters;                     // split K: per tile, in the workspace
    float* partials;                   // (tile, slice, 256) fp32, in the workspace
    // the RMSNorm in front of the product
    const void* nx;
    const void* nres;
    const void* nw;
    void* ns;
    float* nrstd;
    int64_t nx_ld, nres_ld, ns_ld;
    float eps;
    int32_t nw_f32;
    // the conv step behind it
    void* conv_state;
    const float* conv_w;
    const float* conv_bias;
    int64_t cs_b, cs_d, cs_w, cw_d, cw_w;
    int32_t conv_width, conv_silu;
};

// 16-byte vector of T <-> 8 floats (bf16 / fp16 only)
template <typename T>
__device__ __forceinline__ void unpack8(const uint4& v, float (&o)[8]) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if constexpr (__is_same(T, bf16_t)) {
            o[2 * k] = __uint_as_float(w[k] << 16);
            o[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
        } else {
            o[2 * k] = float(__builtin_bit_cast(_Float16, uint16_t(w[k] & 0xffffu)));
            o[2 * k + 1] = float(__builtin_bit_cast(_Float16, uint16_t(w[k] >> 16)));
        }
    }
}

template <typename T>
__device__ __forceinline__ uint32_t pack2_io(float lo, float hi) {
    if constexpr (__is_same(T, bf16_t)) {
        return io<bf16_t>::pack2(lo, hi);
    } else {
        return uint32_t(__builtin_bit_cast(uint16_t, _Float16(lo))) |
               (uint32_t(__builtin_bit_cast(uint16_t, _Float16(hi))) << 16);
    }
}

template <typename T>
__device__ __forceinline__ uint4 pack8(const float (&v)[8]) {
    return make_uint4(pack2_io<T>(v[0], v[1]), pack2_io<T>(v[2], v[3]), pack2_io<T>(v[4], v[5]),
                      pack2_io<T>(v[6], v[7]));
}

// The RMSNorm input rows of one wave (rows w, w + NW, ... of the tile): every
// load is issued before any row is summed, at addresses clamped instead of
// branched around, so a wave waits for memory once.
template <int R>
struct NormRows {
    uint4 x[R][2], res[R][2], w[2][2];
};

template <typename T, int NW>
__device__ __forceinline__ void norm_request(const LinArgs& a, int b0, int w, int lane, NormRows<16 / NW>& r) {
    const int nvec = int(a.k_in) / 8;
    const int v0 = lane < nvec ? lane : 0, v1 = lane + 64 < nvec ? lane + 64 : 0;
#pragma unroll
    for (int i = 0; i < 16 / NW; ++i) {
        const int row = b0 + w + i * NW;
        const int64_t rc = row < a.batch ? row : 0;     // a row past the batch reads the first and is dropped
        const uint4* xr = reinterpret_cast<const uint4*>(static_cast<const T*>(a.nx) + rc * a.nx_ld);
        r.x[i][0] = xr[v0];
        r.x[i][1] = xr[v1];
        // (without a residual the input stands in for it, unused)
        const uint4* rr = a.nres ? reinterpret_cast<const uint4*>(static_cast<const T*>(a.nres) + rc * a.nres_ld) : xr;
        r.res[i][0] = rr[v0];
        r.res[i][1] = rr[v1];
    }
    // weight: one vector per 8 elements, or two in fp32
    const uint4* wp = static_cast<const uint4*>(a.nw);
    const int two = a.nw_f32 ? 1 : 0;
    r.w[0][0] = wp[v0 << two];
    r.w[0][1] = wp[(v0 << two) + two];
    r.w[1][0] = wp[v1 << two];
    r.w[1][1] = wp[(v1 << two) + two];
}

// Normalises the requested rows into xs (rows of ld elements), with the
// arithmetic of the RMSNorm forward kernel for a row of one register segment:
// lane l owns the 8-element vectors l and l + 64 of the row (k_in <= 1024),
// sums s^2 with fmas in element order and then over the wave by xor shuffles,
// and rounds s = x + residual and the output to T the same way, so the rows
// equal that kernel's output bit for bit.  With write_s, s goes to a.ns (and
// 1 / rms to a.nrstd).
template <typename T, int NW>
__device__ __forceinline__ void norm_finish(const LinArgs& a, int b0, int w, int lane, const NormRows<16 / NW>& r,
                                            uint16_t* xs, int ld, bool write_s) {
    const int nvec = int(a.k_in) / 8;
    float w1[2][8];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        float wv[8];
        if (a.nw_f32) {
            const uint32_t u[8] = {r.w[k][0].x, r.w[k][0].y, r.w[k][0].z, r.w[k][0].w,
                                   r.w[k][1].x, r.w[k][1].y, r.w[k][1].z, r.w[k][1].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) wv[e] = __uint_as_float(u[e]);
        } else {
            unpack8<T>(r.w[k][0], wv);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) w1[k][e] = 1.f + wv[e];
    }
    // all the wave's rows together, so that their sums' chains overlap (a row
    // past the batch is normalised too, and dropped)
    constexpr int R = 16 / NW;
    float sv[R][2][8], acc[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        acc[i] = 0.f;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int vi = k * 64 + lane;
            unpack8<T>(r.x[i][k], sv[i][k]);
            if (a.nres) {
                float rv[8];
                unpack8<T>(r.res[i][k], rv);
#pragma unroll
                for (int e = 0; e < 8; ++e) sv[i][k][e] = round_io<T>(sv[i][k][e] + rv[e]);
            }
            float part = acc[i];
#pragma unroll
            for (int e = 0; e < 8; ++e) part = __builtin_fmaf(sv[i][k][e], sv[i][k][e], part);
            acc[i] = vi < nvec ? part : acc[i];
        }
    }
#pragma unroll
    for (int i = 0; i < R; ++i) acc[i] = wave_allsum(acc[i]);
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int rr = w + i * NW, row = b0 + rr;
        if (row >= a.batch) break;                     // wave-uniform; no barrier inside
        const float rstd = rsqrtf(acc[i] / float(a.k_in) + a.eps);
        if (write_s && a.nrstd && lane == 0) a.nrstd[row] = rstd;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int vi = k * 64 + lane;
            if (vi < nvec) {
                float o[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = (sv[i][k][e] * rstd) * w1[k][e];
                *reinterpret_cast<uint4*>(xs + rr * ld + vi * 8) = pack8<T>(o);
                if (write_s && a.nres && a.ns)
                    *reinterpret_cast<uint4*>(static_cast<T*>(a.ns) + row * a.ns_ld + vi * 8) = pack8<T>(sv[i][k]);
            }
        }
    }
}

// kNorm: the input rows are computed in the kernel by the RMSNorm (x +
// residual) and read from LDS (extern xs, 16 rows of k_in + 8 elements: the
// padding puts the 16 rows of a 16-byte read on different banks)
// NB: K steps of a wave in flight at once.
// Code size counts here: the instruction cache is cold at every launch, and a
// wave that runs straight through a kernel once waits for most of its lines.
// Rows past n_out or the batch are therefore not masked (they read the first
// row, and only outputs that are never stored depend on them), a K step past
// the end is a branch on a scalar, and NB is no larger than the shape needs.
template <typename T, int NW, int KV, int NB, bool kNorm>
__global__ __launch_bounds__(64 * NW) void decode_linear_kernel(const LinArgs a) {
    constexpr int KS = 4 * KV;                        // k per step: 16 or 32
    __shared__ __attribute__((aligned(16))) float part[NW * 256];
    __shared__ int last;
    extern __shared__ __attribute__((aligned(16))) uint16_t xs[];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int i = lane & 15, q = lane >> 4;
    const int64_t n0 = int64_t(blockIdx.x) * 16, n = n0 + i;
    const int b0 = blockIdx.y * 16, b = b0 + i, kidx = blockIdx.z;
    const bool nv = n < a.n_out, bv = b < a.batch;
    NormRows<kNorm ? 16 / NW : 1> rows;
    if constexpr (kNorm) norm_request<T, NW>(a, b0, w, lane, rows);
    const uint16_t* wrow = static_cast<const uint16_t*>(a.weight) + (nv ? n : 0) * a.w_ld + KV * q;
    const int xld = int(a.k_in) + 8;                  // (kNorm: k_in <= 1024)
    const uint16_t* xrow = kNorm ? xs + i * xld + KV * q
                                 : static_cast<const uint16_t*>(a.x) + (bv ? b : 0) * a.x_ld + KV * q;
    // this workgroup's K steps: [kb, ke) (slices are whole steps)
    const int64_t kend = (kidx + 1) * a.kslice < a.k_in ? (kidx + 1) * a.kslice : a.k_in;
    const int kb = int(kidx * a.kslice / KS), ke = int(kend / KS);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    // NB steps of this wave are requested before any is used (steps past the
    // end read the last step again)
    rowvec<KV> av[NB], xv[NB];
    auto load_w = [&](int kt0) {
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int kt = kt0 + NW * u;
            av[u] = *reinterpret_cast<const rowvec<KV>*>(wrow + int64_t(kt < ke ? kt : ke - 1) * KS);
        }
    };
    auto load_x = [&](int kt0) {
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int kt = kt0 + NW * u;
            xv[u] = *reinterpret_cast<const rowvec<KV>*>(xrow + int64_t(kt < ke ? kt : ke - 1) * KS);
        }
    };
    // the first batch of weights (and rows) is requested before the rows are
    // normalised, so the waits for memory overlap
    load_w(kb + w);
    if constexpr (!kNorm) load_x(kb + w);
    // the output of thread t < 256 and what its epilogue reads, the conv state
    // and taps among it, requested here at clamped addresses, unconverted
    const int ol = t >> 2, ob = b0 + (ol & 15);
    const int64_t on = n0 + 4 * (ol >> 4) + (t & 3);
    const bool out_ok = t < 256 && ob < a.batch && on < a.n_out;
    const bool conv_ok = a.has_conv && out_ok && on < a.conv_dim;
    uint16_t* cst = static_cast<uint16_t*>(a.conv_state) + (conv_ok ? ob * a.cs_b + on * a.cs_d : 0);
    uint16_t craw[3] = {};
    float cw[4] = {}, cbias = 0.f;
    if (a.has_conv) {
        const float* cwp = a.conv_w + (conv_ok ? on * a.cw_d : 0);
#pragma unroll
        for (int k = 0; k < 3; ++k) craw[k] = cst[(k + 1 < a.conv_width ? k + 1 : 0) * a.cs_w];
#pragma unroll
        for (int k = 0; k < 4; ++k) cw[k] = cwp[(k < a.conv_width ? k : 0) * a.cw_w];
        if (a.conv_bias) cbias = a.conv_bias[conv_ok ? on : 0];
    }
    if constexpr (kNorm) {
        norm_finish<T, NW>(a, b0, w, lane, rows, xs, xld, blockIdx.x == 0);
        __syncthreads();
    }
    for (int kt0 = kb + w; kt0 < ke; kt0 += NW * NB) {
        if (kt0 != kb + w) load_w(kt0);
        if (kNorm || kt0 != kb + w) load_x(kt0);
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            if (kt0 + NW * u >= ke) break;            // wave-uniform
            if constexpr (KV == 8) acc = mfma32<T>(av[u], xv[u], acc);
            else acc = mfma16<T>(av[u], xv[u], acc);
        }
    }
    *reinterpret_cast<f32x4*>(part + (w * 64 + lane) * 4) = acc;
    __syncthreads();
    // thread t < 256 sums output (lane t / 4, component t % 4) over the waves
    float o = 0.f;
    if (t < 256) {
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) o += part[ww * 256 + t];
    }
    if (a.ksplit > 1) {
        // every exchange between the workgroups of a tile is an atomic
        // read-modify-write, performed where the whole device sees it, so no
        // cache write-back or invalidation is needed: the partial goes into
        // its slot by 64-bit atomic swaps (two outputs each), which complete
        // (vmcnt 0) before the counter is advanced; the workgroup that
        // advances it last takes the slots back with atomic swaps (a
        // read-modify-write, which the compiler does not turn into a plain
        // load as it does an OR of 0), in slice order
        const int tile = blockIdx.y * gridDim.x + blockIdx.x;
        unsigned long long* pt = reinterpret_cast<unsigned long long*>(a.partials + tile * a.ksplit * 256);
        if (t < 128) {
            float o0 = 0.f, o1 = 0.f;
#pragma unroll
            for (int ww = 0; ww < NW; ++ww) {
                o0 += part[ww * 256 + 2 * t];
                o1 += part[ww * 256 + 2 * t + 1];
            }
            (void)atomicExch(pt + kidx * 128 + t,
                             (static_cast<unsigned long long>(__float_as_uint(o1)) << 32) | __float_as_uint(o0));
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (t == 0) last = atomicAdd(a.counters + tile, 1) == a.ksplit - 1;
        __syncthreads();
        if (!last) return;
        if (t < 128) {
            // every slot is requested before the first is added (one wait)
            unsigned long long sv[kLinMaxSplit];
#pragma unroll
            for (int k = 0; k < kLinMaxSplit; ++k) sv[k] = k < a.ksplit ? atomicExch(pt + k * 128 + t, 0ull) : 0ull;
            float o0 = 0.f, o1 = 0.f;
#pragma unroll
            for (int k = 0; k < kLinMaxSplit; ++k) {
                o0 += __uint_as_float(uint32_t(sv[k]));
                o1 += __uint_as_float(uint32_t(sv[k] >> 32));
            }
            part[2 * t] = o0;                         // every read of part is behind the barriers above
            part[2 * t + 1] = o1;
        }
        if (t == 0) (void)atomicExch(a.counters + tile, 0);
        __syncthreads();
        if (t < 256) o = part[t];
    }
    if (!out_ok) return;
    if (a.bias) {
        o += a.bias_f32 ? static_cast<const float*>(a.bias)[on] : io<T>::load(static_cast<const T*>(a.bias) + on);
    }
    if (conv_ok) {
        // the causal conv step of channel on, fed the product as it would be
        // stored (rounded to T), in the order of the conv update kernel
        const int W = a.conv_width;
        float cacc = cbias;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (k >= W) break;
            float sk = round_io<T>(o);
            if (k < 3 && k != W - 1) {
                const uint16_t raw = craw[k < 3 ? k : 0];
                sk = io<T>::load(reinterpret_cast<const T*>(&raw));
            }
            cacc = __builtin_fmaf(cw[k], sk, cacc);
            io<T>::store(reinterpret_cast<T*>(cst) + k * a.cs_w, sk);
        }
        if (a.conv_silu) cacc *= sigmoidf_(cacc);
        o = cacc;
    }
    io<T>::store(static_cast<T*>(a.y) + ob * a.y_ld + on, o);
}

template <typename T, int KV, bool kNorm>
void launch_kvn(const LinArgs& a, hipStream_t stream) {
    const dim3 grid{unsigned((a.n_out + 15) / 16), unsigned((a.batch + 15) / 16), unsigned(a.ksplit)};
    const int64_t steps = (a.kslice + 4 * KV - 1) / (4 * KV);   // K steps per workgroup
    const size_t lds = kNorm ? size_t(16 * (a.k_in + 8) * 2) : 0;
    // (the wave count is part of the order in which a tile's steps are summed)
    const int waves = steps <= 16 ? 4 : steps <= 32 ? 8 : 16;
    const int64_t per = (steps + waves - 1) / waves;
    auto go = [&](auto NWC, auto NBC) {
        constexpr int nw = decltype(NWC)::value, nb = decltype(NBC)::value;
        hipLaunchKernelGGL((decode_linear_kernel<T, nw, KV, nb, kNorm>), grid, dim3(64 * nw), lds, stream, a);
    };
    using std::integral_constant;
    if (waves == 4 && per <= 2) go(integral_constant<int, 4>{}, integral_constant<int, 2>{});
    else if (waves == 4) go(integral_constant<int, 4>{}, integral_constant<int, 4>{});
    else if (waves == 8) go(integral_constant<int, 8>{}, integral_constant<int, 4>{});
    else go(integral_constant<int, 16>{}, integral_constant<int, 4>{});
}

template <typename T>
void launch_t(const LinArgs& a, hipStream_t stream) {
    // (with the norm the rows come from LDS, 16-byte aligned)
    const bool xok = a.nx || (a.x_ld % 8 == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15) == 0);
    const bool wide = a.k_in % 32 == 0 && xok && a.w_ld % 8 == 0 && (reinterpret_cast<uintptr_t>(a.weight) & 15) == 0;
    if (a.nx) {
        if (wide) launch_kvn<T, 8, true>(a, stream);
        else launch_kvn<T, 4, true>(a, stream);
    } else {
        if (wide) launch_kvn<T, 8, false>(a, stream);
        else launch_kvn<T, 4, false>(a, stream);
    }
}

}  // namespace

DecodeLinearSplit decode_linear_split(int64_t batch, int64_t n_out, int64_t k_in) {
    DecodeLinearSplit sp{1, k_in, 0};
    const int64_t unit = k_in % 32 == 0 ? 32 : 16;               // slices are whole K steps of either kernel
    const int64_t units = k_in / unit;
    const int64_t tiles = ((n_out + 15) / 16) * ((batch + 15) / 16);
    if (tiles <= 0 || units < 4 || tiles >= kLinSplitMaxTiles) return sp;
    const int64_t ks = kLinMaxSplit < units / 2 ? kLinMaxSplit : units / 2;   // at least 2 units per slice
    if (ks < 2) return sp;
    const int64_t per = (units + ks - 1) / ks;
    sp.ksplit = (units + per - 1) / per;
    sp.kslice = per * unit;
    if (sp.ksplit < 2) return DecodeLinearSplit{1, k_in, 0};
    sp.workspace_bytes = kLinCounterBytes + tiles * sp.ksplit * 256 * 4;
    return sp;
}

hipError_t decode_linear_launch(const ss_decode_linear_args* c, hipStream_t stream) {
    LinArgs a{};
    a.weight = c->weight; a.x = c->x; a.y = c->y; a.bias = c->bias;
    a.w_ld = c->w_row_stride; a.x_ld = c->x_row_stride; a.y_ld = c->y_row_stride;
    a.n_out = c->n_out; a.batch = int32_t(c->batch); a.k_in = c->k_in;
    a.bias_f32 = c->bias_dtype == SS_F32;
    a.ksplit = 1;
    a.kslice = a.k_in;
    const DecodeLinearSplit sp = decode_linear_split(c->batch, c->n_out, c->k_in);
    if (c->workspace && sp.ksplit > 1 && c->workspace_bytes >= sp.workspace_bytes && !c->norm) {
        a.ksplit = int32_t(sp.ksplit);
        a.kslice = sp.kslice;
        a.counters = static_cast<int*>(c->workspace);
        a.partials = reinterpret_cast<float*>(static_cast<char*>(c->workspace) + kLinCounterBytes);
    }
    if (c->conv && c->conv->dim > 0) {
        const ss_conv1d_update_args& v = *c->conv;
        a.has_conv = 1;
        a.conv_dim = v.dim; a.conv_width = int32_t(v.width); a.conv_silu = v.silu;
        a.conv_state = v.conv_state; a.conv_w = v.weight; a.conv_bias = v.has_bias ? v.bias : nullptr;
        a.cs_b = v.state_batch_stride; a.cs_d = v.state_dim_stride; a.cs_w = v.state_width_stride;
        a.cw_d = v.w_dim_stride; a.cw_w = v.w_width_stride;
    }
    if (c->norm) {
        const ss_rmsnorm_args& v = *c->norm;
        a.nx = v.x; a.nres = v.residual; a.nw = v.weight; a.ns = v.residual_out; a.nrstd = v.rstd;
        a.nx_ld = v.x_row_stride; a.nres_ld = v.residual_row_stride; a.ns_ld = v.residual_out_row_stride;
        a.eps = v.eps;
        a.nw_f32 = v.w_dtype == SS_F32;
    }
    if (c->dtype == SS_BF16) launch_t<bf16_t>(a, stream);
    else launch_t<_Float16>(a, stream);
    return hipGetLastError();
}

}  // namespace ss
