// polar_norm.hip — per-matrix normalisation X / (‖X‖_F·1.01 + 1e-6) ahead of the
// Polar Express iteration, with the rounding points of the reference recipe
// (examples/five_steps.py:18, tests/test_polar_step.py:39), evaluated there as
// bf16 torch ops:
//
//     norm = bf16(sqrt(Σ x²))            (fp32 sum of squares)
//     d    = bf16(bf16(norm · 1.01f) + 1e-6f)
//     y    = bf16(x / d)                 (fp32 division)
//
// Two bandwidth-bound passes: per-chunk fp32 partial sums of squares, then a
// scale pass in which every block re-sums its matrix's partials in the same
// fixed order (so all blocks of a matrix agree, and results are run-to-run
// identical).
//
// Also the two element-wise passes of the Muon update around the iteration:
// the momentum pass (fp32 momentum buffer and Nesterov blend, the bf16 input of
// the iteration and its sums of squares in the normalisation's own order) and
// the parameter update p = p·(1 − lr·wd) − lr·scale·O.
//
// And the row-padding copy that gives the DMA-fed stage kernels rows of a whole
// number of 64-element K-steps: X [rows, n] -> Xp [rows, np], np a multiple of 8
// (of 64 as used), the columns n .. np-1 zero, one 16-byte chunk of Xp per thread.
#include "polar_kernels.h"
#include "polar_norm.hpp"
#include "polar_tile.hpp"

namespace muon_polar {

namespace {

constexpr int kNormThreads = 256;
constexpr int kNormStride = kNormThreads * 8;  // elements a block covers per iteration

// Iterations whose loads each thread issues before it uses the first of them (the
// vector loops below).  Every thread still takes its elements in increasing order,
// so the sums are those of one iteration at a time; what changes is the number of
// loads in flight per wave, which sets these bandwidth-bound passes' rate.
constexpr int kNormUnroll = 4;      // norm passes: 16 bytes per thread and iteration
constexpr int kMomentumUnroll = 2;  // momentum pass: 64 bytes per thread and iteration
constexpr int kParamUnroll = 2;     // parameter pass: 48 bytes per thread and iteration

// Element-wise loops (matrices of m·n % 8 != 0, whose sums run one element per thread
// and step): loads issued ahead per thread, again in increasing order.  One at a time
// each wave waited out every round trip: the Muon update of [20,127,2051] took 193 us,
// that of [1,2047,4097] 574, the chain of [1,333,9999] 197; with these and the 16-byte
// accesses below 180, 551 and 193.  (The padding copy keeps its 2-byte loads of odd rows:
// unaligned 16-byte ones took it from 9.5 to 14.4 us at [1,333,9999].)
constexpr int kElemUnroll = 8;

// 16 bytes at any element's address: global memory takes unaligned vector accesses, at
// the cost of a second line where one straddles it.
template <typename V, typename T>
__device__ __forceinline__ V load16_any(const T *p) {
    V v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
template <typename V, typename T>
__device__ __forceinline__ void store16_any(T *p, V v) {
    __builtin_memcpy(p, &v, 16);
}

// Sum of v over the block in a fixed order: butterfly within each wave, then the
// four wave totals in index order.  `red` holds 4 floats of LDS.
__device__ __forceinline__ float block_sum(float v, float *red) {
    v = wave_sum(v);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) red[wave] = v;
    __syncthreads();
    const float t = ((red[0] + red[1]) + red[2]) + red[3];
    __syncthreads();
    return t;
}

// Sum of squares of chunk c of matrix b into partial[b * chunks + c].
__global__ __launch_bounds__(kNormThreads) void norm_partial_kernel(const uint16_t *__restrict__ x,
                                                                    float *__restrict__ partial,
                                                                    int64_t mn, int chunks,
                                                                    int64_t chunk, int vec) {
    __shared__ float red[4];
    const int b = blockIdx.x / chunks, c = blockIdx.x - b * chunks;
    const uint16_t *base = x + int64_t(b) * mn;
    const int64_t e0 = int64_t(c) * chunk;
    const int64_t e1 = e0 + chunk < mn ? e0 + chunk : mn;
    float acc = 0.0f;
    if (vec) {  // mn % 8 == 0 and 16-byte aligned rows of 8 elements
        for (int64_t e = e0 + threadIdx.x * 8; e < e1; e += kNormUnroll * kNormStride) {
            u32x4 v[kNormUnroll];
#pragma unroll
            for (int u = 0; u < kNormUnroll; ++u)
                if (e + u * kNormStride < e1)
                    v[u] = *reinterpret_cast<const u32x4 *>(base + e + u * kNormStride);
#pragma unroll
            for (int u = 0; u < kNormUnroll; ++u) {
                if (e + u * kNormStride >= e1) break;
#pragma unroll
                for (int w = 0; w < 4; ++w) acc = add_squares(acc, v[u][w]);
            }
        }
    } else {
        for (int64_t e = e0 + threadIdx.x; e < e1; e += kElemUnroll * kNormThreads) {
            uint32_t v[kElemUnroll];
#pragma unroll
            for (int u = 0; u < kElemUnroll; ++u)
                if (e + u * kNormThreads < e1) v[u] = base[e + u * kNormThreads];
#pragma unroll
            for (int u = 0; u < kElemUnroll; ++u) {
                if (e + u * kNormThreads >= e1) break;
                const float f = bf16_bits_to_f32(v[u]);
                acc = fmaf(f, f, acc);
            }
        }
    }
    const float t = block_sum(acc, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// y = bf16(x / d) over chunk c of matrix b, d from the matrix's partial sums.
__global__ __launch_bounds__(kNormThreads) void norm_scale_kernel(const uint16_t *__restrict__ x,
                                                                  uint16_t *__restrict__ y,
                                                                  const float *__restrict__ partial,
                                                                  int64_t mn, int chunks,
                                                                  int64_t chunk, int vec) {
    __shared__ float red[4];
    const int b = blockIdx.x / chunks, c = blockIdx.x - b * chunks;
    float s = 0.0f;
    for (int i = threadIdx.x; i < chunks; i += kNormThreads) s += partial[int64_t(b) * chunks + i];
    const float d = norm_divisor(block_sum(s, red));

    const uint16_t *xb = x + int64_t(b) * mn;
    uint16_t *yb = y + int64_t(b) * mn;
    const int64_t e0 = int64_t(c) * chunk;
    const int64_t e1 = e0 + chunk < mn ? e0 + chunk : mn;
    if (vec) {
        const __amdgpu_buffer_rsrc_t rs_y = store_rsrc(yb + e0);
        for (int64_t e = e0 + threadIdx.x * 8; e < e1; e += kNormUnroll * kNormStride) {
            u32x4 v[kNormUnroll];
#pragma unroll
            for (int u = 0; u < kNormUnroll; ++u)
                if (e + u * kNormStride < e1)
                    v[u] = *reinterpret_cast<const u32x4 *>(xb + e + u * kNormStride);
#pragma unroll
            for (int u = 0; u < kNormUnroll; ++u) {
                if (e + u * kNormStride >= e1) break;
                u32x4 o;
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t lo = f32_to_bf16_bits(bf16_bits_to_f32(v[u][w] & 0xffffu) / d);
                    const uint32_t hi = f32_to_bf16_bits(bf16_bits_to_f32(v[u][w] >> 16) / d);
                    o[w] = lo | (hi << 16);
                }
                store16_sc1(rs_y, static_cast<uint32_t>((e + u * kNormStride - e0) * 2), o);
            }
        }
    } else {
        for (int64_t e = e0 + threadIdx.x * 8; e < e1; e += kNormStride) {
            if (e + 8 <= e1) {
                const u32x4 v = load16_any<u32x4>(xb + e);
                u32x4 o;
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t lo = f32_to_bf16_bits(bf16_bits_to_f32(v[w] & 0xffffu) / d);
                    const uint32_t hi = f32_to_bf16_bits(bf16_bits_to_f32(v[w] >> 16) / d);
                    o[w] = lo | (hi << 16);
                }
                store16_any(yb + e, o);
            } else {
                for (int64_t i = e; i < e1; ++i)
                    yb[i] = f32_to_bf16_bits(bf16_bits_to_f32(xb[i]) / d);
            }
        }
    }
}

// torch.lerp's two-branch form (ATen Lerp.h): start + w·(end − start) for |w| < 0.5,
// else end − (end − start)·(1 − w); every operation rounded on its own.
__device__ __forceinline__ float lerp_rounded(float start, float end, float w) {
#pragma clang fp contract(off)
    return fabsf(w) < 0.5f ? start + w * (end - start) : end - (end - start) * (1.0f - w);
}

// Where matrix b of the Muon update's fp32 tensors (and of its gradient, G = float or
// the bits of a bf16) lies: rows of one batched tensor, or tensors of their own, whose
// pointers travel in the kernel arguments (no table in memory to fill and to wait for):
// one matrix in each (the common case: 8 x [768,768] 13.0 us a launch, 13.6 with a branch
// around the division), or `per` of them.  One pointer per matrix took a launch for every 128 of them: the update
// of 4 x [4096,32,32] 1073 us, now 671.
template <typename G>
struct BatchedMats {
    const G *g;
    float *w;
    int64_t mn;
    __device__ __forceinline__ const G *grad(int b) const { return g + int64_t(b) * mn; }
    __device__ __forceinline__ float *buf(int b) const { return w + int64_t(b) * mn; }
};
template <typename G>
struct ListedMats {
    const G *g[kMuonListMax];
    float *w[kMuonListMax];
    __device__ __forceinline__ const G *grad(int b) const { return g[b]; }
    __device__ __forceinline__ float *buf(int b) const { return w[b]; }
};
template <typename G>
struct ListedTensors {
    ListedMats<G> t;
    int64_t mn;
    int32_t per;
    __device__ __forceinline__ const G *grad(int b) const {
        return t.g[b / per] + int64_t(b % per) * mn;
    }
    __device__ __forceinline__ float *buf(int b) const {
        return t.w[b / per] + int64_t(b % per) * mn;
    }
};
struct BatchedParam {
    float *p;
    __device__ __forceinline__ float *at(int) const { return p; }
};
struct ListedParams {
    float *p[kMuonListMax];
    __device__ __forceinline__ float *at(int b) const { return p[b]; }
};

// 8 consecutive gradient values as fp32 (exact for bf16); kVec: 16-byte aligned.
template <bool kVec>
__device__ __forceinline__ void load8(const float *g, float (&v)[8]) {
    if (kVec) {
        const f32x4 lo = *reinterpret_cast<const f32x4 *>(g);
        const f32x4 hi = *reinterpret_cast<const f32x4 *>(g + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = lo[i];
            v[i + 4] = hi[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = g[i];
    }
}
template <bool kVec>
__device__ __forceinline__ void load8(const uint16_t *g, float (&v)[8]) {
    if (kVec) {
        const u32x4 w = *reinterpret_cast<const u32x4 *>(g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = bf16_bits_to_f32(w[i] & 0xffffu);
            v[2 * i + 1] = bf16_bits_to_f32(w[i] >> 16);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = bf16_bits_to_f32(g[i]);
    }
}
__device__ __forceinline__ float grad_value(float g) { return g; }
__device__ __forceinline__ float grad_value(uint16_t g) { return bf16_bits_to_f32(g); }

// Momentum pass of the Muon update over chunk c of matrix b (chunks as in
// norm_partial_kernel):
//     buf ← lerp(buf, g, w)                  (w = 1 − momentum)
//     g'  = lerp(g, buf, momentum) | buf     (Nesterov or plain)
//     x0  = bf16(g'),   partial[b, c] = Σ x0²  in norm_partial_kernel's order
// kOrder8: mn % 8 == 0 (8 consecutive elements per thread and step, the vector
// path's order); kVec: also 16-byte aligned g, buf and x0 (vector accesses).
//
// Bound by HBM: 12 bytes per element of an fp32 gradient, 10 of a bf16 one, and the
// 2 of x0.  Separate tensors are read and written where they lie: gathering them into
// one batch and copying the results back moved 40 bytes per element more (with the
// parameter pass's) in two launches per tensor: an optimizer step over [768,768] x 8,
// [3072,768] x 2 and [768,3072] x 2 took 841 us with it and takes 655; the update of one
// [1024,4096] with a bf16 gradient 218 us with an fp32 copy of it, 206 without.
template <bool kOrder8, bool kVec, typename G, typename Mats>
__global__ __launch_bounds__(kNormThreads) void muon_momentum_kernel(
    const Mats mats, uint16_t *__restrict__ x0, float *__restrict__ partial, int64_t mn,
    int chunks, int64_t chunk, float w, float beta, int nesterov) {
#pragma clang fp contract(off)
    __shared__ float red[4];
    const int b = blockIdx.x / chunks, c = blockIdx.x - b * chunks;
    const int64_t base = int64_t(b) * mn;
    const G *__restrict__ gb = mats.grad(b);
    float *__restrict__ bufb = mats.buf(b);
    const int64_t e0 = int64_t(c) * chunk;
    const int64_t e1 = e0 + chunk < mn ? e0 + chunk : mn;
    float acc = 0.0f;
    auto one = [&](float gv, float bv, uint32_t &h) {
        const float nb = lerp_rounded(bv, gv, w);
        const float u = nesterov ? lerp_rounded(gv, nb, beta) : nb;
        h = f32_to_bf16_bits(u);
        const float r = bf16_bits_to_f32(h);
        acc = fmaf(r, r, acc);
        return nb;
    };
    if (kOrder8) {
        constexpr int kU = kVec ? kMomentumUnroll : 1;
        const __amdgpu_buffer_rsrc_t rs_x0 = store_rsrc(x0 + base + e0);
        for (int64_t e = e0 + threadIdx.x * 8; e < e1; e += kU * kNormStride) {
            float gv[kU][8], bv[kU][8];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int64_t eu = e + u * kNormStride;
                if (eu >= e1) break;
                load8<kVec>(gb + eu, gv[u]);
                load8<kVec>(static_cast<const float *>(bufb + eu), bv[u]);
            }
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int64_t eu = e + u * kNormStride;
                if (eu >= e1) break;
                float nb[8];
                uint32_t h[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) nb[i] = one(gv[u][i], bv[u][i], h[i]);
                if (kVec) {
                    *reinterpret_cast<f32x4 *>(bufb + eu) = f32x4{nb[0], nb[1], nb[2], nb[3]};
                    *reinterpret_cast<f32x4 *>(bufb + eu + 4) =
                        f32x4{nb[4], nb[5], nb[6], nb[7]};
                    store16_sc1(rs_x0, static_cast<uint32_t>((eu - e0) * 2),
                                u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16),
                                      h[4] | (h[5] << 16), h[6] | (h[7] << 16)});
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        bufb[eu + i] = nb[i];
                        x0[base + eu + i] = static_cast<uint16_t>(h[i]);
                    }
                }
            }
        }
    } else {
        for (int64_t e = e0 + threadIdx.x; e < e1; e += kElemUnroll * kNormThreads) {
            float gv[kElemUnroll], bv[kElemUnroll];
#pragma unroll
            for (int u = 0; u < kElemUnroll; ++u) {
                const int64_t eu = e + u * kNormThreads;
                if (eu >= e1) break;
                gv[u] = grad_value(gb[eu]);
                bv[u] = bufb[eu];
            }
#pragma unroll
            for (int u = 0; u < kElemUnroll; ++u) {
                const int64_t eu = e + u * kNormThreads;
                if (eu >= e1) break;
                uint32_t h;
                bufb[eu] = one(gv[u], bv[u], h);
                x0[base + eu] = static_cast<uint16_t>(h);
            }
        }
    }
    const float t = block_sum(acc, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// p ← p·decay + alpha·O over `total` elements of tensor blockIdx.y (fp32 p, bf16 O;
// each product and the sum rounded on their own).
template <bool kVec, typename Params>
__global__ __launch_bounds__(kNormThreads) void muon_param_update_kernel(
    const Params params, const uint16_t *__restrict__ o_all, int64_t total, float decay,
    float alpha) {
#pragma clang fp contract(off)
    float *__restrict__ p = params.at(blockIdx.y);
    const uint16_t *__restrict__ o = o_all + int64_t(blockIdx.y) * total;
    const int64_t stride = int64_t(gridDim.x) * kNormThreads * 8;
    if (kVec) {
        // kParamUnroll grid strides per trip, every load of the trip issued first
        for (int64_t e = (int64_t(blockIdx.x) * kNormThreads + threadIdx.x) * 8; e < total;
             e += kParamUnroll * stride) {
            u32x4 ov[kParamUnroll];
            f32x4 p0[kParamUnroll], p1[kParamUnroll];
#pragma unroll
            for (int u = 0; u < kParamUnroll; ++u) {
                const int64_t eu = e + u * stride;
                if (eu >= total) break;
                ov[u] = *reinterpret_cast<const u32x4 *>(o + eu);
                p0[u] = *reinterpret_cast<const f32x4 *>(p + eu);
                p1[u] = *reinterpret_cast<const f32x4 *>(p + eu + 4);
            }
#pragma unroll
            for (int u = 0; u < kParamUnroll; ++u) {
                const int64_t eu = e + u * stride;
                if (eu >= total) break;
                f32x4 q0 = p0[u], q1 = p1[u];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    q0[2 * i] = q0[2 * i] * decay + alpha * bf16_bits_to_f32(ov[u][i] & 0xffffu);
                    q0[2 * i + 1] = q0[2 * i + 1] * decay + alpha * bf16_bits_to_f32(ov[u][i] >> 16);
                    q1[2 * i] = q1[2 * i] * decay + alpha * bf16_bits_to_f32(ov[u][i + 2] & 0xffffu);
                    q1[2 * i + 1] =
                        q1[2 * i + 1] * decay + alpha * bf16_bits_to_f32(ov[u][i + 2] >> 16);
                }
                *reinterpret_cast<f32x4 *>(p + eu) = q0;
                *reinterpret_cast<f32x4 *>(p + eu + 4) = q1;
            }
        }
    } else {
        for (int64_t e = (int64_t(blockIdx.x) * kNormThreads + threadIdx.x) * 8; e < total;
             e += stride) {
            if (e + 8 <= total) {
                const u32x4 ov = load16_any<u32x4>(o + e);
                f32x4 q0 = load16_any<f32x4>(p + e), q1 = load16_any<f32x4>(p + e + 4);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    q0[2 * i] = q0[2 * i] * decay + alpha * bf16_bits_to_f32(ov[i] & 0xffffu);
                    q0[2 * i + 1] = q0[2 * i + 1] * decay + alpha * bf16_bits_to_f32(ov[i] >> 16);
                    q1[2 * i] = q1[2 * i] * decay + alpha * bf16_bits_to_f32(ov[i + 2] & 0xffffu);
                    q1[2 * i + 1] =
                        q1[2 * i + 1] * decay + alpha * bf16_bits_to_f32(ov[i + 2] >> 16);
                }
                store16_any(p + e, q0);
                store16_any(p + e + 4, q1);
            } else {
                for (int64_t i = e; i < total; ++i)
                    p[i] = p[i] * decay + alpha * bf16_bits_to_f32(o[i]);
            }
        }
    }
}

__global__ __launch_bounds__(kNormThreads) void pad_rows_kernel(const uint16_t *__restrict__ x,
                                                                uint16_t *__restrict__ xp,
                                                                int64_t chunks, int32_t n,
                                                                int32_t row_chunks, int32_t vec) {
    // row_chunks = np / 8: chunks per padded row; vec: 16-byte loads of whole
    // chunks (n % 8 == 0 and x 16-byte aligned)
    const int64_t stride = int64_t(gridDim.x) * kNormThreads;
    for (int64_t q0 = int64_t(blockIdx.x) * kNormThreads; q0 < chunks; q0 += stride) {
        const int64_t q = q0 + threadIdx.x;
        if (q >= chunks) break;
        const __amdgpu_buffer_rsrc_t rs = store_rsrc(xp + q0 * 8);  // this block's chunks
        const int64_t r = q / row_chunks;
        const int c0 = static_cast<int>(q - r * row_chunks) * 8;
        const uint16_t *src = x + r * n + c0;
        u32x4 v;
        if (vec && c0 + 8 <= n) {
            v = *reinterpret_cast<const u32x4 *>(src);
        } else {
            uint32_t h[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) h[e] = c0 + e < n ? uint32_t(src[e]) : 0u;
            v = u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                      h[6] | (h[7] << 16)};
        }
        store16_sc1(rs, static_cast<uint32_t>(threadIdx.x) * 16u, v);
    }
}

}  // namespace

hipError_t launch_pad_rows(const uint16_t *x, uint16_t *xp, int64_t rows, int64_t n, int64_t np,
                           hipStream_t stream) {
    if (rows <= 0 || n <= 0 || np < n || np % 8 != 0 || np >= (int64_t(1) << 30))
        return hipErrorInvalidValue;
    int32_t row_chunks = static_cast<int32_t>(np / 8), nn = static_cast<int32_t>(n);
    int64_t chunks = rows * row_chunks;
    int32_t vec = (n % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0) ? 1 : 0;
    const int64_t blocks = (chunks + kNormThreads - 1) / kNormThreads;
    const unsigned grid = static_cast<unsigned>(blocks < 8192 ? blocks : 8192);
    void *args[] = {&x, &xp, &chunks, &nn, &row_chunks, &vec};
    return hipLaunchKernel(reinterpret_cast<const void *>(&pad_rows_kernel), dim3(grid),
                           dim3(kNormThreads), args, 0, stream);
}

// Smaller chunks give more blocks to the passes of a small matrix; every block of
// the scale pass re-sums all of its matrix's partials, so the chunk is the smallest
// power of two from 4096 for which batch · chunks² stays within 2^24 partial loads.
// Measured (the Muon update's element-wise passes / the normalisation):
// [1,4096,14336] 330 / 61 us with 65536-element chunks, 314 / 60 with 16384, 319 / 74
// with 8192; [12,768,768] 53 / 19 us with 65536, 35 / 10 with 4096.
int64_t norm_chunk(int64_t batch, int64_t mn) {
    constexpr int64_t kMin = 4096, kMax = int64_t(1) << 20, kBudget = int64_t(1) << 24;
    int64_t chunk = kMin;
    while (chunk < kMax) {
        const int64_t c = (mn + chunk - 1) / chunk;
        if (c <= kBudget / c / (batch > 0 ? batch : 1)) break;
        chunk *= 2;
    }
    return chunk;
}

int64_t norm_chunks(int64_t batch, int64_t mn) {
    const int64_t chunk = norm_chunk(batch, mn);
    return (mn + chunk - 1) / chunk;
}

hipError_t launch_norm_scale(const uint16_t *x, uint16_t *y, const float *partial,
                             int64_t batch, int64_t mn, bool vec, hipStream_t stream) {
    int64_t chunk = norm_chunk(batch, mn);
    const int64_t chunks = norm_chunks(batch, mn);
    const int64_t grid = batch * chunks;
    if (grid <= 0 || grid >= (int64_t(1) << 31)) return hipErrorInvalidValue;
    int ch = static_cast<int>(chunks), v = vec ? 1 : 0;
    void *a2[] = {&x, &y, &partial, &mn, &ch, &chunk, &v};
    return hipLaunchKernel(reinterpret_cast<const void *>(&norm_scale_kernel),
                           dim3(static_cast<unsigned>(grid)), dim3(kNormThreads), a2, 0, stream);
}

namespace {

template <typename G, typename Mats>
hipError_t launch_momentum_pass(const Mats &mats, uint16_t *x0, float *partial, int64_t matrices,
                                int64_t mn, int64_t chunk, float w, float beta, bool nesterov,
                                bool vec, hipStream_t stream) {
    const int64_t chunks = (mn + chunk - 1) / chunk;
    const int64_t grid = matrices * chunks;
    if (grid <= 0 || grid >= (int64_t(1) << 31)) return hipErrorInvalidValue;
    const void *fn =
        mn % 8 != 0 ? reinterpret_cast<const void *>(&muon_momentum_kernel<false, false, G, Mats>)
        : vec       ? reinterpret_cast<const void *>(&muon_momentum_kernel<true, true, G, Mats>)
                    : reinterpret_cast<const void *>(&muon_momentum_kernel<true, false, G, Mats>);
    int ch = static_cast<int>(chunks), nv = nesterov ? 1 : 0;
    void *args[] = {const_cast<Mats *>(&mats), &x0, &partial, &mn, &ch, &chunk, &w, &beta, &nv};
    return hipLaunchKernel(fn, dim3(static_cast<unsigned>(grid)), dim3(kNormThreads), args, 0,
                           stream);
}

template <typename G>
hipError_t momentum_of(const MuonTensors &t, uint16_t *x0, float *partial, int64_t mn, float w,
                       float beta, bool nesterov, bool vec, hipStream_t stream) {
    const int64_t chunk = norm_chunk(t.count * t.matrices, mn);
    if (t.count == 1) {
        const BatchedMats<G> mats{static_cast<const G *>(t.grad[0]), static_cast<float *>(t.buf[0]),
                                  mn};
        return launch_momentum_pass<G>(mats, x0, partial, t.matrices, mn, chunk, w, beta, nesterov,
                                       vec, stream);
    }
    for (int64_t i0 = 0; i0 < t.count; i0 += kMuonListMax) {
        const int64_t cnt = t.count - i0 < kMuonListMax ? t.count - i0 : kMuonListMax;
        ListedTensors<G> mats{{}, mn, static_cast<int32_t>(t.matrices)};
        for (int64_t i = 0; i < cnt; ++i) {
            mats.t.g[i] = static_cast<const G *>(t.grad[i0 + i]);
            mats.t.w[i] = static_cast<float *>(t.buf[i0 + i]);
        }
        const int64_t m0 = i0 * t.matrices;
        uint16_t *xi = x0 + m0 * mn;
        float *pi = partial + m0 * ((mn + chunk - 1) / chunk);
        const hipError_t e =
            t.matrices == 1
                ? launch_momentum_pass<G>(mats.t, xi, pi, cnt, mn, chunk, w, beta, nesterov, vec,
                                          stream)
                : launch_momentum_pass<G>(mats, xi, pi, cnt * t.matrices, mn, chunk, w, beta,
                                          nesterov, vec, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <typename Params>
hipError_t launch_param_pass(const Params &params, const uint16_t *o, int64_t tensors,
                             int64_t total, float decay, float alpha, bool vec,
                             hipStream_t stream) {
    // 8 elements per thread; at most 8 waves' worth of blocks per CU on 256 CUs,
    // a grid-stride loop beyond that
    const int64_t blocks = (total + kNormThreads * 8 - 1) / (kNormThreads * 8);
    const int64_t most = (4096 + tensors - 1) / tensors;
    void *args[] = {const_cast<Params *>(&params), &o, &total, &decay, &alpha};
    const void *fn = vec ? reinterpret_cast<const void *>(&muon_param_update_kernel<true, Params>)
                         : reinterpret_cast<const void *>(&muon_param_update_kernel<false, Params>);
    return hipLaunchKernel(
        fn, dim3(static_cast<unsigned>(blocks < most ? blocks : most), static_cast<unsigned>(tensors)),
        dim3(kNormThreads), args, 0, stream);
}

}  // namespace

hipError_t launch_muon_momentum(const MuonTensors &t, uint16_t *x0, float *partial, int64_t mn,
                                float w, float beta, bool nesterov, bool vec,
                                hipStream_t stream) {
    return t.grad_bf16
               ? momentum_of<uint16_t>(t, x0, partial, mn, w, beta, nesterov, vec, stream)
               : momentum_of<float>(t, x0, partial, mn, w, beta, nesterov, vec, stream);
}

hipError_t launch_muon_param_update(const MuonTensors &t, const uint16_t *o, int64_t mn,
                                    float decay, float alpha, bool vec, hipStream_t stream) {
    const int64_t per_tensor = t.matrices * mn;
    if (t.count <= 0 || per_tensor <= 0) return hipErrorInvalidValue;
    if (t.count == 1)
        return launch_param_pass(BatchedParam{static_cast<float *>(t.param[0])}, o, 1, per_tensor,
                                 decay, alpha, vec, stream);
    for (int64_t i0 = 0; i0 < t.count; i0 += kMuonListMax) {
        const int64_t cnt = t.count - i0 < kMuonListMax ? t.count - i0 : kMuonListMax;
        ListedParams params{};
        for (int64_t i = 0; i < cnt; ++i) params.p[i] = static_cast<float *>(t.param[i0 + i]);
        hipError_t e = launch_param_pass(params, o + i0 * per_tensor, cnt, per_tensor, decay, alpha,
                                         vec, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_normalize(const uint16_t *x, uint16_t *y, float *partial, int64_t batch,
                            int64_t mn, bool vec, hipStream_t stream) {
    int64_t chunk = norm_chunk(batch, mn);
    const int64_t chunks = norm_chunks(batch, mn);
    const int64_t grid = batch * chunks;
    if (grid <= 0 || grid >= (int64_t(1) << 31)) return hipErrorInvalidValue;
    int ch = static_cast<int>(chunks), v = vec ? 1 : 0;
    void *a1[] = {&x, &partial, &mn, &ch, &chunk, &v};
    hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(&norm_partial_kernel),
                                   dim3(static_cast<unsigned>(grid)), dim3(kNormThreads), a1, 0,
                                   stream);
    if (e != hipSuccess) return e;
    void *a2[] = {&x, &y, &partial, &mn, &ch, &chunk, &v};
    return hipLaunchKernel(reinterpret_cast<const void *>(&norm_scale_kernel),
                           dim3(static_cast<unsigned>(grid)), dim3(kNormThreads), a2, 0, stream);
}

}  // namespace muon_polar
