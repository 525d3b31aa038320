// polar_resident.hip — whole steps of a small matrix in one workgroup.
//
// A matrix whose iterate and A (then P) fit one CU's LDS runs its normalisation and all
// its steps in one launch: X is read once, kept in LDS as the wide form [s][l] (s the
// shorter side; a tall matrix is transposed on the way in and out), and Y written once.
// What bounds such calls through the stage kernels is not their work but three launches
// per step of 5 to 6 us each, most of it start, first load and drain.
//
// Sums run in the stage kernels' unsplit order (k ascending, one chain per output, a·X
// added before the 64-element K-step that holds the output's rows), so the results are
// theirs bit for bit (but for shorter sides of 32, 96 or 160, which have no padded rows here:
// infinities in X or A stay infinite where the stages' 64-row tiles make NaN of 0 * inf); so
// is the normalisation's sum of squares.  Y may be X: a workgroup
// has all of its matrix in LDS before it writes any of it.
//
// 16 waves.  Gram and poly: one 32x32 block of the upper triangle per wave at a time
// (2x2 16x16x32 MFMAs).  Apply: wave w computes all its column blocks of row block
// w % NB together, so that each P fragment is read once and the blocks' MFMAs are
// independent; they stay in registers until every wave has read X.
// LDS rows are padded by 16 bytes: 16 rows at one 16-byte chunk then lie in 16 different
// places of the 256-byte bank window.
#include "polar_kernels.h"
#include "polar_norm.hpp"
#include "polar_schedule.hpp"
#include "polar_tile.hpp"

namespace muon_polar {

namespace {

constexpr int kWaves = 16, kThreads = 64 * kWaves;
constexpr int kRowPad = 8;         // elements
constexpr int kColBlocks = 4;  // 32-column blocks of Y per wave, at most (resident_fits)
constexpr int kMaxChunks = 64;     // partial sums of the normalisation
constexpr int kTailBytes = 4 * (kMaxChunks + kWaves);
constexpr int kLdsBytes = 160 * 1024;

using lds_bf16x4 = __attribute__((address_space(3))) bf16x4;

// v's words rotated left by k (0 to 3).
__device__ __forceinline__ u32x4 rotate_words(u32x4 v, int k) {
    if (k & 1) v = u32x4{v[1], v[2], v[3], v[0]};
    if (k & 2) v = u32x4{v[2], v[3], v[0], v[1]};
    return v;
}

// NB: 32-row blocks of the shorter side.  All of the LDS, as one workgroup per CU runs
// whatever it takes: 16 waves of over 64 registers (117 to 128) leave no room for another.
template <int NB>
__global__ __launch_bounds__(kThreads) void resident_kernel(ResidentArgs g) {
    __shared__ __attribute__((aligned(1024))) uint8_t smem[kLdsBytes];
    constexpr int kSp = 32 * NB;
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63, l15 = lane & 15, lq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = g.n, mn = g.m * g.n;
    const int s = g.tall ? g.n : g.m, l = g.tall ? g.m : g.n;
    const int lblocks = (l + 31) >> 5;
    const int xs = 32 * lblocks + kRowPad, as = kSp + kRowPad;  // row strides in elements
    uint16_t *X = reinterpret_cast<uint16_t *>(smem);
    uint16_t *A = X + kSp * xs;
    float *partial = reinterpret_cast<float *>(smem + kLdsBytes - kTailBytes);
    float *red = partial + kMaxChunks;
    const uint16_t *x = g.x + int64_t(blockIdx.x) * mn;
    uint16_t *y = g.y + int64_t(blockIdx.x) * mn;

    // Elements of the matrix in memory order: 16-byte accesses between the first and the
    // last 16-byte boundary.  Element e = r * n + c sits in LDS at place(r, c); the next
    // one is `in` further, or `wrap` at a row's end.  r by a float reciprocal: e + 0.5 is
    // at least 0.5 / n away from a multiple of n, far more than its error for e < 2^17.
    const float inv_n = 1.0f / static_cast<float>(n);
    auto row_of = [&](int e) { return static_cast<int>((static_cast<float>(e) + 0.5f) * inv_n); };
    auto place = [&](int r, int c) { return g.tall ? c * xs + r : r * xs + c; };
    const int in = g.tall ? xs : 1, wrap = g.tall ? 1 - (n - 1) * xs : xs - (n - 1);
    auto head_of = [&](const uint16_t *p) {
        const int h = static_cast<int>((0u - static_cast<uint32_t>(
                                                  reinterpret_cast<uintptr_t>(p))) & 15u) / 2;
        return h < mn ? h : mn;
    };

    // ------------------------------------------------------------ normalisation
    // Chunks of 4096 elements, one per group of four waves at a time, each thread and sum
    // in norm_partial_kernel's order.
    float d = 1.0f;
    if (g.normalize) {
        const int grp = wave >> 2, t = tid & 255;
        for (int c0 = 0; c0 < g.chunks; c0 += kWaves / 4) {
            const int c = c0 + grp, e0 = c * 4096, e1 = e0 + 4096 < mn ? e0 + 4096 : mn;
            float acc = 0.0f;
            if (c < g.chunks) {
                if (g.vec) {
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const int e = e0 + 8 * t + 2048 * u;
                        if (e < e1) {
                            const u32x4 v = *reinterpret_cast<const u32x4 *>(x + e);
#pragma unroll
                            for (int w = 0; w < 4; ++w) acc = add_squares(acc, v[w]);
                        }
                    }
                } else {
                    uint16_t h[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u)
                        h[u] = e0 + t + 256 * u < e1 ? x[e0 + t + 256 * u] : 0;
#pragma unroll
                    for (int u = 0; u < 16; ++u) {
                        if (e0 + t + 256 * u >= e1) break;
                        const float f = bf16_bits_to_f32(h[u]);
                        acc = fmaf(f, f, acc);
                    }
                }
            }
            acc = wave_sum(acc);
            if (lane == 0) red[wave] = acc;
            __syncthreads();
            if (t == 0 && c < g.chunks)
                partial[c] = ((red[4 * grp] + red[4 * grp + 1]) + red[4 * grp + 2]) + red[4 * grp + 3];
            __syncthreads();
        }
        // as norm_scale_kernel: one partial per thread, the second to fourth waves add zero
        d = norm_divisor(wave_sum(lane < g.chunks ? partial[lane] : 0.0f));
    }
    auto scaled = [&](uint32_t h) -> uint32_t {
        return g.normalize ? f32_to_bf16_bits(bf16_bits_to_f32(h) / d) : h;
    };

    // ------------------------------------------------------------ X into LDS
    {
        constexpr int kBatch = 4;  // vectors in flight per thread
        const int head = head_of(x), nvec = (mn - head) / 8;
        const bool whole = n % 8 == 0 && head == 0;  // vectors stay inside a row
        const bool rows8 = whole && !g.tall, cols8 = whole && g.tall;
        u32x4 v[kBatch];
        auto fetch = [&](int i0) {
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const int i = i0 + u * kThreads;
                if (i < nvec) v[u] = *reinterpret_cast<const u32x4 *>(x + head + 8 * i);
            }
        };
        fetch(tid);
        for (int i = tid; i < kSp * xs / 8; i += kThreads)
            *reinterpret_cast<u32x4 *>(X + 8 * i) = u32x4{0u, 0u, 0u, 0u};
        __syncthreads();
        for (int i0 = tid; i0 < nvec; i0 += kBatch * kThreads) {
            if (i0 != tid) fetch(i0);
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const int i = i0 + u * kThreads;
                if (i >= nvec) break;
                const int e0 = head + 8 * i, r = row_of(e0);
                int c = e0 - r * n;
                uint16_t *dst = X + place(r, c);
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    v[u][w] = scaled(v[u][w] & 0xffffu) | (scaled(v[u][w] >> 16) << 16);
                if (rows8) {
                    *reinterpret_cast<u32x4 *>(dst) = v[u];
                } else if (cols8) {
                    // a column of 8: each lane starts at another pair, as all of them
                    // starting at their first would meet in two of the 16 bank groups
                    const u32x4 q = rotate_words(v[u], lane & 3);
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        uint16_t *pair = dst + 2 * ((w + lane) & 3) * xs;
                        pair[0] = static_cast<uint16_t>(q[w]);
                        pair[xs] = static_cast<uint16_t>(q[w] >> 16);
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        *dst = static_cast<uint16_t>(v[u][e >> 1] >> (16 * (e & 1)));
                        const bool end = ++c == n;
                        c = end ? 0 : c;
                        dst += end ? wrap : in;
                    }
                }
            }
        }
        // the ends, at most 7 elements each
        for (int q = tid; q < head + (mn - head - 8 * nvec); q += kThreads) {
            const int e = q < head ? q : 8 * nvec + q;
            const int r = row_of(e);
            X[place(r, e - r * n)] = static_cast<uint16_t>(scaled(x[e]));
        }
    }
    __syncthreads();

    // fragment of rows row0 .. row0+15 of a K-contiguous matrix, k32 step kk
    auto frag = [&](const uint16_t *mat, int stride, int row0, int kk) {
        return *reinterpret_cast<const bf16x8 *>(mat + (row0 + l15) * stride + 32 * kk + 8 * lq);
    };
    // fragment of 16 columns of X contracted along its rows, from the lane's places in the
    // fragment's first and fifth of 8 rows
    auto frag_x = [&](const uint16_t *p, const uint16_t *q) {
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4 *)(p));
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4 *)(q));
        return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    // block (bi, bj)'s lane values (row 16i + l15, columns 16j + 4 lq ..) into A, mirrored
    auto put_a = [&](int bi, int bj, int i, int j, u32x2 v) {
        const int r = 32 * bi + 16 * i + l15, c = 32 * bj + 16 * j + 4 * lq;
        *reinterpret_cast<u32x2 *>(A + r * as + c) = v;
        if (bi != bj) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                A[(c + e) * as + r] = static_cast<uint16_t>(v[e >> 1] >> (16 * (e & 1)));
        }
    };
    auto pack = [](float v0, float v1, float v2, float v3) {
        return u32x2{uint32_t(f32_to_bf16_bits(v0)) | (uint32_t(f32_to_bf16_bits(v1)) << 16),
                     uint32_t(f32_to_bf16_bits(v2)) | (uint32_t(f32_to_bf16_bits(v3)) << 16)};
    };

    constexpr int kUpper = NB * (NB + 1) / 2;
    constexpr int kPerWave = (kUpper + kWaves - 1) / kWaves;
    for (int step = 0; step < g.steps; ++step) {
        const float ca = g.coef[3 * step], cb = g.coef[3 * step + 1], cc = g.coef[3 * step + 2];
        // -------------------------------------------------------- A = X·Xᵀ
#pragma unroll
        for (int t = 0; t < kPerWave; ++t) {
            const int blk = wave + kWaves * t;
            if (blk < kUpper) {
                int bi, bj;
                upper_tile_of(blk, NB, bi, bj);
                f32x4 acc[2][2] = {};
#pragma unroll 4
                for (int kk = 0; kk < lblocks; ++kk) {
                    bf16x8 fr[2], fc[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        fr[i] = frag(X, xs, 32 * bi + 16 * i, kk);
                        fc[i] = frag(X, xs, 32 * bj + 16 * i, kk);
                    }
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[i][j] = mfma_16x16x32(fc[j], fr[i], acc[i][j]);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        put_a(bi, bj, i, j,
                              pack(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]));
            }
        }
        __syncthreads();
        // -------------------------------------------------------- P = b·A + c·A·A
        u32x2 pv[kPerWave][2][2];
#pragma unroll
        for (int t = 0; t < kPerWave; ++t) {
            const int blk = wave + kWaves * t;
            if (blk < kUpper) {
                int bi, bj;
                upper_tile_of(blk, NB, bi, bj);
                f32x4 acc[2][2] = {};
#pragma unroll
                for (int kk = 0; kk < NB; ++kk) {
                    bf16x8 fr[2], fc[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        fr[i] = frag(A, as, 32 * bi + 16 * i, kk);
                        fc[i] = frag(A, as, 32 * bj + 16 * i, kk);
                    }
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[i][j] = mfma_16x16x32(fc[j], fr[i], acc[i][j]);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const int r = 32 * bi + 16 * i + l15, c = 32 * bj + 16 * j + 4 * lq;
                        const u32x2 av = *reinterpret_cast<const u32x2 *>(A + r * as + c);
                        float v[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float ae =
                                bf16_bits_to_f32((av[e >> 1] >> (16 * (e & 1))) & 0xffffu);
                            v[e] = fmaf(cc, acc[i][j][e], cb * ae);
                        }
                        pv[t][i][j] = pack(v[0], v[1], v[2], v[3]);
                    }
            }
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < kPerWave; ++t) {
            const int blk = wave + kWaves * t;
            if (blk < kUpper) {
                int bi, bj;
                upper_tile_of(blk, NB, bi, bj);
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) put_a(bi, bj, i, j, pv[t][i][j]);
            }
        }
        __syncthreads();
        // -------------------------------------------------------- Y = a·X + P·X
        constexpr int kGroups = kWaves / NB;
        const int rb = wave % NB, grp = wave / NB;
        const int kax = rb & ~1;  // k32 step before which a·X is added
        constexpr int kCols = kColBlocks;
        f32x4 acc[kCols][2][2];
        if (grp < kGroups) {
#pragma unroll
            for (int t = 0; t < kCols; ++t)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[t][i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (int kk = 0; kk < NB; ++kk) {
                // one lane address per row, opaque: the blocks differ by constants
                int at = (32 * kk + 8 * lq + (l15 >> 2)) * xs + 32 * grp + 4 * (l15 & 3);
                asm volatile("" : "+v"(at));
                const uint16_t *xk = X + at, *xk4 = xk + 4 * xs;
                bf16x8 fp[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) fp[i] = frag(A, as, 32 * rb + 16 * i, kk);
                if (kk == kax) {
                    int ar = (32 * rb + l15) * xs + 32 * grp + 4 * lq;
                    asm volatile("" : "+v"(ar));
#pragma unroll
                    for (int t = 0; t < kCols; ++t) {
                        if (grp + kGroups * t >= lblocks) break;
#pragma unroll
                        for (int i = 0; i < 2; ++i)
#pragma unroll
                            for (int j = 0; j < 2; ++j) {
                                const u32x2 xv = *reinterpret_cast<const u32x2 *>(
                                    X + ar + 16 * i * xs + 32 * kGroups * t + 16 * j);
#pragma unroll
                                for (int e = 0; e < 4; ++e)
                                    acc[t][i][j][e] = fmaf(
                                        ca,
                                        bf16_bits_to_f32((xv[e >> 1] >> (16 * (e & 1))) & 0xffffu),
                                        acc[t][i][j][e]);
                            }
                    }
                }
#pragma unroll
                for (int t = 0; t < kCols; ++t) {
                    if (grp + kGroups * t >= lblocks) break;
                    bf16x8 fc[2];
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        fc[j] = frag_x(xk + 32 * kGroups * t + 16 * j,
                                       xk4 + 32 * kGroups * t + 16 * j);
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[t][i][j] = mfma_16x16x32(fc[j], fp[i], acc[t][i][j]);
                }
            }
        }
        __syncthreads();
        // Y over X, inside [s, l] (the padding stays zero)
        if (grp < kGroups) {
#pragma unroll
            for (int t = 0; t < kCols; ++t) {
                const int cblk = grp + kGroups * t;
                if (cblk < lblocks) {
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            const int r = 32 * rb + 16 * i + l15;
                            const int c = 32 * cblk + 16 * j + 4 * lq;
                            if (r >= s) continue;
                            uint16_t *dst = X + r * xs + c;
                            const f32x4 &v = acc[t][i][j];
                            const u32x2 h = pack(v[0], v[1], v[2], v[3]);
                            if (c + 4 <= l) {
                                *reinterpret_cast<u32x2 *>(dst) = h;
                            } else {
#pragma unroll
                                for (int e = 0; e < 4; ++e)
                                    if (c + e < l)
                                        dst[e] = static_cast<uint16_t>(h[e >> 1] >> (16 * (e & 1)));
                            }
                        }
                }
            }
        }
        __syncthreads();
    }

    // ------------------------------------------------------------ Y out
    const int head = head_of(y), nvec = (mn - head) / 8;
    const bool whole = n % 8 == 0 && head == 0;
    const bool rows8 = whole && !g.tall, cols8 = whole && g.tall;
    for (int i = tid; i < nvec; i += kThreads) {
        const int e0 = head + 8 * i, r = row_of(e0);
        int c = e0 - r * n;
        const uint16_t *src = X + place(r, c);
        u32x4 v;
        if (rows8) {
            v = *reinterpret_cast<const u32x4 *>(src);
        } else if (cols8) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint16_t *pair = src + 2 * ((w + lane) & 3) * xs;
                v[w] = uint32_t(pair[0]) | (uint32_t(pair[xs]) << 16);
            }
            v = rotate_words(v, -lane & 3);
        } else {
            uint32_t h[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                h[e] = *src;
                const bool end = ++c == n;
                c = end ? 0 : c;
                src += end ? wrap : in;
            }
            v = u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                      h[6] | (h[7] << 16)};
        }
        *reinterpret_cast<u32x4 *>(y + e0) = v;
    }
    for (int q = tid; q < head + (mn - head - 8 * nvec); q += kThreads) {
        const int e = q < head ? q : 8 * nvec + q;
        const int r = row_of(e);
        y[e] = X[place(r, e - r * n)];
    }
}

}  // namespace

bool resident_fits(int64_t m, int64_t n) {
    const int64_t s = m < n ? m : n, l = m < n ? n : m;
    const int64_t nb = (s + 31) / 32, lb = (l + 31) / 32;
    if (nb > kResidentBlocks || lb > kColBlocks * (kWaves / nb)) return false;
    const int64_t bytes =
        2 * 32 * nb * (32 * lb + kRowPad + 32 * nb + kRowPad) + kTailBytes;
    return bytes <= kLdsBytes;
}

hipError_t launch_resident(const ResidentArgs &g, int64_t batch, hipStream_t stream) {
    if (!resident_fits(g.m, g.n) || batch <= 0 || batch >= (int64_t(1) << 31) || g.steps < 0 ||
        g.steps > kResidentSteps || g.chunks > kMaxChunks)
        return hipErrorInvalidValue;
    const void *k = nullptr;
    switch (((g.m < g.n ? g.m : g.n) + 31) / 32) {
        case 1: k = reinterpret_cast<const void *>(&resident_kernel<1>); break;
        case 2: k = reinterpret_cast<const void *>(&resident_kernel<2>); break;
        case 3: k = reinterpret_cast<const void *>(&resident_kernel<3>); break;
        case 4: k = reinterpret_cast<const void *>(&resident_kernel<4>); break;
        case 5: k = reinterpret_cast<const void *>(&resident_kernel<5>); break;
        case 6: k = reinterpret_cast<const void *>(&resident_kernel<6>); break;
        default: return hipErrorInvalidValue;
    }
    ResidentArgs copy = g;
    void *args[] = {&copy};
    return hipLaunchKernel(k, dim3(static_cast<unsigned>(batch)), dim3(kThreads), args, 0, stream);
}

}  // namespace muon_polar
