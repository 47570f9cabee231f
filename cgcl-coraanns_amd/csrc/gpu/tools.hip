// Index-build and evaluation tools on the GPU (C-ABI in include/cora_gpu.h, cora_tool_*):
// rotation of a row block, Lloyd k-means, nearest-centroid assignment and exhaustive
// top-k (ground truth). They reuse the engine's split-FP16 and FP32 GEMMs, row-norm and top-k
// select kernels; host arrays in, host arrays out, device memory in a block a call (dev_block.h).
#include <float.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <random>
#include <string>
#include <vector>

#include "../../../include/cora_gpu.h"
#include "dev_block.h"
#include "engine_internal.h"
#include "host_copy.h"

using namespace cora;

namespace {

thread_local std::string g_tool_error;

// ---- nearest centroid ----
//
// The distances ||x||^2 + ||c||^2 - 2 <x, c> come from a GEMM, in FP32 or on split-FP16 operands,
// each within (K + 34) 2^-24 ((||x|| + ||c||)^2) of the exact value (K products' and sums'
// roundings, the norms' and the combination's, a shift's). Where another centroid lies within
// the two bounds of the smallest distance, the row's candidates are evaluated again in FP64
// (ties -> lower id), so the answer is the FP64 one whichever GEMM ran. On Gaussian mixtures that
// is about one row in a hundred.
//
// The bound grows with the norms. For the split GEMM, rows and centroids that share an offset
// larger than their spread are shifted by it first (set_shift), or every centroid would be a
// candidate. What remains is rows far from all centroids and centroids that repeat: a row of
// more than kNearEvals evaluations is crowded, and the crowded rows of a chunk keep the GEMM's
// answer, its smallest distance, where they would cost more than kCrowdedEvals * (rows + 4096)
// evaluations. After the FP32 GEMM a row of more than kNearFew candidates keeps it.
constexpr uint32_t kNearEvals = 256, kCrowdedEvals = 16, kNearFew = 16;

// Two bounds above the smallest computed distance: no centroid beyond it can be the nearest.
// A candidate's norm is at most ||x|| plus its distance.
__device__ __forceinline__ float nearest_cut(float best, float xnorm, uint32_t dim) {
    const float r = 2.0f * sqrtf(fmaxf(xnorm, 0.0f)) + sqrtf(fmaxf(best, 0.0f));
    return best + 2.2f * (float)(dim + 34) * 0x1p-24f * r * r;
}

// Rows of x and cent may be read four values at a time (the callers of cora_tool_assign_noalloc own
// both arrays, at any alignment).
__device__ __forceinline__ bool quad_rows(const float *x, const float *cent, uint32_t dim) {
    return dim % 4 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(cent)) & 15) == 0;
}

// sum (x - c)^2 in FP64 for N centroids at a time by a group of eight lanes (the same in all of
// them)
template <int N>
__device__ __forceinline__ void group_l2(const float *__restrict__ x, const float *const (&c)[N], uint32_t dim,
                                         bool quads, uint32_t gl, double (&s)[N]) {
#pragma unroll
    for (int j = 0; j < N; ++j)
        s[j] = 0.0;
    const auto term = [](float a, float b, double acc) {
        const double d = (double)a - (double)b;
        return fma(d, d, acc);
    };
    if (quads) {
        for (uint32_t i = 4 * gl; i < dim; i += 32) {
            const float4 a = *reinterpret_cast<const float4 *>(x + i);
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const float4 b = *reinterpret_cast<const float4 *>(c[j] + i);
                s[j] = term(a.x, b.x, s[j]);
                s[j] = term(a.y, b.y, s[j]);
                s[j] = term(a.z, b.z, s[j]);
                s[j] = term(a.w, b.w, s[j]);
            }
        }
    } else {
        for (uint32_t i = gl; i < dim; i += 8) {
            const float a = x[i];
#pragma unroll
            for (int j = 0; j < N; ++j)
                s[j] = term(a, c[j][i], s[j]);
        }
    }
#pragma unroll
    for (int o = 4; o > 0; o >>= 1)
#pragma unroll
        for (int j = 0; j < N; ++j)
            s[j] += __shfl_xor(s[j], o, 64);
}

// argmin over each row of dist [rows][k] (FP32 GEMM); ties -> lower index. A second pass over the
// row lists its candidates where there is another; more than kNearFew are crowded.
__global__ __launch_bounds__(64) void row_argmin_kernel(const float *__restrict__ dist, uint32_t k,
                                                        const float *__restrict__ x, const float *__restrict__ xn,
                                                        const float *__restrict__ cent, uint32_t dim,
                                                        uint32_t *__restrict__ out) {
    __shared__ uint32_t s_cand[kNearFew];
    const float *row = dist + (size_t)blockIdx.x * k;
    const uint32_t lane = threadIdx.x;
    float best = FLT_MAX, next = FLT_MAX;
    uint32_t bi = 0xFFFFFFFFu;
    for (uint32_t j = lane; j < k; j += 64) {
        const float v = row[j];
        if (v < best || (v == best && j < bi)) {
            next = best;
            best = v;
            bi = j;
        } else {
            next = fminf(next, v);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(best, o, 64), on = __shfl_xor(next, o, 64);
        const uint32_t oi = __shfl_xor(bi, o, 64);
        const bool take = ov < best || (ov == best && oi < bi);
        next = fminf(fminf(next, on), take ? best : ov);
        if (take) {
            best = ov;
            bi = oi;
        }
    }
    if (bi != 0xFFFFFFFFu) {
        const float cut = nearest_cut(best, xn[blockIdx.x], dim);
        uint32_t n = 0;
        for (uint32_t j0 = 0; next <= cut && j0 < k && n <= kNearFew; j0 += 64) {
            const uint32_t j = j0 + lane;
            const bool in = j < k && row[j] <= cut;
            const unsigned long long m = __ballot(in);
            const uint32_t at = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (in && at < kNearFew)
                s_cand[at] = j;
            n += (uint32_t)__popcll(m);
        }
        __syncthreads();
        if (n > 1 && n <= kNearFew) {
            const bool quads = quad_rows(x, cent, dim);
            double bd = __longlong_as_double(0x7FF0000000000000ll);
            for (uint32_t i = lane / 8; i < n; i += 8) {
                const float *const c[1] = {cent + (size_t)s_cand[i] * dim};
                double d[1];
                group_l2<1>(x + (size_t)blockIdx.x * dim, c, dim, quads, lane & 7, d);
                if (i < 8 || d[0] < bd || (d[0] == bd && s_cand[i] < bi)) {
                    bd = d[0];
                    bi = s_cand[i];
                }
            }
#pragma unroll
            for (int o = 32; o >= 8; o >>= 1) {
                const double od = __shfl_xor(bd, o, 64);
                const uint32_t oi = __shfl_xor(bi, o, 64);
                if (od < bd || (od == bd && oi < bi)) {
                    bd = od;
                    bi = oi;
                }
            }
        }
    }
    if (lane == 0)
        out[blockIdx.x] = bi == 0xFFFFFFFFu ? 0u : bi;
}

__device__ __forceinline__ float float_of_key(uint32_t key) {
    return __uint_as_float((key & 0x80000000u) ? (key & 0x7FFFFFFFu) : ~key);
}

// The same from the split-FP16 GEMM's smallest and second smallest distance of every 128
// centroids (launch_nearest_gemm): a wave per row; rows with more than one candidate go to
// list [rows], crowded ones from its end (count: how many of each).
__global__ __launch_bounds__(256) void nearest_rows_kernel(const unsigned long long *__restrict__ best,
                                                           const uint32_t *__restrict__ second, uint32_t rows,
                                                           uint32_t tiles, const float *__restrict__ xn, uint32_t dim,
                                                           uint32_t *__restrict__ out, uint32_t *__restrict__ list,
                                                           uint32_t *__restrict__ count) {
    __shared__ uint32_t s_n[2], s_at[2];
    const uint32_t row = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x & 63;
    if (threadIdx.x < 2)
        s_n[threadIdx.x] = 0;
    __syncthreads();
    uint32_t n = 0;  // evaluations: a tile's best, or the whole tile
    if (row < rows) {
        const unsigned long long *b = best + (size_t)row * tiles;
        const uint32_t *sec = second + (size_t)row * tiles;
        unsigned long long mine = ~0ull;
        for (uint32_t t = lane; t < tiles; t += 64)
            mine = min(mine, b[t]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            mine = min(mine, (unsigned long long)__shfl_xor(mine, o, 64));
        const float d = float_of_key((uint32_t)(mine >> 32));
        const bool finite = (mine >> 32) < 0xFF7FFFFFull;  // below +FLT_MAX's key
        if (lane == 0)
            out[row] = finite ? (uint32_t)mine : 0u;
        if (finite) {
            const float cut = nearest_cut(d, xn[row], dim);
            for (uint32_t t = lane; t < tiles; t += 64)
                n += float_of_key(sec[t]) <= cut ? 128u : float_of_key((uint32_t)(b[t] >> 32)) <= cut ? 1u : 0u;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1)
                n += __shfl_xor(n, o, 64);
        }
    }
    // one atomic a workgroup and list: they run one after the other
    const uint32_t which = n > kNearEvals ? 1u : 0u;
    uint32_t at = 0;
    if (n > 1 && lane == 0)
        at = atomicAdd(&s_n[which], 1u);
    __syncthreads();
    if (threadIdx.x < 2 && s_n[threadIdx.x])
        s_at[threadIdx.x] = atomicAdd(&count[threadIdx.x], s_n[threadIdx.x]);
    __syncthreads();
    if (n > 1 && lane == 0) {
        at += s_at[which];
        list[which ? rows - 1 - at : at] = row;
    }
}

// The listed rows' nearest centroid in FP64 over the candidates: a tile's best, or all 128
// centroids of a tile whose second smallest distance is a candidate too. A workgroup per row,
// its 32 groups of eight lanes a centroid each (four where a whole tile is evaluated). What
// bounds it, when few rows are listed, is the chain of a row: 12 MB of 256-dimensional rows,
// k = 256: one wave a centroid, 32 of them in turn, 159 us; this shape 8.6 us.
__global__ __launch_bounds__(256) void nearest_exact_kernel(const unsigned long long *__restrict__ best,
                                                            const uint32_t *__restrict__ second, uint32_t tiles,
                                                            const float *__restrict__ x, const float *__restrict__ xn,
                                                            const float *__restrict__ cent, uint32_t k, uint32_t dim,
                                                            const uint32_t *__restrict__ list,
                                                            const uint32_t *__restrict__ count, uint32_t rows,
                                                            uint32_t *__restrict__ out) {
    __shared__ unsigned long long s_min[4];
    __shared__ double s_d[4];
    __shared__ uint32_t s_c[4];
    __shared__ uint32_t s_item[256], s_whole[256], s_items, s_wholes;
    const uint32_t t = threadIdx.x, wave = t / 64, lane = t & 63, group = t / 8, gl = t & 7;
    const uint32_t near = count[0];
    const bool quads = quad_rows(x, cent, dim);
    const bool crowded = (uint64_t)count[1] * k <= kCrowdedEvals * ((uint64_t)rows + 4096);
    const uint32_t n = near + (crowded ? count[1] : 0u);
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
        const uint32_t row = list[i < near ? i : rows - 1 - (i - near)];
        const unsigned long long *b = best + (size_t)row * tiles;
        const uint32_t *sec = second + (size_t)row * tiles;
        unsigned long long mine = ~0ull;
        for (uint32_t j = t; j < tiles; j += 256)
            mine = min(mine, b[j]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            mine = min(mine, (unsigned long long)__shfl_xor(mine, o, 64));
        if (lane == 0)
            s_min[wave] = mine;
        __syncthreads();
        mine = min(min(s_min[0], s_min[1]), min(s_min[2], s_min[3]));
        const float cut = nearest_cut(float_of_key((uint32_t)(mine >> 32)), xn[row], dim);
        const float *xr = x + (size_t)row * dim;
        double bd = __longlong_as_double(0x7FF0000000000000ll);
        uint32_t bc = 0xFFFFFFFFu;
        const auto take = [&](double d, uint32_t c) {
            if (d < bd || (d == bd && c < bc)) {
                bd = d;
                bc = c;
            }
        };
        // 256 tiles at a time: single candidates and whole tiles to two lists
        for (uint32_t t0 = 0; t0 < tiles; t0 += 256) {
            if (t == 0)
                s_items = s_wholes = 0;
            __syncthreads();
            const uint32_t tile = t0 + t;
            if (tile < tiles) {
                if (float_of_key(sec[tile]) <= cut)
                    s_whole[atomicAdd(&s_wholes, 1u)] = tile;
                else if (float_of_key((uint32_t)(b[tile] >> 32)) <= cut)
                    s_item[atomicAdd(&s_items, 1u)] = (uint32_t)b[tile];
            }
            __syncthreads();
            const uint32_t items = s_items, wholes = s_wholes;
            for (uint32_t j = group; j < items; j += 32) {
                const float *const c[1] = {cent + (size_t)s_item[j] * dim};
                double d[1];
                group_l2<1>(xr, c, dim, quads, gl, d);
                take(d[0], s_item[j]);
            }
            for (uint32_t j = 0; j < wholes; ++j) {
                const uint32_t c0 = 128 * s_whole[j] + group;
                const float *c[4];
                double d[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    c[u] = cent + (size_t)min(c0 + 32 * u, k - 1) * dim;
                group_l2<4>(xr, c, dim, quads, gl, d);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (c0 + 32 * u < k)
                        take(d[u], c0 + 32 * u);
            }
            __syncthreads();  // the lists are written again
        }
#pragma unroll
        for (int o = 32; o >= 8; o >>= 1) {
            const double od = __shfl_xor(bd, o, 64);
            const uint32_t oc = __shfl_xor(bc, o, 64);
            take(od, oc);
        }
        if (lane == 0) {
            s_d[wave] = bd;
            s_c[wave] = bc;
        }
        __syncthreads();
        if (t == 0) {
            for (int w = 1; w < 4; ++w)
                take(s_d[w], s_c[w]);
            if (bc != 0xFFFFFFFFu)
                out[row] = bc;
        }
        __syncthreads();
    }
}

// grid-stride over rows (a dispatch counts its work-items in 32 bits)
__global__ void accumulate_kernel(const float *__restrict__ x, const uint32_t *__restrict__ assign,
                                  uint32_t rows, uint32_t dim, float *__restrict__ sums,
                                  uint32_t *__restrict__ counts) {
    for (uint32_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const uint32_t c = assign[r];
        for (uint32_t d = threadIdx.x; d < dim; d += blockDim.x)
            atomicAdd(&sums[(size_t)c * dim + d], x[(size_t)r * dim + d]);
        if (threadIdx.x == 0)
            atomicAdd(&counts[c], 1u);
    }
}

__global__ void update_kernel(float *__restrict__ cent, const float *__restrict__ sums,
                              const uint32_t *__restrict__ counts, uint32_t k, uint32_t dim) {
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i >= (size_t)k * dim)
        return;
    const uint32_t c = (uint32_t)(i / dim);
    if (counts[c])
        cent[i] = sums[i] / (float)counts[c];
}

// The k selected of one base block, as (distance, global id) candidates:
// cd/ci[row][slot0 + t] for t < k, from the block's distances [rows][len].
__global__ void gather_block_topk_kernel(const float *__restrict__ dist, uint32_t len,
                                         const int32_t *__restrict__ idx, uint32_t rows, uint32_t k,
                                         uint32_t base0, uint32_t stride, uint32_t slot0,
                                         float *__restrict__ cd, uint32_t *__restrict__ ci) {
    const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (t >= (size_t)rows * k)
        return;
    const size_t r = t / k, j = t % k;
    const uint32_t i = (uint32_t)idx[t];
    cd[r * stride + slot0 + j] = dist[r * len + i];
    ci[r * stride + slot0 + j] = base0 + i;
}

#define TCHK(call)                                                                  \
    do {                                                                            \
        hipError_t e_ = (call);                                                     \
        if (e_ != hipSuccess) {                                                     \
            g_tool_error = std::string(#call) + ": " + hipGetErrorString(e_);       \
            return CORA_ERR_RUNTIME;                                                \
        }                                                                           \
    } while (0)

// Assign rows [0, n) of device matrix x to the nearest of k device centroids (FP32 GEMM, the
// distances in d_dist [chunk][k]).
int assign_rows(const float *d_x, size_t n, uint32_t dim, const float *d_c, const float *d_cn,
                uint32_t k, uint32_t *d_assign, float *d_xn, float *d_dist, size_t chunk,
                hipStream_t s) {
    for (size_t b = 0; b < n; b += chunk) {
        const uint32_t rows = (uint32_t)std::min(chunk, n - b);
        launch_row_norms(d_x + b * dim, rows, dim, d_xn, s);
        launch_dist_gemm(d_x + b * dim, d_xn, d_c, d_cn, rows, k, dim, d_dist, s);
        row_argmin_kernel<<<rows, 64, 0, s>>>(d_dist, k, d_x + b * dim, d_xn, d_c, dim, d_assign + b);
    }
    TCHK(hipGetLastError());
    return CORA_OK;
}

// Rows or centroids as split-FP16 operands: [rows][Kp] hi and lo halves (Kp: the dimension
// rounded up to the GEMM's step), scales and squared norms.
struct SplitRows {
    uint16_t *hi, *lo;
    float *scale, *norm;
    void add_to(DevBlock &block, size_t rows, size_t Kp) {
        block.add(hi, rows * Kp);
        block.add(lo, rows * Kp);
        block.add(scale, rows);
        block.add(norm, rows);
    }
    void fill(const float *d_x, size_t row0, uint32_t rows, uint32_t dim, uint32_t Kp, hipStream_t s,
              const float *shift = nullptr, float *zeros = nullptr, uint32_t *zero_counts = nullptr) {
        launch_split_f16_padded(d_x, rows, dim, Kp, hi + row0 * Kp, lo + row0 * Kp, scale + row0, norm + row0, s,
                                nullptr, shift, zeros, zero_counts);
    }
};

// Nearest centroids on the FP16 matrix cores (three FP16 products per term; FP32 has no fast
// matrix path): the distance matrix is never written, 12 bytes per row and 128 centroids
// are. 300,000 x 768 against 8,192: GEMM and argmin 39.4 -> 12.1 ms; k-means of
// 262,144 x 128, k = 1,024: 1.35 -> 0.66 ms an iteration.
struct Nearest {
    uint32_t dim = 0, Kp = 0, k = 0, tiles = 0;
    size_t chunk = 0;
    SplitRows c;
    unsigned long long *best;
    uint32_t *second, *list, *count;
    float *offset;
    const float *shift = nullptr;  // subtracted from rows and centroids (device), or nullptr
    static bool supported(uint64_t dim, uint64_t k) { return k * split_padded(dim) < (1ull << 31); }
    void init(DevBlock &block, uint64_t dim_, uint64_t k_, size_t max_rows) {
        dim = (uint32_t)dim_;
        k = (uint32_t)k_;
        Kp = split_padded(dim_);
        tiles = nearest_tiles(k);
        // 32-bit element offsets of a chunk's rows, 1 GiB of tile minima, and a wave per row within the
        // 2^32 work-items of a dispatch
        chunk = std::max<size_t>(1, std::min<size_t>({max_rows, ((1ull << 31) - 1) / Kp, (1ull << 30) / (12ull * tiles),
                                                      size_t{1} << 25}));
        c.add_to(block, k, Kp);
        block.add(best, chunk * tiles);
        block.add(second, chunk * tiles);
        block.add(list, chunk);
        block.add(count, 2);
        block.add(offset, dim);
    }
    // The mean of up to 64 of the (host) centroids, where it is longer than their spread about it:
    // taking away less would not make the norms much smaller.
    int set_shift(const float *h_c) {
        const size_t step = std::max<size_t>(1, k / 64), n = (k + step - 1) / step;
        std::vector<double> sum(dim, 0.0), squares(dim, 0.0);
        for (size_t i = 0; i < k; i += step)
            for (uint32_t d = 0; d < dim; ++d) {
                const double v = h_c[i * dim + d];
                sum[d] += v;
                squares[d] += v * v;
            }
        std::vector<float> mean(dim);
        double square = 0.0, offset2 = 0.0;
        for (uint32_t d = 0; d < dim; ++d) {
            mean[d] = (float)(sum[d] / (double)n);
            offset2 += (double)mean[d] * mean[d];
            square += squares[d] / (double)n;
        }
        if (!(offset2 > 0.5 * square && offset2 < (double)FLT_MAX))  // nor where it is not finite
            return CORA_OK;
        TCHK(hipMemcpy(offset, mean.data(), dim * 4, hipMemcpyHostToDevice));
        shift = offset;
        return CORA_OK;
    }
    // (k-means: its sums [k][dim] and counts [k] cleared)
    void set_centroids(const float *d_c, hipStream_t s, float *sums = nullptr, uint32_t *counts = nullptr) {
        c.fill(d_c, 0, k, dim, Kp, s, shift, sums, counts);
    }
    // rows [r0, r0 + n) of x (split in xs from row s0): assign[r0 ..]
    void assign(const float *d_x, const SplitRows &xs, size_t s0, size_t n, const float *d_c, uint32_t *d_assign,
                hipStream_t s) {
        for (size_t b = 0; b < n; b += chunk) {
            const uint32_t rows = (uint32_t)std::min(chunk, n - b);
            const size_t at = s0 + b;
            const float *xn = xs.norm + at;
            launch_nearest_gemm(xs.hi + at * Kp, xs.lo + at * Kp, xs.scale + at, xn, c.hi, c.lo, c.scale, c.norm, rows,
                                k, Kp, best, second, count, s);
            nearest_rows_kernel<<<(rows + 3) / 4, 256, 0, s>>>(best, second, rows, tiles, xn, dim, d_assign + b, list,
                                                               count);
            nearest_exact_kernel<<<std::clamp<uint32_t>(rows / 8, 256, 2048), 256, 0, s>>>(best, second, tiles, d_x + b * dim, xn,
                                                                                d_c, k, dim, list, count, rows,
                                                                                d_assign + b);
        }
    }
};

// The split operands of whole arrays take as much device memory again as the arrays. Where it is
// not there, the call goes on without them, on the FP32 GEMM, which reads the rows as they are:
// what fitted the device before still does.
thread_local bool g_no_split = false;  // cora_tool_debug_no_split
bool split_or_fp32(DevBlock &split) {
    if (g_no_split)
        return false;
    if (split.alloc() == hipSuccess)
        return true;
    (void)hipGetLastError();
    return false;
}

// rows whose distances to k centroids the FP32 GEMM forms at a time: 1 GiB of them, and row tiles
// of 64 within a launch's second dimension
size_t fp32_chunk_rows(size_t rows, uint64_t k) {
    return std::max<size_t>(1, std::min<size_t>({rows, (size_t)(1u << 30) / (k * 4), size_t{1} << 21}));
}

// rows of a chunk that is computed on while the next ones are copied: whole GEMM tiles, 64 MiB
size_t copy_chunk_rows(uint64_t dim) { return std::max<size_t>(1, (size_t{64} << 20) / (dim * 4) / 128) * 128; }

// ---- scratch of the allocation-free assignment (cora_tool_assign_noalloc) ----
// Centroid norms, row norms and one block of distances live in this static device array;
// every GPU the library runs on holds its own copy until the process ends. Its host-side
// name is not a device address: host code uses the per-device address that
// hipGetSymbolAddress returns (scratch_address) for kernel arguments.
constexpr size_t kScratchFloats = size_t{4} << 20;  // 16 MiB
static_assert(CORA_NOALLOC_MAX_CENTROIDS * 3 + 192 <= kScratchFloats,
              "the scratch holds the centroid norms and at least one row of distances");
static __device__ __align__(256) float scratch[kScratchFloats];

std::mutex g_scratch_mu;
std::map<int, float *> g_scratch_addr;  // device ordinal -> address of its scratch
// one allocation-free call at a time per device: a call holds its device's lock from the
// scratch address until its kernels have finished
std::mutex g_scratch_use_mu;
std::map<int, std::mutex> g_scratch_use;  // device ordinal -> lock of its scratch

std::mutex &scratch_lock(int device) {
    std::lock_guard<std::mutex> lock(g_scratch_use_mu);
    return g_scratch_use[device];  // std::map never moves its elements
}

// The calling device's scratch address, resolved once per device (the device is current).
int scratch_address(int device, float **out) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    auto it = g_scratch_addr.find(device);
    if (it == g_scratch_addr.end()) {
        float *ptr = nullptr;
        TCHK(hipGetSymbolAddress(reinterpret_cast<void **>(&ptr), HIP_SYMBOL(scratch)));
        if (!ptr) {
            g_tool_error = "hipGetSymbolAddress returned no address for the scratch array";
            return CORA_ERR_RUNTIME;
        }
        it = g_scratch_addr.emplace(device, ptr).first;
    }
    *out = it->second;
    return CORA_OK;
}

constexpr size_t round_floats(size_t n) { return (n + 63) / 64 * 64; }  // 256-byte slots

}  // namespace

void cora::set_tool_error(const char *msg) { g_tool_error = msg; }

extern "C" {

const char *cora_tool_last_error(void) { return g_tool_error.c_str(); }

int cora_tool_debug_no_split(int on) {
    const int was = g_no_split;
    g_no_split = on != 0;
    return was;
}

int cora_tool_rotate(const float *h_x, uint64_t n, uint64_t dim, const float *h_R, uint64_t P,
                     float *h_out, int device) {
    if (!h_x || !h_R || !h_out || !n || !dim || P < dim)
        return CORA_ERR_INVALID_ARGUMENT;
    TCHK(hipSetDevice(device));
    const size_t chunk = 1u << 20;
    DevBlock block;
    float *x, *r, *o;
    block.add(x, std::min<size_t>(n, chunk) * dim);
    block.add(r, dim * P);
    block.add(o, std::min<size_t>(n, chunk) * P);
    TCHK(block.alloc());
    Staging st(device);
    TCHK(hipMemcpy(r, h_R, dim * P * 4, hipMemcpyHostToDevice));
    for (size_t b = 0; b < n; b += chunk) {
        const size_t rows = std::min<size_t>(chunk, n - b);
        int rc = 0;
        TCHK(st.upload(h_x + b * dim, x, rows * dim * 4, copy_chunk_rows(dim) * dim * 4, rc,
                       [&](size_t off, size_t len) {
                           const size_t r0 = off / (dim * 4), m = len / (dim * 4);
                           launch_rotate(x + r0 * dim, r, o + r0 * P, (uint32_t)m, (uint32_t)dim, (uint32_t)P, nullptr);
                           return 0;
                       }));
        TCHK(hipGetLastError());
        TCHK(st.download(o, h_out + b * P, rows * P * 4));  // the rows are read before the next ones come
    }
    return CORA_OK;
}

}  // extern "C"

namespace {

// Re-seed every empty cluster by splitting a populated one, as Faiss's Lloyd k-means does
// after each update (the k-means the reference's index recipe trains with): cluster j is
// chosen with probability proportional to (size_j - 1), its centroid is copied, the two
// copies are pushed apart by a relative 1/1024 in alternating directions per dimension,
// and the size is assumed to split evenly. Without it a centroid left empty stays where it
// was; on well-separated data such centroids drift towards the origin and end up closer
// to every query than any populated cluster, so probe lists fill with empty clusters.
// Returns the number of clusters re-seeded; cent [k][dim] and counts are host copies.
uint32_t split_empty_clusters(std::vector<float> &cent, std::vector<uint32_t> &counts, uint32_t dim,
                              std::mt19937_64 &gen) {
    const uint32_t k = (uint32_t)counts.size();
    constexpr float kEps = 1.0f / 1024.0f;
    uint32_t split = 0;
    for (uint32_t ci = 0; ci < k; ++ci) {
        if (counts[ci])
            continue;
        uint64_t total = 0;
        for (uint32_t j = 0; j < k; ++j)
            total += counts[j] > 1 ? counts[j] - 1 : 0;
        if (!total)
            break;  // nothing left to split
        uint64_t r = std::uniform_int_distribution<uint64_t>(0, total - 1)(gen);
        uint32_t cj = 0;
        for (; cj < k; ++cj) {
            const uint64_t w = counts[cj] > 1 ? counts[cj] - 1 : 0;
            if (r < w)
                break;
            r -= w;
        }
        float *a = &cent[(size_t)ci * dim], *b = &cent[(size_t)cj * dim];
        for (uint32_t d = 0; d < dim; ++d) {
            const float v = b[d];
            a[d] = v * (d % 2 == 0 ? 1 + kEps : 1 - kEps);
            b[d] = v * (d % 2 == 0 ? 1 - kEps : 1 + kEps);
        }
        counts[ci] = counts[cj] / 2;
        counts[cj] -= counts[ci];
        ++split;
    }
    return split;
}

}  // namespace

extern "C" {

// Lloyd k-means on n rows (FP32 squared L2), initial centroids = k distinct rows chosen
// with a seeded generator; after each update, empty clusters are re-seeded by splitting
// populated ones (split_empty_clusters).
int cora_tool_kmeans(const float *h_x, uint64_t n, uint64_t dim, uint64_t k, uint32_t iters,
                     uint64_t seed, float *h_centroids, int device) {
    if (!h_x || !h_centroids || !n || !dim || !k || k > n || k > 0x7FFFFFFF)
        return CORA_ERR_INVALID_ARGUMENT;
    TCHK(hipSetDevice(device));
    std::vector<uint64_t> pick(n);
    for (uint64_t i = 0; i < n; ++i)
        pick[i] = i;
    std::mt19937_64 gen(seed);
    for (uint64_t i = 0; i < k; ++i) {
        std::uniform_int_distribution<uint64_t> u(i, n - 1);
        std::swap(pick[i], pick[u(gen)]);
    }
    std::vector<float> init(k * dim);
    for (uint64_t i = 0; i < k; ++i)
        memcpy(&init[i * dim], h_x + pick[i] * dim, dim * 4);
    bool split = Nearest::supported(dim, k);
    const size_t chunk = fp32_chunk_rows(n, k);
    DevBlock block, split_block, fp32_block;
    float *x, *c, *sums, *cn, *xn, *dist;
    uint32_t *asg, *cnt;
    Nearest near;
    SplitRows xs;
    block.add(x, n * dim);
    block.add(c, k * dim);
    block.add(asg, n);
    block.add(sums, k * dim);
    block.add(cnt, k);
    TCHK(block.alloc());
    if (split) {
        near.init(split_block, dim, k, n);
        xs.add_to(split_block, n, near.Kp);
        split = split_or_fp32(split_block);
    }
    if (!split) {
        fp32_block.add(cn, k);
        fp32_block.add(xn, chunk);
        fp32_block.add(dist, chunk * k);
        TCHK(fp32_block.alloc());
    }
    if (split)
        if (int rc = near.set_shift(init.data()))
            return rc;
    Staging st(device);
    int rc_copy = 0;
    TCHK(st.upload(h_x, x, n * dim * 4, copy_chunk_rows(dim) * dim * 4, rc_copy, [&](size_t off, size_t len) {
        const size_t r0 = off / (dim * 4);
        if (split)
            xs.fill(x + off / 4, r0, (uint32_t)(len / (dim * 4)), (uint32_t)dim, near.Kp, nullptr,
                    near.shift);
        return 0;
    }));
    TCHK(hipMemcpy(c, init.data(), k * dim * 4, hipMemcpyHostToDevice));
    std::vector<uint32_t> counts(k);
    std::mt19937_64 split_gen(seed ^ 0x9E3779B97F4A7C15ull);
    for (uint32_t it = 0; it < iters; ++it) {
        if (split) {
            near.set_centroids(c, nullptr, sums, cnt);
            near.assign(x, xs, 0, n, c, asg, nullptr);
        } else {
            launch_row_norms(c, (uint32_t)k, (uint32_t)dim, cn, nullptr);
            if (int rc = assign_rows(x, n, (uint32_t)dim, c, cn, (uint32_t)k, asg, xn, dist, chunk, nullptr))
                return rc;
            TCHK(hipMemset(sums, 0, k * dim * 4));
            TCHK(hipMemset(cnt, 0, k * 4));
        }
        accumulate_kernel<<<(uint32_t)std::min<uint64_t>(n, 1u << 20), 64>>>(x, asg, (uint32_t)n,
                                                (uint32_t)dim, sums, cnt);
        update_kernel<<<(uint32_t)((k * dim + 255) / 256), 256>>>(c, sums,
                                                                   cnt, (uint32_t)k,
                                                                   (uint32_t)dim);
        TCHK(hipGetLastError());
        TCHK(hipMemcpy(counts.data(), cnt, k * 4, hipMemcpyDeviceToHost));
        if (std::find(counts.begin(), counts.end(), 0u) != counts.end()) {
            TCHK(hipMemcpy(init.data(), c, k * dim * 4, hipMemcpyDeviceToHost));
            if (split_empty_clusters(init, counts, (uint32_t)dim, split_gen))
                TCHK(hipMemcpy(c, init.data(), k * dim * 4, hipMemcpyHostToDevice));
        }
    }
    TCHK(hipDeviceSynchronize());
    TCHK(hipMemcpy(h_centroids, c, k * dim * 4, hipMemcpyDeviceToHost));
    return CORA_OK;
}

int cora_tool_assign(const float *h_x, uint64_t n, uint64_t dim, const float *h_centroids,
                     uint64_t k, uint32_t *h_assign, int device) {
    if (!h_x || !h_centroids || !h_assign || !n || !dim || !k)
        return CORA_ERR_INVALID_ARGUMENT;
    TCHK(hipSetDevice(device));
    const size_t rows_dev = std::min<size_t>(n, 1u << 22);
    const size_t chunk = fp32_chunk_rows(rows_dev, k);
    bool split = Nearest::supported(dim, k);
    DevBlock block, split_block, fp32_block;
    float *x, *c, *cn, *xn, *dist;
    uint32_t *asg;
    Nearest near;
    SplitRows xs;
    block.add(x, rows_dev * dim);
    block.add(c, k * dim);
    block.add(asg, rows_dev);
    TCHK(block.alloc());
    const size_t copy_rows = std::min(rows_dev, copy_chunk_rows(dim));
    if (split) {
        near.init(split_block, dim, k, copy_rows);
        xs.add_to(split_block, copy_rows, near.Kp);
        split = split_or_fp32(split_block);
    }
    if (!split) {
        fp32_block.add(cn, k);
        fp32_block.add(xn, chunk);
        fp32_block.add(dist, chunk * k);
        TCHK(fp32_block.alloc());
    }
    TCHK(hipMemcpy(c, h_centroids, k * dim * 4, hipMemcpyHostToDevice));
    if (split) {
        if (int rc = near.set_shift(h_centroids))
            return rc;
        near.set_centroids(c, nullptr);
    } else
        launch_row_norms(c, (uint32_t)k, (uint32_t)dim, cn, nullptr);
    Staging st(device);
    for (size_t b = 0; b < n; b += rows_dev) {
        const size_t rows = std::min(rows_dev, n - b);
        int rc = 0;
        TCHK(st.upload(h_x + b * dim, x, rows * dim * 4, copy_rows * dim * 4, rc, [&](size_t off, size_t len) {
            const size_t r0 = off / (dim * 4), m = len / (dim * 4);
            float *xc = x + r0 * dim;
            uint32_t *ac = asg + r0;
            if (!split)
                return assign_rows(xc, m, (uint32_t)dim, c, cn, (uint32_t)k, ac, xn,
                                   dist, chunk, nullptr);
            xs.fill(xc, 0, (uint32_t)m, (uint32_t)dim, near.Kp, nullptr, near.shift);
            near.assign(xc, xs, 0, m, c, ac, nullptr);
            return (int)CORA_OK;
        }));
        if (rc)
            return rc;
        TCHK(hipGetLastError());
        TCHK(hipMemcpy(h_assign + b, asg, rows * 4, hipMemcpyDeviceToHost));
    }
    return CORA_OK;
}

// The same assignment on device arrays the caller owns, with no allocation: centroid norms,
// row norms and distance blocks in the static scratch array (nothing in it has to start at
// zero: every value is written before it is read). Calls on one GPU from several host threads
// take turns (a per-device lock held until the call's kernels have finished), so they never
// share the array at the same time.
int cora_tool_assign_noalloc(const float *d_x, uint64_t n, uint64_t dim, const float *d_centroids,
                             uint64_t k, uint32_t *d_assign, int device) {
    if (!d_x || !d_centroids || !d_assign || !n || !dim || !k) {
        g_tool_error = "assign_noalloc: null array or zero size";
        return CORA_ERR_INVALID_ARGUMENT;
    }
    if (k > CORA_NOALLOC_MAX_CENTROIDS || dim > CORA_NOALLOC_MAX_DIM || n > 0xFFFFFFFFull) {
        g_tool_error = "assign_noalloc: at most " + std::to_string(CORA_NOALLOC_MAX_CENTROIDS) +
                       " centroids, dimension " + std::to_string(CORA_NOALLOC_MAX_DIM) +
                       " and 2^32 - 1 rows (the scratch holds " + std::to_string(kScratchFloats * 4 >> 20) + " MiB)";
        return CORA_ERR_INVALID_ARGUMENT;
    }
    TCHK(hipSetDevice(device));
    std::lock_guard<std::mutex> use(scratch_lock(device));
    float *base = nullptr;
    if (int rc = scratch_address(device, &base))
        return rc;
    // layout: centroid norms [k], then per block row norms [chunk] and distances [chunk][k]
    const size_t cn_slot = round_floats(k);
    // rows per block: what the scratch holds, and row offsets of a block within 2^31 elements
    const size_t chunk = std::min<size_t>({n, (kScratchFloats - cn_slot - 64) / (k + 1), ((1ull << 31) - 1) / dim});
    float *cn = base, *xn = base + cn_slot, *dist = xn + round_floats(chunk);
    if (chunk == 0 || (size_t)(dist - base) + chunk * k > kScratchFloats) {
        g_tool_error = "assign_noalloc: the scratch cannot hold one row of distances";
        return CORA_ERR_INVALID_ARGUMENT;
    }
    launch_row_norms(d_centroids, (uint32_t)k, (uint32_t)dim, cn, nullptr);
    if (int rc = assign_rows(d_x, n, (uint32_t)dim, d_centroids, cn, (uint32_t)k, d_assign, xn, dist, chunk,
                             nullptr))
        return rc;
    TCHK(hipStreamSynchronize(nullptr));
    return CORA_OK;
}

}  // extern "C"

namespace {

__global__ void gather_ids_kernel(const uint32_t *__restrict__ ci, uint32_t stride, const int32_t *__restrict__ idx,
                                  uint32_t rows, uint32_t k, uint32_t *__restrict__ out) {
    const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (t < (size_t)rows * k)
        out[t] = ci[t / k * stride + (uint32_t)idx[t]];
}

// cora_tool_topk with the base in nblk blocks of blk rows (the last a few less; each holds at least k)
int topk_call(const float *h_base, uint64_t nb, const float *h_q, uint64_t nq, uint64_t dim, uint64_t k, int metric,
              uint32_t *h_ids, int device, size_t nblk, size_t blk) {
    const size_t qchunk = std::max<size_t>(1, std::min<size_t>(nq, (size_t)(1ull << 30) / blk));
    const size_t stride = nblk * k;
    // the distances from split-FP16 operands; a dimension rounded up to the GEMM's step, and
    // 32-bit element offsets
    const uint32_t Kp = split_padded(dim);
    bool split = blk * Kp < (1ull << 31) && qchunk * Kp < (1ull << 31);
    SplitRows bs, qs;
    DevBlock block, split_block;
    float *b, *bn, *q, *qn, *dist, *cd;
    int32_t *ids;
    uint32_t *ci, *out;
    block.add(b, nb * dim);
    block.add(bn, nb);
    block.add(q, qchunk * dim);
    block.add(qn, qchunk);
    block.add(dist, qchunk * blk);
    block.add(ids, qchunk * k);
    block.add(cd, qchunk * stride);
    block.add(ci, qchunk * stride);
    block.add(out, qchunk * k);
    TCHK(block.alloc());
    if (split) {
        bs.add_to(split_block, nb, Kp);
        qs.add_to(split_block, qchunk, Kp);
        split = split_or_fp32(split_block);
    }
    if (metric != 0) {  // an[m] + bn[n] - 2 * ip with zero norms = -2 ip: same order as -ip
        TCHK(hipMemset(bn, 0, nb * 4));
        TCHK(hipMemset(qn, 0, qchunk * 4));
    }
    const auto load_queries = [&](size_t s, size_t rows) -> int {
        TCHK(hipMemcpy(q, h_q + s * dim, rows * dim * 4, hipMemcpyHostToDevice));
        if (split)
            qs.fill(q, 0, (uint32_t)rows, (uint32_t)dim, Kp, nullptr);
        else if (metric == 0)
            launch_row_norms(q, (uint32_t)rows, (uint32_t)dim, qn, nullptr);
        return CORA_OK;
    };
    // the k best of block j for the loaded queries
    const auto scan = [&](size_t j, size_t rows) {
        const size_t b0 = j * blk, len = std::min(blk, (size_t)nb - b0);
        if (split)
            launch_dist_gemm_f16x3_rows(qs.hi, qs.lo, qs.scale,
                                        metric == 0 ? qs.norm : qn,
                                        bs.hi + b0 * Kp, bs.lo + b0 * Kp,
                                        bs.scale + b0,
                                        (metric == 0 ? bs.norm : bn) + b0, (uint32_t)rows,
                                        (uint32_t)len, Kp, dist, nullptr);
        else
            launch_dist_gemm(q, qn, b + b0 * dim, bn + b0,
                             (uint32_t)rows, (uint32_t)len, (uint32_t)dim, dist, nullptr);
        launch_select(dist, (uint32_t)rows, (uint32_t)len, (uint32_t)k, ids, nullptr);
        const size_t n = rows * k;
        gather_block_topk_kernel<<<(unsigned)((n + 255) / 256), 256>>>(
            dist, (uint32_t)len, ids, (uint32_t)rows, (uint32_t)k, (uint32_t)b0,
            (uint32_t)stride, (uint32_t)(j * k), cd, ci);
    };
    Staging st(device);
    const size_t first = std::min<size_t>(qchunk, nq);
    if (int rc = load_queries(0, first))
        return rc;
    int rc = 0;
    TCHK(st.upload(h_base, b, nb * dim * 4, blk * dim * 4, rc, [&](size_t off, size_t len) {
        const size_t r0 = off / (dim * 4), m = len / (dim * 4);
        if (split)
            bs.fill(b + r0 * dim, r0, (uint32_t)m, (uint32_t)dim, Kp, nullptr);
        else if (metric == 0)
            launch_row_norms(b + r0 * dim, (uint32_t)m, (uint32_t)dim, bn + r0, nullptr);
        scan(r0 / blk, first);
        return 0;
    }));
    for (size_t s = 0; s < nq; s += qchunk) {
        const size_t rows = std::min<size_t>(qchunk, nq - s);
        if (s) {
            if ((rc = load_queries(s, rows)))
                return rc;
            for (size_t j = 0; j < nblk; ++j)
                scan(j, rows);
        }
        const size_t n = rows * k;
        if (nblk > 1)
            launch_select(cd, (uint32_t)rows, (uint32_t)stride, (uint32_t)k, ids, nullptr);
        if (nblk > 1)
            gather_ids_kernel<<<(unsigned)((n + 255) / 256), 256>>>(ci, (uint32_t)stride,
                                                                    ids, (uint32_t)rows, (uint32_t)k,
                                                                    out);
        TCHK(hipGetLastError());
        TCHK(hipMemcpy(h_ids + s * k, nblk > 1 ? out : ci, n * 4, hipMemcpyDeviceToHost));
    }
    return CORA_OK;
}

}  // namespace

extern "C" {

// Exhaustive top-k of nq queries over nb base rows by distances to FP32 accuracy (L2: ||q-x||^2
// through the norm expansion; IP: -<q,x>; split-FP16 products, no further from 64 bits than the
// FP32 GEMM's where measured, dimensions 64 to 1,024), ascending, ties by base index. Callers that need the
// exact order re-rank a few extra candidates in FP64.
int cora_tool_topk(const float *h_base, uint64_t nb, const float *h_q, uint64_t nq, uint64_t dim,
                   uint64_t k, int metric, uint32_t *h_ids, int device) {
    if (!h_base || !h_q || !h_ids || !nb || !nq || !dim || !k || k > nb ||
        k > (uint64_t)kSelectMaxProbe || nb > 0x7FFFFFFF)
        return CORA_ERR_INVALID_ARGUMENT;
    TCHK(hipSetDevice(device));
    // Two levels: the base is cut into nblk blocks; each (query chunk, block) distance tile is
    // selected to its k best, and a query's nblk * k candidates are selected again, ties by slot,
    // which is by id: a block's k are in order of (distance, id) and the blocks in order of id.
    // Blocks of at most 2^20 rows, and of about 2^18 where that leaves a merge of at most 4,096
    // candidates: the first blocks' distances are formed while the later ones are copied.
    size_t nblk = (nb + (1u << 20) - 1) >> 20;
    while (nblk < ((nb + (1u << 18) - 1) >> 18) && (nblk + 1) * k <= 4096)
        ++nblk;
    const size_t blk = (nb + nblk - 1) / nblk;
    nblk = (nb + blk - 1) / blk;
    return topk_call(h_base, nb, h_q, nq, dim, k, metric, h_ids, device, nblk, blk);
}

}  // extern "C"
