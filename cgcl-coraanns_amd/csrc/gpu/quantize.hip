// RaBitQ quantisation of index rows on the GPU (index build): the sign codes and their factors are
// the host builder's bit for bit (csrc/host/index.cpp, which restates rabitq_impl.hpp:76-137
// one_bit_code_with_factor, 276-333 best_rescale_factor, 336-360 quantize_ex and 405-500
// ex_bits_code_with_factor), the ex-codes and theirs at every row whose best t lies at or above
// kQzTight * t_end (see there).
//
// One wave per row. The host forms its double-precision sums in index order. Most of them
// become floats: the sum is formed in parallel here and taken where every value within the
// two orders' rounding bound rounds to one float (nearly always), else formed again in order.
// Float expressions are evaluated term by term as the host does (contraction off), and
// t * |o| + 1e-5 is one fused multiply-add, as the host compiler emits it (and std::fma makes
// explicit).
//
// best_rescale_factor sweeps t upward through the points where some coordinate's code
// increments, in (t, coordinate) order, keeping the t that maximises
// <code + 1/2, |o|> / ||code + 1/2||. Here the sweep runs over windows of t of at most kQzWin
// events: the lanes list their coordinates' increments inside the window, the events are
// sorted in registers on a 22-bit position in the window (events on one position are put in
// order by their own t and coordinate), and each lane evaluates its consecutive events from
// an exclusive sum over the lanes before it. The values |o| are floats of similar size, so the
// host's running sum hardly ever rounds; where that can be shown from their lowest set bits
// every order gives the host's sum, and where not the events are applied one by one. A
// window holding too many events is halved; one holding a single value of t has at most one
// event per coordinate (P <= 1024). Events at or above t_end (first increments of tiny
// coordinates) come last, in a window of their own.
//
// Bound by VALU issue (28,000 instructions a row at P = 768, half of them the sort and the FP64
// square root and division of each of its ~4,900 events). 60,000 rows of 768: 4.0 ms; 110 ms
// with lane 0 forming every sum and applying every event and the windows sorted in LDS as
// (t, event) pairs, 12 ms where only num's initial value was formed in order but a row
// whose initial value had rounded then applied its events one by one (a tail of waves with
// several such rows).
#include <float.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <string>

#include "../../../include/cora_gpu.h"
#include "dev_block.h"
#include "engine_internal.h"
#include "host_copy.h"
#include "lane_ops.h"

#pragma clang fp contract(off)

namespace cora {
namespace {

constexpr int kQzMaxP = 1024;
constexpr int kQzWin = 1024;          // events per sorted window
constexpr int kQzTarget = 896;        // events per window aimed at
constexpr int kQzCap = 127;           // 2^7 - 1 (7 ex-bits)
constexpr int kQzNEnum = 10;
// Where the sweep starts, as a share of t_end. The host starts at 0.77 (kTightStart[7] of
// rabitq_impl.hpp:263-273), so a row whose best t lies between gets the best code from 0.81 up
// here: on Gaussian mixtures 1,630 of 300,000 rows at P = 64, about 55 of 200,000 at 128, 1 of
// 100,000 at 256, none of 340,000 at 384 to 1,024.
constexpr double kQzTight = 0.81;
constexpr double kQzEps = 1e-5;
constexpr float kQzConstEpsilon = 1.9f;  // rabitq_impl.hpp:18
constexpr uint32_t kQzKeyBits = 22;      // sort key of an event: position in its window, then its slot
constexpr uint32_t kQzSlotBits = 32 - kQzKeyBits;
static_assert((1u << kQzSlotBits) == (uint32_t)kQzWin, "a slot of the window per key");

struct QzArgs {
    const float *x;        // [rows][P] rotated rows
    const float *cent;     // [nlist][P] rotated centroids
    const uint32_t *assign;  // [rows]
    uint32_t rows, P;
    int metric;
    uint8_t *bits;         // [rows][P/8] sign bits, dimension 8b + j at bit 7 - j of byte b
    float *f1;             // [rows][3] f_add, f_rescale, f_error
    uint8_t *code;         // [rows][P] ex-code values (complemented for negative residuals)
    float *f2;             // [rows][2] f_add_ex, f_rescale_ex
};

__device__ __forceinline__ void qz_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// t of the increment to code value u of a coordinate with |o| = a (the host's
// static_cast<double>(u) / oi)
__device__ __forceinline__ double inc_t(int u, double a) { return (double)u / a; }

// largest u >= 0 with u / a < tb (a > 0); 0 when none
__device__ int u_floor(double tb, double a) {
    double g = floor(tb * a);
    int u = g < 0.0 ? 0 : (g > 1e9 ? 1000000000 : (int)g);
    while (u > 0 && !(inc_t(u, a) < tb))
        --u;
    while (inc_t(u + 1, a) < tb)
        ++u;
    return u;
}

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o, 64);
    return v;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o, 64);
    return v;
}

__device__ __forceinline__ int wave_min(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v = min(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ __forceinline__ float lane_value(float v, uint32_t lane) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}

// Exponent of the lowest set bit of a positive normal float (it is a multiple of 2 to this
// power); a large value for 0, a very small one for a denormal or a NaN.
__device__ __forceinline__ int low_bit_exp(float a) {
    const uint32_t u = __float_as_uint(a), e = (u >> 23) & 0xFFu;
    if (a == 0.0f)
        return 1000;
    if (e == 0 || e == 255)
        return -1000;
    return (int)e - 127 - 23 + __builtin_ctz((u & 0x7FFFFFu) | 0x800000u);
}

// A double sum of n terms that the host forms in index order and rounds to float. s is the
// same sum in another order and mag the sum of the terms' magnitudes: the two differ by at
// most 2 (n + 8) 2^-53 mag (each is within (n - 1) 2^-53 / (1 - ...) mag of the exact sum). The
// float is the host's when every value that close rounds to it; *ok says so.
__device__ __forceinline__ float sure_float(double s, double mag, uint32_t n, bool &ok) {
    const double e = mag * ((double)(n + 8) * 0x1p-52);
    const float lo = (float)(s - e), hi = (float)(s + e);
    ok = lo == hi && __float_as_uint(lo) == __float_as_uint(hi);
    return lo;
}

// The smaller of a and b where pick is 0, the larger where it is ~0
__device__ __forceinline__ uint32_t pick_of(uint32_t a, uint32_t b, uint32_t pick) {
    return max(min(a, b), min(max(a, b), pick));  // v_med3_u32
}

// One bitonic step (compile-time size and stride) over a wave's 64 NR keys, element
// lane * NR + r in k[r].
template <int NR, uint32_t kSize, uint32_t kStride>
__device__ __forceinline__ void sort_step(uint32_t (&k)[NR], uint32_t lane) {
    constexpr uint32_t N = 64 * NR;
    if constexpr (kStride >= NR) {
        constexpr uint32_t ls = kStride / NR;
        const bool asc = kSize == N || (lane & (kSize / NR)) == 0;
        const uint32_t pick = asc == ((lane & ls) == 0) ? 0u : ~0u;
#pragma unroll
        for (int r = 0; r < NR; ++r)
            k[r] = pick_of(k[r], lane_xor<ls>(k[r]), pick);
    } else {
        const uint32_t pick = kSize < NR || kSize == N || (lane & (kSize / NR)) == 0 ? 0u : ~0u;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            constexpr int st = (int)kStride;
            const int q = r ^ st;
            if (q > r) {
                const uint32_t x = k[r], y = k[q];
                if constexpr (kSize < NR) {
                    const bool asc = (r & (int)kSize) == 0;
                    k[r] = asc ? min(x, y) : max(x, y);
                    k[q] = asc ? max(x, y) : min(x, y);
                } else {
                    k[r] = pick_of(x, y, pick);
                    k[q] = pick_of(x, y, ~pick);
                }
            }
        }
    }
}

template <int NR, uint32_t kSize, uint32_t kStride>
__device__ __forceinline__ void sort_steps(uint32_t (&k)[NR], uint32_t lane) {
    sort_step<NR, kSize, kStride>(k, lane);
    if constexpr (kStride > 1)
        sort_steps<NR, kSize, kStride / 2>(k, lane);
    else if constexpr (kSize < 64 * NR)
        sort_steps<NR, kSize * 2, kSize>(k, lane);
}

// One wave's 64 NR keys, element lane * NR + r in k[r], sorted ascending.
template <int NR>
__device__ __forceinline__ void sort_keys(uint32_t (&k)[NR], uint32_t lane) {
    sort_steps<NR, 2, 1>(k, lane);
}

// The sweep's state (wave-uniform)
struct QzSweep {
    double num, den;       // <code + 1/2, |o|> and ||code + 1/2||^2 after the events applied so far
    double best_ip, best_t;
};

// Applies a window's n events (s_e[slot] = coordinate << 8 | code value, s_key[slot] their
// keys) in (t, coordinate) order. NR registers a lane hold them (n <= 64 NR). exact: the events'
// |o| are multiples of the last place that num has at the end of the sweep, so their own sums
// are exact in any order and num rounds only where it passes a power of two: the lanes then form
// the running sums of their consecutive events in parallel, and num before and after that event
// from them. Otherwise the events are applied one after the other.
template <int NR>
__device__ void apply_events(QzSweep &w, uint32_t n, const uint32_t *s_e, uint32_t *s_key, const float *s_abs,
                             bool exact, uint32_t lane) {
    // opaque here, or the sort's lane masks are formed once for the row and held (and spilled)
    // in SGPRs
    asm volatile("" : "+v"(lane));
    uint32_t k[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const uint32_t i = lane * NR + r;
        k[r] = i < n ? s_key[i] : 0xFFFFFFFFu;
    }
    sort_keys<NR>(k, lane);
    const auto t_of = [&](uint32_t e) { return inc_t((int)(e & 255u), (double)s_abs[e >> 8]); };
    // events on the same key, or on neighbouring ones (a key comes from a t that is rounded a few
    // times more): neighbours now, put in order by their own t (then by coordinate) with odd-even
    // exchanges
    const auto close = [](uint32_t x, uint32_t y) {
        const int d = (int)(x >> kQzSlotBits) - (int)(y >> kQzSlotBits);
        return d >= -1 && d <= 1;
    };
    bool tie = false;
    const uint32_t up = __shfl_down(k[0], 1, 64);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const uint32_t nx = r + 1 < NR ? k[r + 1 < NR ? r + 1 : r] : up;
        const uint32_t i = lane * NR + r;
        tie |= i + 1 < n && close(k[r], nx);
    }
    const auto to_lds = [&]() {
        qz_sync();
#pragma unroll
        for (int r = 0; r < NR; ++r)
            if (lane * NR + r < n)
                s_key[lane * NR + r] = k[r];
        qz_sync();
    };
    if (__any(tie)) {
        to_lds();
        for (bool again = true; again;) {
            again = false;
            for (uint32_t odd = 0; odd < 2; ++odd) {
                bool moved = false;
                for (uint32_t i = 2 * lane + odd; i + 1 < n; i += 128) {
                    const uint32_t a = s_key[i], b = s_key[i + 1];
                    if (!close(a, b))
                        continue;
                    const uint32_t ea = s_e[a & (kQzWin - 1)], eb = s_e[b & (kQzWin - 1)];
                    const double ta = t_of(ea), tb = t_of(eb);
                    if (ta > tb || (ta == tb && (ea >> 8) > (eb >> 8))) {
                        s_key[i] = b;
                        s_key[i + 1] = a;
                        moved = true;
                    }
                }
                again |= __any(moved) != 0;
                qz_sync();
            }
        }
#pragma unroll
        for (int r = 0; r < NR; ++r)
            if (lane * NR + r < n)
                k[r] = s_key[lane * NR + r];
    }
    uint32_t ev[NR];
    double sn = 0.0;
    uint32_t sd = 0;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        ev[r] = lane * NR + r < n ? s_e[k[r] & (kQzWin - 1)] : 0u;
        if (lane * NR + r < n) {
            sn += (double)s_abs[ev[r] >> 8];
            sd += 2 * (ev[r] & 255u);
        }
    }
    // sums over the lanes before this one
    double pn = sn;
    uint32_t pd = sd;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double yn = __shfl_up(pn, o, 64);
        const uint32_t yd = __shfl_up(pd, o, 64);
        if (lane >= (uint32_t)o) {
            pn += yn;
            pd += yd;
        }
    }
    const double total_n = __shfl(pn, 63, 64);
    const uint32_t total_d = __shfl(pd, 63, 64);
    // the power of two above num; the events pass it at most once, or are applied in turn
    const double up2 = ldexp(1.0, ilogb(w.num) + 1);
    if (!exact || !(w.num > 0.0 && w.num + total_n < 2.0 * up2)) {
        to_lds();
        for (uint32_t i = 0; i < n; ++i) {
            const uint32_t e = s_e[s_key[i] & (kQzWin - 1)];
            w.den += (double)(2 * (int)(e & 255u));
            w.num += (double)s_abs[e >> 8];
            const double ip = w.num / sqrt(w.den);
            if (ip > w.best_ip) {
                w.best_ip = ip;
                w.best_t = t_of(e);
            }
        }
        qz_sync();
        return;
    }
    // pc: the sum of the events up to the one that passes it (infinity: none does), and num there
    double pc = __longlong_as_double(0x7FF0000000000000ll), vc = 0.0;
    if (!(w.num + total_n < up2)) {
        double c = pn - sn, mine = 0.0;
        bool passed = false;
#pragma unroll
        for (int r = 0; r < NR; ++r)
            if (lane * NR + r < n) {
                c += (double)s_abs[ev[r] >> 8];
                if (!passed && !(w.num + c < up2)) {
                    passed = true;
                    mine = c;
                }
            }
        pc = __shfl(mine, __builtin_ctzll(__ballot(passed)), 64);
        vc = w.num + pc;
    }
    double sum = pn - sn, den = w.den + (double)(pd - sd);
    double best = w.best_ip;
    uint32_t best_e = 0;
    bool found = false;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        if (lane * NR + r < n) {
            den += (double)(2 * (int)(ev[r] & 255u));
            sum += (double)s_abs[ev[r] >> 8];
            const double num = sum < pc ? w.num + sum : vc + (sum - pc);
            const double ip = num / sqrt(den);
            if (ip > best) {
                best = ip;
                best_e = ev[r];
                found = true;
            }
        }
    }
    // the first of the largest: lanes hold consecutive events
    double mx = best;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        mx = fmax(mx, __shfl_xor(mx, o, 64));
    const unsigned long long who = __ballot(found && best == mx);
    if (who) {
        const uint32_t e = __builtin_amdgcn_readlane(best_e, (uint32_t)__builtin_ctzll(who));
        w.best_ip = mx;
        w.best_t = t_of(e);
    }
    w.num = total_n < pc ? w.num + total_n : vc + (total_n - pc);
    w.den += (double)total_d;
    qz_sync();
}

// One wave per row, coordinates 64 r + lane (RMAX >= P / 64). Three waves a SIMD: the sort's
// registers and the lists of a window in LDS allow no more.
template <int RMAX>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(RMAX > 12 ? 2 : 3))) void quantize_kernel(const QzArgs a) {
    __shared__ float s_abs[64 * RMAX];
    __shared__ uint32_t s_e[kQzWin], s_key[kQzWin];
    const uint32_t lane = threadIdx.x, P = a.P;
    const int R = (int)(P / 64);
    for (uint32_t row = blockIdx.x; row < a.rows; row += gridDim.x) {
        const float *x = a.x + (size_t)row * P;
        const float *cg = a.cent + (size_t)a.assign[row] * P;
        // the residual and the centroid; read again after the sweep, whose registers they
        // would take (256 VGPRs and one wave a SIMD at P = 768, against three)
        float o[RMAX], c[RMAX];
        const auto load_row = [&]() {
#pragma unroll
            for (int r = 0; r < RMAX; ++r) {
                o[r] = c[r] = 0.0f;
                if (r < R) {
                    c[r] = cg[64 * r + lane];
                    o[r] = x[64 * r + lane] - c[r];
                }
            }
        };
        load_row();
        // a sum the host forms in index order, one term after the other (every lane)
        const auto in_order = [&](auto term) -> double {
            double s = 0.0;
#pragma unroll
            for (int r = 0; r < RMAX; ++r)
                if (r < R)
                    for (uint32_t l = 0; l < 64; ++l)
                        s += term(lane_value(o[r], l), lane_value(c[r], l));
            return s;
        };
        // the float of such a sum: from the parallel sum where its rounding is sure
        const auto sum_float = [&](auto term) -> float {
            double s = 0.0, mag = 0.0;
#pragma unroll
            for (int r = 0; r < RMAX; ++r)
                if (r < R) {
                    const double v = term(o[r], c[r]);
                    s += v;
                    mag += fabs(v);
                }
            bool ok;
            const float f = sure_float(wave_sum(s), wave_sum(mag), P, ok);
            if (ok)
                return f;
            return (float)in_order(term);
        };
        // ---- one-bit code and factors (quantize_one_bit) ----
        {
            unsigned long long mine = 0;
#pragma unroll
            for (int r = 0; r < RMAX; ++r)
                if (r < R) {
                    const unsigned long long m = __ballot(o[r] > 0.0f);
                    mine = lane == (uint32_t)r ? m : mine;
                }
            // bit 8b + j of the ballot -> bit 7 - j of byte b
            if (lane < (uint32_t)R)
                *reinterpret_cast<unsigned long long *>(a.bits + (size_t)row * (P / 8) + 8 * lane) =
                    __builtin_bswap64(__builtin_bitreverse64(mine));
        }
        const auto sign_xu = [](float ov) { return (ov > 0.0f ? 1.0f : 0.0f) - 0.5f; };
        const float l2_sqr = sum_float([](float ov, float) { return (double)ov * ov; });
        const float l2 = sqrtf(l2_sqr);
        const float oc = sum_float([](float ov, float cv) { return (double)ov * cv; });
        {
            float ip_resi = sum_float([&](float ov, float) { return (double)ov * sign_xu(ov); });
            const float ip_cent = sum_float([&](float ov, float cv) { return (double)cv * sign_xu(ov); });
            if (lane == 0) {
                if (ip_resi == 0.0f)
                    ip_resi = INFINITY;
                const float xu_sqr = (float)((double)P * 0.25);
                const float err = l2 * kQzConstEpsilon *
                                  sqrtf((((l2_sqr * xu_sqr) / (ip_resi * ip_resi)) - 1.0f) / (float)(P - 1));
                float *f = a.f1 + (size_t)row * 3;
                if (a.metric == 0) {
                    f[0] = l2_sqr + (2.0f * l2_sqr * ip_cent / ip_resi);
                    f[1] = -2.0f * l2_sqr / ip_resi;
                    f[2] = 2.0f * err;
                } else {
                    f[0] = 1.0f - oc + (l2_sqr * ip_cent / ip_resi);
                    f[1] = -l2_sqr / ip_resi;
                    f[2] = err;
                }
            }
        }
        // ---- ex-code (quantize_ex_bits, best_rescale_factor) ----
        const float norm = l2;
        float mx = 0.0f;
#pragma unroll
        for (int r = 0; r < RMAX; ++r)
            if (r < R) {
                const float v = fabsf(o[r] / norm);
                s_abs[64 * r + lane] = v;
                mx = fmaxf(mx, v);
            }
#pragma unroll
        for (int s = 32; s > 0; s >>= 1)
            mx = fmaxf(mx, __shfl_xor(mx, s, 64));
        qz_sync();
        const double max_o = (double)mx;
        const double t_end = (double)(kQzCap + kQzNEnum) / max_o;
        const double t_start = t_end * kQzTight;
        // per coordinate, a byte each: the next increment, the last main one U (code values
        // c + 1 .. U, all with t < t_end, c the initial code; U = c when the first is not) and the
        // next increment after the window being listed (all at most 128)
        uint32_t st[RMAX];
        uint32_t nmain = 0, den0 = 0;
        double lo = t_end, num0 = 0.0, sum_end = 0.0;
        int low = 1000, low_ev = 1000;  // lowest bits of all |o|, and of those with main increments
#pragma unroll
        for (int r = 0; r < RMAX; ++r) {
            st[r] = 1;
            if (r < R) {
                const float af = s_abs[64 * r + lane];
                const double ai = (double)af;
                const int ci = (int)fma(t_start, ai, kQzEps);
                const double t1 = inc_t(ci + 1, ai);
                int U = ci;
                low = min(low, low_bit_exp(af));
                if (t1 < t_end) {
                    U = ci + 1;
                    if (ci + 2 <= kQzCap && inc_t(ci + 2, ai) < t_end)
                        U = min(kQzCap, u_floor(t_end, ai));
                    lo = fmin(lo, t1);
                    low_ev = min(low_ev, low_bit_exp(af));
                }
                st[r] = (uint32_t)(ci + 1) | (uint32_t)U << 8;
                nmain += (uint32_t)(U - ci);
                den0 += (uint32_t)(ci * ci + ci);
                num0 += (ci + 0.5) * ai;
                sum_end += (max(U, ci + 1) + 0.5) * ai;
            }
        }
        nmain = wave_sum_u32(nmain);
        low = wave_min(low);
        low_ev = wave_min(low_ev);
#pragma unroll
        for (int s = 32; s > 0; s >>= 1)
            lo = fmin(lo, __shfl_xor(lo, s, 64));
        QzSweep w;
        w.den = (double)P * 0.25 + (double)wave_sum_u32(den0);  // exact
        w.best_ip = w.best_t = 0.0;
        num0 = wave_sum(num0);
        // Every term of num is a multiple of 2^(low - 1) and no partial sum, in any order and with
        // all events, exceeds sum (last code + 1/2) |o|: where that is below 2^53 such units all
        // additions are exact and their order does not matter. (At P = 768 this holds unless some
        // |o| is below about 2^-18 without trailing zero bits: 94 of 100 Gaussian rows.) Otherwise
        // the initial sum is formed in order. The main increments belong to coordinates of some
        // size and are practically always multiples of num's last place (see apply_events).
        const double bound = 1.0001 * wave_sum(sum_end);
        const bool exact_all = low > -900 && bound < ldexp(1.0, 52 + min(low, 500));
        const bool exact_main = low_ev > -900 && bound < ldexp(1.0, 52 + min(low_ev, 500));
        if (!exact_all) {
            num0 = 0.0;
            for (uint32_t i = 0; i < P; ++i) {
                const double ai = (double)s_abs[i];
                const int ci = (int)fma(t_start, ai, kQzEps);
                num0 += (ci + 0.5) * ai;
            }
        }
        w.num = num0;
        const auto apply = [&](uint32_t n, bool exact) {
            if (n > 256)
                apply_events<16>(w, n, s_e, s_key, s_abs, exact, lane);
            else if (n)
                apply_events<4>(w, n, s_e, s_key, s_abs, exact, lane);
        };
        // main increments in windows [ta, tb) of t
        if (nmain > 0) {
            const uint32_t nwin = (nmain + kQzTarget - 1) / kQzTarget;
            const double width = (t_end - lo) / (double)nwin;
            double ta = lo;
            uint32_t wi = 1;
            while (ta < t_end) {
                double tb = wi >= nwin ? t_end : fmin(t_end, lo + width * (double)wi);
                if (!(tb > ta))
                    tb = t_end;
                uint32_t n;
                for (;;) {
                    const double scale = (double)((1u << kQzKeyBits) - 1u) / (tb - ta);
                    n = 0;
#pragma unroll
                    for (int r = 0; r < RMAX; ++r)
                        if (r < R) {
                            const double ai = (double)s_abs[64 * r + lane];
                            const uint32_t U = (st[r] >> 8) & 255u;
                            uint32_t u = st[r] & 255u;
                            // the last increment u1 / a < tb: floor(tb a), and where tb a is that
                            // close to a whole number, the division's own answer
                            const double v = fmin(tb * ai, 256.0), m = rint(v);
                            uint32_t u1 = (uint32_t)v;
                            if (fabs(v - m) <= v * 0x1p-48)
                                u1 = inc_t((int)m, ai) < tb ? (uint32_t)m : (uint32_t)m - 1u;
                            u1 = min(u1, U);
                            const uint32_t cnt = u1 + 1 > u ? u1 + 1 - u : 0u;
                            // slots in coordinate order
                            uint32_t slot = n;
                            for (uint32_t bit = 0; bit < 8; ++bit) {
                                if (!__any(cnt >> bit))
                                    break;
                                const unsigned long long mk = __ballot((cnt >> bit) & 1u);
                                slot += __builtin_amdgcn_mbcnt_hi((uint32_t)(mk >> 32),
                                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)mk, 0u))
                                        << bit;
                                n += (uint32_t)__popcll(mk) << bit;
                            }
                            st[r] = (st[r] & 0xFFFFu) | (u + cnt) << 16;
                            // keys from u * (scale / a), the quotient by one Newton step: roundings
                            // away from u / a, see apply_events
                            const double ra0 = __builtin_amdgcn_rcp(ai);
                            const double ks = scale * fma(fma(-ai, ra0, 1.0), ra0, ra0), k0 = ta * scale;
                            const uint32_t e = (64u * r + lane) << 8;
                            for (uint32_t j = 0; j < cnt && slot < (uint32_t)kQzWin; ++j, ++slot, ++u) {
                                const int key = (int)fma((double)u, ks, -k0);
                                s_e[slot] = e | u;
                                s_key[slot] =
                                    (uint32_t)min(max(key, 0), (1 << kQzKeyBits) - 1) << kQzSlotBits | slot;
                            }
                        }
                    if (n <= (uint32_t)kQzWin)
                        break;
                    double mid = ta + (tb - ta) * 0.5;
                    if (!(mid > ta))
                        mid = nextafter(ta, t_end);  // a single value of t: at most P events
                    tb = mid;
                }
#pragma unroll
                for (int r = 0; r < RMAX; ++r)
                    st[r] = (st[r] & 0xFF00u) | st[r] >> 16;
                qz_sync();
                apply(n, exact_main);
                ta = tb;
                if (ta >= lo + width * (double)wi)
                    ++wi;
            }
        }
        // increments at or above t_end: the first ones of coordinates without a main one, at
        // most P of them. Their keys are the leading bits of t as a float (monotone; infinity last).
        {
            uint32_t n = 0;
#pragma unroll
            for (int r = 0; r < RMAX; ++r)
                if (r < R) {
                    const double ai = (double)s_abs[64 * r + lane];
                    const int ci = (int)fma(t_start, ai, kQzEps);
                    const double t1 = inc_t(ci + 1, ai);
                    const bool in = t1 >= t_end;
                    const unsigned long long m = __ballot(in);
                    if (in) {
                        const uint32_t slot = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                        s_e[slot] = ((64u * r + lane) << 8) | (uint32_t)(ci + 1);
                        s_key[slot] = (__float_as_uint((float)t1) >> (32 - kQzKeyBits) << kQzSlotBits) | slot;
                    }
                    n += (uint32_t)__popcll(m);
                }
            qz_sync();
            apply(n, exact_all);
        }
        const double t = w.best_t;
        load_row();
        // codes (quantize_ex)
        float cd[RMAX], hv[RMAX];  // the code value, and code + 1/2 of the magnitude
#pragma unroll
        for (int r = 0; r < RMAX; ++r) {
            cd[r] = hv[r] = 0.0f;
            if (r < R) {
                const uint32_t v =
                    (uint32_t)min((int)fma(t, (double)s_abs[64 * r + lane], kQzEps), kQzCap) & 0xFFu;
                const uint32_t d = o[r] < 0.0f ? ~v & (uint32_t)kQzCap : v;
                a.code[(size_t)row * P + 64 * r + lane] = (uint8_t)d;
                hv[r] = (float)v + 0.5f;
                cd[r] = (float)d;
            }
        }
        {
            double s = 0.0, mag = 0.0;
#pragma unroll
            for (int r = 0; r < RMAX; ++r)
                if (r < R) {
                    const double v = (double)hv[r] * (double)s_abs[64 * r + lane];
                    s += v;
                    mag += fabs(v);
                }
            s = wave_sum(s);
            // 1 / ipnorm falls as ipnorm grows: the float is the host's when both ends agree
            const double e = wave_sum(mag) * ((double)(P + 8) * 0x1p-52);
            float ipnorm_inv = (float)(1.0 / (s - e));
            if (!(ipnorm_inv == (float)(1.0 / (s + e)))) {
                double ipnorm = 0.0;
#pragma unroll
                for (int r = 0; r < RMAX; ++r)
                    if (r < R)
                        for (uint32_t l = 0; l < 64; ++l)
                            ipnorm += (double)lane_value(hv[r], l) * (double)s_abs[64 * r + l];
                ipnorm_inv = (float)(1.0 / ipnorm);
            }
            if (!isnormal(ipnorm_inv))
                ipnorm_inv = 1.0f;
            const float cb = -((float)(1 << 7) - 0.5f);
            // <o, xu> and <c, xu> with xu = code - 127.5 (the sign bit in bit 7)
            const auto xu_of = [&](float dv, float ov) { return (dv + (ov >= 0.0f ? (float)(1u << 7) : 0.0f)) + cb; };
            const auto pair_sum = [&](auto value) -> float {
                double s = 0.0, mag = 0.0;
#pragma unroll
                for (int r = 0; r < RMAX; ++r)
                    if (r < R) {
                        const double v = (double)value(r, o[r], c[r]) * xu_of(cd[r], o[r]);
                        s += v;
                        mag += fabs(v);
                    }
                bool ok;
                const float f = sure_float(wave_sum(s), wave_sum(mag), P, ok);
                if (ok)
                    return f;
                double q = 0.0;
#pragma unroll
                for (int r = 0; r < RMAX; ++r)
                    if (r < R)
                        for (uint32_t l = 0; l < 64; ++l) {
                            const float ov = lane_value(o[r], l), cv = lane_value(c[r], l);
                            q += (double)value(r, ov, cv) * xu_of(lane_value(cd[r], l), ov);
                        }
                return (float)q;
            };
            float ip_resi = pair_sum([](int, float ov, float) { return ov; });
            const float ip_cent = pair_sum([](int, float, float cv) { return cv; });
            if (lane == 0) {
                if (ip_resi == 0.0f)
                    ip_resi = INFINITY;
                float *f = a.f2 + (size_t)row * 2;
                if (a.metric == 0) {
                    f[0] = l2_sqr + (2.0f * l2_sqr * ip_cent / ip_resi);
                    f[1] = ipnorm_inv * -2.0f * l2;
                } else {
                    f[0] = 1.0f - oc + (l2_sqr * ip_cent / ip_resi);
                    f[1] = ipnorm_inv * -l2;
                }
            }
        }
        qz_sync();
    }
}

#define QCHK(call)                                                                  \
    do {                                                                            \
        hipError_t e_ = (call);                                                     \
        if (e_ != hipSuccess) {                                                     \
            set_tool_error((std::string(#call) + ": " + hipGetErrorString(e_)).c_str()); \
            return CORA_ERR_RUNTIME;                                                \
        }                                                                           \
    } while (0)

}  // namespace
}  // namespace cora

using namespace cora;

extern "C" {

int cora_tool_quantize(const float *h_x, uint64_t n, uint64_t dim, const float *h_R, uint64_t P,
                       const float *h_centroids, uint64_t nlist, const uint32_t *h_assign, int metric,
                       uint8_t *h_bits, float *h_f1, uint8_t *h_code, float *h_f2, int device) {
    if (!h_x || !h_R || !h_centroids || !h_assign || !h_bits || !h_f1 || !h_code || !h_f2 || !n || !dim ||
        P < dim || P % 64 || P > (uint64_t)kQzMaxP || !nlist || (metric != 0 && metric != 1)) {
        set_tool_error("cora_tool_quantize: invalid argument (P % 64 == 0, dim <= P <= 1024, metric 0 or 1)");
        return CORA_ERR_INVALID_ARGUMENT;
    }
    for (uint64_t i = 0; i < n; ++i)
        if (h_assign[i] >= nlist) {
            set_tool_error("cora_tool_quantize: cluster id out of range");
            return CORA_ERR_INVALID_ARGUMENT;
        }
    QCHK(hipSetDevice(device));
    const size_t chunk = std::min<size_t>(n, (size_t)1 << 20);
    DevBlock block;
    float *x, *r, *xr, *c, *f1, *f2;
    uint32_t *asg;
    uint8_t *bits, *code;
    block.add(x, chunk * dim);
    block.add(r, dim * P);
    block.add(xr, chunk * P);
    block.add(c, nlist * P);
    block.add(asg, chunk);
    block.add(bits, chunk * P / 8);
    block.add(f1, chunk * 3);
    block.add(code, chunk * P);
    block.add(f2, chunk * 2);
    QCHK(block.alloc());
    QCHK(hipMemcpy(r, h_R, dim * P * 4, hipMemcpyHostToDevice));
    QCHK(hipMemcpy(c, h_centroids, nlist * P * 4, hipMemcpyHostToDevice));
    int cus = 256;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    auto *kernel = P <= 128   ? quantize_kernel<2>
                   : P <= 256 ? quantize_kernel<4>
                   : P <= 512 ? quantize_kernel<8>
                   : P <= 768 ? quantize_kernel<12>
                              : quantize_kernel<16>;
    // the waves that are resident together: a second round of a few would run alone
    int per_cu = 0;
    QCHK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64, 0));
    const size_t waves = (size_t)cus * std::max(1, per_cu);
    // rows rotated and quantised while the next ones are copied: four rounds of the resident waves
    const size_t step = std::min(chunk, 4 * waves);
    Staging st(device);
    for (size_t b = 0; b < n; b += chunk) {
        const size_t rows = std::min(chunk, (size_t)n - b);
        QCHK(hipMemcpy(asg, h_assign + b, rows * 4, hipMemcpyHostToDevice));
        int rc = 0;
        QCHK(st.upload(h_x + b * dim, x, rows * dim * 4, step * dim * 4, rc, [&](size_t off, size_t len) {
            const size_t r0 = off / (dim * 4), m = len / (dim * 4);
            float *out = xr + r0 * P;
            launch_rotate(x + r0 * dim, r, out, (uint32_t)m, (uint32_t)dim, (uint32_t)P, nullptr);
            QzArgs qa{out,    c,  asg + r0, (uint32_t)m, (uint32_t)P, metric, bits + r0 * (P / 8), f1 + r0 * 3,
                      code + r0 * P, f2 + r0 * 2};
            kernel<<<(uint32_t)std::min<size_t>(m, waves), 64>>>(qa);
            return 0;
        }));
        QCHK(hipGetLastError());
        QCHK(st.download(bits, h_bits + b * (P / 8), rows * (P / 8)));
        QCHK(st.download(f1, h_f1 + b * 3, rows * 12));
        QCHK(st.download(code, h_code + b * P, rows * P));
        QCHK(st.download(f2, h_f2 + b * 2, rows * 8));
    }
    return CORA_OK;
}

}  // extern "C"
