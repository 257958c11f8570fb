// Gradient preconditioning on the device (toolbox/postprocess.py:20-111): taper, the
// illumination preconditioner built from Gaussian-smoothed illuminations, gradient
// smoothing, mask and scaling, in FP64 like the reference's numpy (the in-place taper
// product keeps the float32 gradient's dtype, as there).
//
// smooth2d (toolbox/tools.py:239-275) convolves with the normalised (2 span + 1)^2
// Gaussian F[a][b] = e_a e_b / (sum e)^2, e_a = exp(-(x_a / span)^2 / 2), x_a = 2a - 2 span
// (zero padding, 'same' size), and divides by the same convolution of a field of ones.
// F is separable, so both become two 1-D passes: along z, then along x, and the ones
// field's convolution is the product of the kernel's partial sums over the valid taps.
// All arrays are [nx][nz] (z fastest).
//
// The work is small (801x267: 1.7 MB a field, 35 M multiply-adds a smoothing with 40 samples
// span), so launches and serial parts decide.  One workgroup per maximum, one thread per
// kernel's weights and a launch per pass of each field took 513 us there in 27 launches; now 8
// launches, 9 with a land mute, 75 us: fields that go through the same pass share a launch (blockIdx.z), sums and
// products ride on the pass that makes their inputs, and every pass leaves the maximum of its
// output in M by an atomic on an order-preserving integer form (a maximum has no order, so the
// bits are those of any other way).
#include "fd_common.h"

namespace swit {
namespace pc {

typedef unsigned long long u64;

// M: maxima as integers that order like the doubles, 0 before any value
constexpr int kMaxForw = 0, kMaxBack = 1, kMaxPre = 2, kMaxTaper = 3, kMaxOut = 4, kMaxima = 5;
__device__ __forceinline__ u64 order_bits(double v) {
    const u64 b = (u64)__double_as_longlong(v);
    return b >> 63 ? ~b : b | 0x8000000000000000ull;
}
__device__ __forceinline__ double max_value(const u64 *m) {
    const u64 b = *m;
    if (b == 0) return -INFINITY;                      // no number among the values
    return __longlong_as_double((long long)(b >> 63 ? b & 0x7fffffffffffffffull : ~b));
}
// r: this thread's maximum by fmax from -infinity (NaN leaves no mark); blocks of kT threads
constexpr int kT = 256;
__device__ __forceinline__ void block_max(double r, u64 *m) {
    __shared__ double sh[kT / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) r = fmax(r, __shfl_xor(r, o));
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = r;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < kT / 64; ++w) r = fmax(r, sh[w]);
        const u64 b = order_bits(r);
        if (b > __hip_atomic_load(m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(m, b);
    }
}

// Weights f[a] = e_a / sum e, a = 0 .. 2 span, of up to three kernels (blockIdx.x), the sum in
// index order; block 0 clears the maxima.
struct Weights {
    int span[3];
    double *f[3];
};
__global__ __launch_bounds__(kT) void k_weights(Weights w, u64 *__restrict__ M) {
    __shared__ double sum;
    if (blockIdx.x == 0 && threadIdx.x < kMaxima) M[threadIdx.x] = 0;
    const int span = w.span[blockIdx.x], n = 2 * span + 1;
    double *f = w.f[blockIdx.x];
    for (int a = threadIdx.x; a < n; a += kT) {
        const double x = span > 0 ? (2.0 * a - 2.0 * span) / span : 0.0;
        f[a] = exp(-0.5 * x * x);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int a = 0; a < n; ++a) s += f[a];
        sum = s;
    }
    __syncthreads();
    for (int a = threadIdx.x; a < n; a += kT) f[a] /= sum;
}

// A pass over one field: in (or, float data, fin; or the land taper's rows), its kernel, output,
// rows from z0 on, the maximum it leaves (null: none).
struct Pass {
    const double *in;
    const float *fin;
    int taper;                  // > 0: hamming(2 ts)[ts + j] on rows j < ts = taper, 0 below
    double *out;
    const double *f;
    int span, z0;
    u64 *max;
    int absolute;
    const double *mask;         // null, or the output is multiplied by it
};
struct Passes {
    Pass p[3];
};
__device__ __forceinline__ double pass_in(const Pass &p, size_t base, int j) {
    if (p.fin) return (double)p.fin[base + j];
    if (p.taper) {
        const double pi = 3.141592653589793;
        return j < p.taper ? 0.54 - 0.46 * cos(2.0 * pi * (p.taper + j) / (2 * p.taper - 1)) : 0.0;
    }
    return p.in[base + j];
}

// Weights of a wave-uniform tap: scalar loads (an earlier launch wrote them).
typedef const __attribute__((address_space(4))) double *Taps;

// out[i][z0 + j] = sum_b in[i][z0 + j + b - span] f[b] over taps inside rows [z0, nz).  A wave
// takes 64 rows of a column, staged with zeros past its ends (they add nothing), so that the tap
// is the same for all lanes; spans past the stage go through memory.  The land taper is the same
// in every column: one column of it.
constexpr int kStageSpan = 128;
__global__ __launch_bounds__(kT) void k_smooth_z(int nx, int nz, Passes ps) {
    __shared__ double stage[kT / 64][64 + 2 * kStageSpan];
    const Pass &p = ps.p[blockIdx.z];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = blockIdx.x * 64 + lane, i = blockIdx.y * (kT / 64) + wave;
    const int nzs = nz - p.z0, span = p.span;
    const bool col_in = i < (p.taper ? 1 : nx);
    const size_t col = (size_t)i * nz + p.z0;
    const bool staged = span <= kStageSpan;
    if (staged && col_in)
        for (int t = lane; t < 64 + 2 * span; t += 64) {
            const int q = (int)blockIdx.x * 64 + t - span;
            stage[wave][t] = q >= 0 && q < nzs ? pass_in(p, col, q) : 0.0;
        }
    __syncthreads();
    if (!col_in || j >= nzs) return;
    double s = 0.0;
    if (staged) {
        const double *q = &stage[wave][lane];
        const Taps f = (Taps)p.f;
#pragma unroll 8
        for (int b = 0; b <= 2 * span; ++b) s += q[b] * f[b];
    } else {
        for (int b = max(0, span - j); b <= min(2 * span, span + nzs - 1 - j); ++b) s += pass_in(p, col, j + b - span) * p.f[b];
    }
    p.out[col + j] = s;
}

// out[i][z0 + j] = (sum_a in[i + a - span][z0 + j] f[a]) / (wx(i) wz(j)), with wx, wz the
// kernel's sums over the taps inside the x range and inside rows [z0, nz); the maximum of out over
// all rows (rows above z0 as they stand).  A wave takes 64 rows of kCols columns: a value that is
// loaded serves all of them.
constexpr int kCols = 4;
__global__ __launch_bounds__(kT) void k_smooth_x(int nx, int nz, Passes ps) {
    const Pass &p = ps.p[blockIdx.z];
    const int lane = threadIdx.x & 63;
    const int i0 = (blockIdx.y * (kT / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kCols;
    const int row = blockIdx.x * 64 + lane, j = row - p.z0, nzs = nz - p.z0, span = p.span;
    double s[kCols], wx[kCols], wz = 0.0, r = -INFINITY;
#pragma unroll
    for (int m = 0; m < kCols; ++m) s[m] = wx[m] = 0.0;
    // the land taper's one column stands for all
    const double *in = p.in + (row < nz ? row : nz - 1);
    const size_t ld = p.taper ? 0 : nz;
    const Taps f = (Taps)p.f;
    auto add = [&](int q, double v) {                   // any column of the window
#pragma unroll
        for (int m = 0; m < kCols; ++m) {
            const int a = q - (i0 + m) + span;
            if (a < 0 || a > 2 * span) continue;
            s[m] += v * f[a];
            wx[m] += f[a];
        }
    };
    constexpr int U = 8;                                // columns in flight
    int q = max(0, i0 - span);
    const int q1 = min(nx - 1, i0 + kCols - 1 + span);
    const int qa = min(q1 + 1, max(q, i0 + kCols - 1 - span)), qb = min(q1, i0 + span);    // all taps valid
    for (; q < qa; ++q) add(q, in[q * ld]);
    for (; q + U - 1 <= qb; q += U) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = in[(q + u) * ld];
        double g[U + kCols - 1];
#pragma unroll
        for (int u = 0; u < U + kCols - 1; ++u) g[u] = f[q - i0 + span - (kCols - 1) + u];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int m = 0; m < kCols; ++m) {
                s[m] += v[u] * g[u + kCols - 1 - m];
                wx[m] += g[u + kCols - 1 - m];
            }
    }
    for (; q <= q1; ++q) add(q, in[q * ld]);
#pragma unroll 8
    for (int b = 0; b <= 2 * span; ++b) wz += b >= span - j && b <= span + nzs - 1 - j ? f[b] : 0.0;
    if (row < nz) {
#pragma unroll
        for (int m = 0; m < kCols; ++m) {
            if (i0 + m >= nx) continue;
            const size_t k = (size_t)(i0 + m) * nz + row;
            double v = j >= 0 ? s[m] / (wx[m] * wz) : p.out[k];
            if (p.mask) v = v * p.mask[k];
            if (j >= 0 || p.mask) p.out[k] = v;
            r = fmax(r, p.absolute ? fabs(v) : v);
        }
    }
    if (p.max) block_max(r, p.max);
}

// precond = smoothed forw / max + smoothed back / max (into c), with its maximum
__global__ __launch_bounds__(kT) void k_precond_sum(size_t n, const double *__restrict__ a,
                                                    const double *__restrict__ b, u64 *__restrict__ M,
                                                    double *__restrict__ c) {
    const double ma = max_value(M + kMaxForw), mb = max_value(M + kMaxBack);
    double r = -INFINITY;
    for (size_t k = (size_t)blockIdx.x * kT + threadIdx.x; k < n; k += (size_t)gridDim.x * kT) {
        const double v = a[k] / ma + b[k] / mb;
        c[k] = v;
        r = fmax(r, v);
    }
    block_max(r, M + kMaxPre);
}

// g = float(grad * taper) (the reference's in-place product on the float32 gradient;
// taper: marine 0 on rows j < mute, 1 below; land: from its smoothed form lt and maximum m,
// ((-(lt / m) (1 - thred)) + 1)^2; none: no product), then g / max(precond / max precond, 1e-4).
// Without a smoothing pass behind it (last): times the mask, with the maximum of |out|.
__global__ __launch_bounds__(kT) void k_apply(int nz, size_t n, int taper_kind, int mute, double thred, int last,
                                              const float *__restrict__ grad, const double *__restrict__ lt,
                                              const double *__restrict__ c, const double *__restrict__ mask,
                                              u64 *__restrict__ M, double *__restrict__ out) {
    const double mp = max_value(M + kMaxPre), mt = max_value(M + kMaxTaper);
    double r = -INFINITY;
    for (size_t k = (size_t)blockIdx.x * kT + threadIdx.x; k < n; k += (size_t)gridDim.x * kT) {
        float g = grad[k];
        if (taper_kind == 1) {
            g = (float)((double)g * ((int)(k % nz) < mute ? 0.0 : 1.0));
        } else if (taper_kind == 2) {
            double v = lt[k] / mt;
            v = v * (1.0 - thred);
            v = -v + 1.0;
            g = (float)((double)g * (v * v));
        }
        double p = c[k] / mp;
        if (p < 1e-4) p = 1e-4;
        double o = (double)g / p;
        if (last && mask) o = o * mask[k];
        out[k] = o;
        r = fmax(r, fabs(o));
    }
    if (last) block_max(r, M + kMaxOut);
}

// out *= vpmax / max|out|
__global__ __launch_bounds__(kT) void k_scale(size_t n, double vpmax, const u64 *__restrict__ M,
                                              double *__restrict__ out) {
    const double sc = vpmax / max_value(M + kMaxOut);
    for (size_t k = (size_t)blockIdx.x * kT + threadIdx.x; k < n; k += (size_t)gridDim.x * kT) out[k] *= sc;
}

}  // namespace pc
}  // namespace swit
