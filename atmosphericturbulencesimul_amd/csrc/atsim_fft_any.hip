// atsim_fft_any.hip -- transforms and Fresnel steps of any image shape.
//
// An axis of a power-of-two length L >= 16 is transformed directly; any other
// length takes Bluestein's chirp convolution: with c_n = e^{s i pi n^2 / L} and
// d_m = e^{-s i pi m^2 / L}, X_k = c_k sum_n (x_n c_n) d_{k-n}, the convolution
// through transforms of length M >= 2 L - 1 (a power of two).  The whole line --
// chirp, transform, filter, inverse transform, chirp -- stays in registers and
// LDS, so an axis is one pass over the images, and the last axis's forward
// transform, the Fresnel factor and its inverse transform are one pass too
// (the axes commute): a Fresnel step of even sides is three passes.
//
// The rows and columns of an image of odd sides are not aligned to anything
// but 8 bytes: every access is one complex value.
//
// Bound: latency at a few hundred lines, then VALU issue (the transforms are
// 3.4 to 4 times as long as the lines).  4 images of 600 x 450 through a Fresnel
// step: 70 us of kernels (rows 18 each, columns 32) and 89 us a call, where
// padded copies of the lines, transforms and a product per axis took 480 us and
// a call 1 900 us, the chirp's filter being made on the host each time.
#include <hip/hip_runtime.h>

#include "atsim_fft.hpp"
#include "atsim_launch.hpp"

namespace atsim {

enum { LINE_FWD = 0, LINE_BWD = 1, LINE_BLUE = 2 };

// one transform of a line's registers (layout of the forward plan's first
// stage before and after): direct, or Bluestein with the chirp of the plan;
// values past L are zero before and meaningless after
template <int M, int MODE, int C>
__device__ __forceinline__ void line_transform(float2* v, float2* lds, int t, int c, int L,
                                               const float2* __restrict__ chirp, const float2* __restrict__ filt,
                                               const float2* __restrict__ tw) {
    using P = Plan<M>;
    constexpr int RI = P::first(-1), RL = P::last(-1);
    if constexpr (MODE == LINE_BLUE) {
        // indices recomputed for each step, not kept live over the others
        t = opaque(t);
        c = opaque(c);
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int n = reg_index<M, RI>(t, q);
            const float2 x = cmul(v[q], chirp[min(n, L - 1)]);
            v[q] = n < L ? x : make_float2(0.f, 0.f);
        }
        fft_regs<M, -1, C, true>(v, lds, t, c, tw);
        t = opaque(t);
        c = opaque(c);
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = cmul(v[q], filt[reg_index<M, RL>(t, q)]);
        fft_regs<M, +1, C, true>(v, lds, t, c, tw);
        t = opaque(t);
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = cmul(v[q], chirp[min(reg_index<M, RI>(t, q), L - 1)]);
    } else {
        fft_regs<M, MODE == LINE_FWD ? -1 : +1, C, true>(v, lds, t, c, tw);
    }
}

template <int M>
struct AnyRow {
    static constexpr int T = M / 16;
    static constexpr int ROWS = 256 / T > 0 ? 256 / T : 1;
};

// lines of length L (<= M; = M when direct) that are contiguous rows
template <int M, int MODE>
__global__ void __launch_bounds__(AnyRow<M>::ROWS * (M / 16))
k_any_row(const float2* in, float2* out, long nrows, int L, const float2* __restrict__ chirp,
          const float2* __restrict__ filt, const float2* __restrict__ tw) {
    using P = Plan<M>;
    constexpr int T = P::T, ROWS = AnyRow<M>::ROWS;
    constexpr int RI = MODE == LINE_BWD ? P::first(+1) : P::first(-1);
    constexpr int RO = MODE == LINE_FWD ? P::last(-1) : MODE == LINE_BWD ? P::last(+1) : P::last(+1);
    __shared__ float2 lds[ROWS * P::LDS];
    const int lr = threadIdx.x / T, t = threadIdx.x - lr * T;
    const long row = (long)blockIdx.x * ROWS + lr;
    const float2* src = in + min(row, nrows - 1) * L;
    float2 v[16];
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = src[min(reg_index<M, RI>(t, q), L - 1)];
    line_transform<M, MODE, 1>(v, lds + lr * P::LDS, t, 0, L, chirp, filt, tw);
    if (row >= nrows) return;
    float2* dst = out + row * L;
    const int t2 = opaque(t);
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int n = reg_index<M, RO>(t2, q);
        if (n < L) dst[n] = v[q];
    }
}

// lines along y: C adjacent columns of an n0-wide image per workgroup.
// FACTOR: forward transform, the Fresnel factor hx[column] hy[n] (FP64 values,
// products in FP64), inverse transform (MODE LINE_BLUE with the two signs'
// plans, or direct); otherwise one transform.
template <int M, int MODE, int C, bool FACTOR>
__global__ void __launch_bounds__(C * (M / 16))
k_any_col(float2* __restrict__ data, int n0, int L, int ntile, const float2* __restrict__ chirp,
          const float2* __restrict__ filt, const float2* __restrict__ chirp2, const float2* __restrict__ filt2,
          const double2* __restrict__ hx, const double2* __restrict__ hy, const float2* __restrict__ tw) {
    using P = Plan<M>;
    constexpr bool FWD_IN = FACTOR || MODE != LINE_BWD;
    constexpr int RI = FWD_IN ? P::first(-1) : P::first(+1);
    constexpr int RM = (FACTOR && MODE != LINE_BLUE) ? P::last(-1) : P::first(-1);  // layout between the two
    constexpr int RO = (FACTOR || MODE != LINE_FWD) ? P::last(+1) : P::last(-1);
    __shared__ float2 lds[C * P::LDSC];
    const int c = threadIdx.x % C, t = threadIdx.x / C;
    const int img = blockIdx.x / ntile, col = (blockIdx.x - img * ntile) * C + c;
    float2* base = data + (size_t)img * n0 * L + min(col, n0 - 1);
    float2 v[16];
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = base[(size_t)min(reg_index<M, RI>(t, q), L - 1) * n0];
    if constexpr (FACTOR) {
        line_transform<M, MODE == LINE_BLUE ? LINE_BLUE : LINE_FWD, C>(v, lds, t, c, L, chirp, filt, tw);
        const double2 fx = hx[min(col, n0 - 1)];
        const int t1 = opaque(t);
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const double2 fy = hy[min(reg_index<M, RM>(t1, q), L - 1)];
            const double fr = fx.x * fy.x - fx.y * fy.y, fi = fx.x * fy.y + fx.y * fy.x;
            v[q] = make_float2((float)(v[q].x * fr - v[q].y * fi), (float)(v[q].x * fi + v[q].y * fr));
        }
        line_transform<M, MODE == LINE_BLUE ? LINE_BLUE : LINE_BWD, C>(v, lds, t, c, L, chirp2, filt2, tw);
    } else {
        line_transform<M, MODE, C>(v, lds, t, c, L, chirp, filt, tw);
    }
    if (col >= n0) return;
    const int t2 = opaque(t);
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int n = reg_index<M, RO>(t2, q);
        if (n < L) base[(size_t)n * n0] = v[q];
    }
}

// hx[k] = e^{-i coeff kt^2}, hy[k] = the same over the other axis / (n0 n1),
// kt the signed frequency (the reference's permut pair on even sides)
__global__ void k_any_factor(double2* __restrict__ hx, double2* __restrict__ hy, int n0, int n1, double coeff) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n0 + n1) return;
    const int n = e < n0 ? n0 : n1, k = e < n0 ? e : e - n0;
    const double kt = k < n / 2 ? k : k - n, s = e < n0 ? 1.0 : 1.0 / ((double)n0 * (double)n1);
    double sn, cs;
    sincos(-coeff * kt * kt, &sn, &cs);
    (e < n0 ? hx : hy)[k] = make_double2(cs * s, sn * s);
}

// The reference's permut (fft.c:570-792) moves to element (j, i) what was at
// permut_source(j, i): its swap loops over xh = n0 / 2 and yh = n1 / 2, the
// last column of an odd width staying where it is.
__device__ __forceinline__ long permut_source(int n0, int n1, int j, int i) {
    const int xh = n0 / 2, yh = n1 / 2;
    int sj = j, si = i;
    if (i < xh) {
        const int s = j - yh;
        if (j < yh) {
            sj = j + yh;
            si = i + xh;
        } else if (s < yh || yh == 0) {
            sj = s;
            si = i + xh;
        } else {
            sj = 0;  // the last row of an odd height: swapped with a row already swapped
        }
    } else if (i < 2 * xh) {
        if (j <= n1 - 1 - yh) {
            sj = j + yh;
            si = i - xh;
        } else if (j < 2 * yh) {
            sj = j - yh;
            si = i - xh;
        }
    }
    return (long)sj * n0 + si;
}

__global__ void k_permut_any(const float2* __restrict__ in, float2* __restrict__ out, int n0, int n1, long nbatch) {
    const long n = (long)n0 * n1, total = n * nbatch;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
        const long b = e / n;
        const int p = (int)(e - b * n), j = p / n0;
        out[e] = in[b * n + permut_source(n0, n1, j, p - j * n0)];
    }
}

// The Fresnel factor of Fresnel_propagate_wavefront (WFpropagate.c:68-152) on
// the spectrum of an image with an odd side: permut, times e^{-i coeff ((ii -
// n0/2)^2 + (jj - n1/2)^2)} / (n0 n1) at the permuted position (ii, jj), permut:
// out[p] = in[sigma(sigma(p))] h(sigma(p)).  Angle and factor in FP64.
__global__ void k_fresnel_odd(const float2* __restrict__ in, float2* __restrict__ out, int n0, int n1, long nbatch,
                              double coeff) {
    const long n = (long)n0 * n1, total = n * nbatch;
    const double inv = 1.0 / ((double)n0 * (double)n1);
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
        const long b = e / n;
        const int p = (int)(e - b * n), j = p / n0;
        const long q = permut_source(n0, n1, j, p - j * n0);
        const int jq = (int)(q / n0), iq = (int)(q - (long)jq * n0);
        const long src = permut_source(n0, n1, jq, iq);
        const long di = iq - n0 / 2, dj = jq - n1 / 2;
        double sn, cs;
        sincos(-coeff * (double)(di * di + dj * dj), &sn, &cs);
        const float2 v = in[b * n + src];
        const double re = (double)v.x * inv, im = (double)v.y * inv;
        out[e] = make_float2((float)(re * cs - im * sn), (float)(re * sn + im * cs));
    }
}

static unsigned grid_for(long total) {
    long g = (total + 255) / 256;
    return (unsigned)(g < 1 ? 1 : (g > 65536 ? 65536 : g));
}
hipError_t launch_permut_any(const float2* in, float2* out, long n0, long n1, long nbatch, hipStream_t st) {
    k_permut_any<<<grid_for(n0 * n1 * nbatch), 256, 0, st>>>(in, out, (int)n0, (int)n1, nbatch);
    return hipGetLastError();
}
hipError_t launch_fresnel_odd(const float2* in, float2* out, long n0, long n1, long nbatch, double coeff,
                              hipStream_t st) {
    k_fresnel_odd<<<grid_for(n0 * n1 * nbatch), 256, 0, st>>>(in, out, (int)n0, (int)n1, nbatch, coeff);
    return hipGetLastError();
}
hipError_t launch_any_factor(double2* hx, double2* hy, long n0, long n1, double coeff, hipStream_t st) {
    k_any_factor<<<(unsigned)((n0 + n1 + 255) / 256), 256, 0, st>>>(hx, hy, (int)n0, (int)n1, coeff);
    return hipGetLastError();
}

template <int M>
static hipError_t any_row(const LinePlan& p, int sign, const float2* in, float2* out, long nrows, hipStream_t st) {
    constexpr int ROWS = AnyRow<M>::ROWS;
    const unsigned grid = (unsigned)((nrows + ROWS - 1) / ROWS);
    const int block = ROWS * (M / 16);
    if (p.chirp) k_any_row<M, LINE_BLUE><<<grid, block, 0, st>>>(in, out, nrows, p.L, p.chirp, p.filt, p.tw);
    else if (sign < 0) k_any_row<M, LINE_FWD><<<grid, block, 0, st>>>(in, out, nrows, p.L, nullptr, nullptr, p.tw);
    else k_any_row<M, LINE_BWD><<<grid, block, 0, st>>>(in, out, nrows, p.L, nullptr, nullptr, p.tw);
    return hipGetLastError();
}

template <int M, int C>
static hipError_t any_col_c(const LinePlan& p, const LinePlan* back, int sign, float2* data, long n0, long nbatch,
                            const double2* hx, const double2* hy, hipStream_t st) {
    const long ntile = (n0 + C - 1) / C;
    if (ntile * nbatch > 0x7fffffffL) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)(ntile * nbatch);
    const int block = C * (M / 16);
#define ANY_COL(MODE, FACTOR)                                                                                \
    k_any_col<M, MODE, C, FACTOR><<<grid, block, 0, st>>>(data, (int)n0, p.L, (int)ntile, p.chirp, p.filt,   \
                                                          back ? back->chirp : nullptr,                      \
                                                          back ? back->filt : nullptr, hx, hy, p.tw)
    if (back && p.chirp) ANY_COL(LINE_BLUE, true);
    else if (back) ANY_COL(LINE_FWD, true);
    else if (p.chirp) ANY_COL(LINE_BLUE, false);
    else if (sign < 0) ANY_COL(LINE_FWD, false);
    else ANY_COL(LINE_BWD, false);
#undef ANY_COL
    return hipGetLastError();
}
template <int M>
static hipError_t any_col(const LinePlan& p, const LinePlan* back, int sign, float2* data, long n0, long nbatch,
                          const double2* hx, const double2* hy, hipStream_t st) {
    // 128-byte row segments (16 columns) as far as the LDS and 1 024 threads go;
    // 4 columns where that leaves CUs without a workgroup (the 256 CUs take one
    // workgroup of 16 columns each, four of 4)
    constexpr int CW = M <= 1024 ? 16 : M == 2048 ? 8 : M == 4096 ? 4 : 2;
    if constexpr (CW > 4) {
        if ((n0 + CW - 1) / CW * nbatch < 256) return any_col_c<M, 4>(p, back, sign, data, n0, nbatch, hx, hy, st);
    }
    return any_col_c<M, CW>(p, back, sign, data, n0, nbatch, hx, hy, st);
}

#define ATSIM_FOR_EACH_M(X) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096) X(8192)

hipError_t launch_any_row(const LinePlan& p, int sign, const float2* in, float2* out, long nrows, hipStream_t st) {
    switch (p.M) {
#define X(MM) \
    case MM: return any_row<MM>(p, sign, in, out, nrows, st);
        ATSIM_FOR_EACH_M(X)
#undef X
        default: return hipErrorInvalidValue;
    }
}
hipError_t launch_any_col(const LinePlan& p, const LinePlan* back, int sign, float2* data, long n0, long nbatch,
                          const double2* hx, const double2* hy, hipStream_t st) {
    switch (p.M) {
#define X(MM) \
    case MM: return any_col<MM>(p, back, sign, data, n0, nbatch, hx, hy, st);
        ATSIM_FOR_EACH_M(X)
#undef X
        default: return hipErrorInvalidValue;
    }
}

}  // namespace atsim
