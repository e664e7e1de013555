// rmedia.hip -- random-media synthesis on the device, the generator of
// src/shared/m_rmedia.f90:40-173 (rmedia__3dgen_ani):
//   uniform noise -> forward FFT -> whitening b/|b| -> filter by
//   sqrt(psdf(k) N dV) -> b(0) = 0 -> inverse FFT -> mean removed, rms scaled
//   to epsil.
// Noise comes from a counter-based generator (one 64-bit mix per cell), so a
// realisation depends on the seed and the grid only, not on launch shapes.
// Transforms are double-precision and of any size (the reference's radix-2
// FFT, m_rfft.f90:46, needs powers of two); sums are deterministic, per block
// and then over the blocks.  The field is written as float.  Grids whose lines fit in LDS
// are transformed by the kernels here; the others by hipFFT.
#include <hipfft/hipfft.h>

#include <cmath>
#include <cstdio>
#include <cstdarg>
#include <cstring>
#include <vector>

#include "swpc_internal.h"

namespace {

thread_local char g_err[512] = "";

int rfail(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}

// splitmix64 finaliser: a bijective mix of a 64-bit counter
__device__ static inline unsigned long long mix64(unsigned long long z)
{
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// cell q's noise, uniform in [0, 1)
__device__ static inline double noise(unsigned long long key, long long q)
{
    return (double)(mix64(key ^ (unsigned long long)q) >> 11) * 0x1.0p-53;
}

__global__ void k_noise(double *r, long long n, unsigned long long seed)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const unsigned long long key = mix64(seed);
    for (long long q = t; q < n; q += (long long)gridDim.x * blockDim.x) r[q] = noise(key, q);
}

struct FilterArgs {
    double2 *b;
    int n1h, n2, n3;           // half spectrum n1/2+1 along the fastest axis
    double k1, k2, k3;         // 2 pi / (n d) per axis
    int n1, n2f, n3f;          // full sizes for the negative wavenumbers
    double a1, a2, a3;
    int ptype;
    double coef, expo, scale;  // psdf = coef * shape(q); scale = N dV
};

// wavenumber of index i of an n-point axis (m_fk.f90 x2k3d)
__device__ static inline double wnum(int i, int n, double k0)
{
    return (i <= n / 2 ? i : i - n) * k0;
}

// whitening and filtering of one spectral value (m_rmedia.f90:107-140)
__device__ static inline double2 filtered(const FilterArgs &a, int i1, int i2, int i3, double2 v)
{
    if (i1 == 0 && i2 == 0 && i3 == 0) return make_double2(0.0, 0.0);  // DC
    const double m1 = wnum(i1, a.n1, a.k1) * a.a1;
    const double m2 = wnum(i2, a.n2f, a.k2) * a.a2;
    const double m3 = wnum(i3, a.n3f, a.k3) * a.a3;
    const double q2 = m1 * m1 + m2 * m2 + m3 * m3;
    double psdf;
    if (a.ptype == 1) psdf = a.coef * exp(-q2 * 0.25);
    else if (a.ptype == 2) psdf = a.coef / ((1.0 + q2) * (1.0 + q2));
    else psdf = a.coef * pow(1.0 + q2, -a.expo);
    const double mag = sqrt(v.x * v.x + v.y * v.y);
    const double f = mag > 0.0 ? sqrt(psdf * a.scale) / mag : 0.0;
    return make_double2(v.x * f, v.y * f);
}

// the half spectrum filtered in place
__global__ void k_filter(FilterArgs a)
{
    const long long total = (long long)a.n1h * a.n2 * a.n3;
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < total;
         q += (long long)gridDim.x * blockDim.x) {
        const int i1 = (int)(q % a.n1h);
        const long long t = q / a.n1h;
        const int i2 = (int)(t % a.n2);
        const int i3 = (int)(t / a.n2);
        a.b[q] = filtered(a, i1, i2, i3, a.b[q]);
    }
}

// per-block partial sums of x (what = 0) or (x - mean)^2 (what = 1)
__global__ void __launch_bounds__(256) k_partial(const double *x, long long n, double mean, int what, double *part)
{
    __shared__ double s[256];
    double acc = 0.0;
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < n; q += (long long)gridDim.x * 256) {
        const double v = x[q] - mean;
        acc += what ? v * v : x[q];
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// one block adds the partials in a fixed order
__global__ void __launch_bounds__(256) k_total(const double *part, int np, double *out)
{
    __shared__ double s[256];
    double acc = 0.0;
    for (int q = threadIdx.x; q < np; q += 256) acc += part[q];
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = s[0];
}

__global__ void k_finish(const double *x, long long n, const double *stats, double epsil, float *out)
{
    const double mean = stats[0], rms = stats[1];
    const double f = rms > 0.0 ? epsil / rms : 0.0;
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long long)gridDim.x * blockDim.x)
        out[q] = (float)((x[q] - mean) * f);
}

// ---------------------------------------------------------------------------
// transforms of whole lines in LDS
//
// A call needs one forward and one inverse transform of one grid, so a
// library plan is made, used twice and dropped: of 51 ms for 198 x 262 x 262
// cells the plans (and the loading of their code) took about 40, the kernels
// 4.  These kernels need no plan: the factors travel as arguments and a block
// makes its own table of roots of unity.  The noise is made where the first
// axis is transformed, and the last axis is transformed, filtered and
// transformed back while its lines are in LDS, so the spectrum crosses memory
// four times (written, and three times read and written) and the real field
// takes its place.  Bound by LDS: a prime factor p costs (p + 1) / 4 reads of
// three 16-byte words per value (131 in a line of 262 cells: half the time).
// ---------------------------------------------------------------------------
struct Factors {
    int n, nf, p[16];   // line length and its factors: fours, at most one two, odd primes
};

// nl lines of f.n points in x (y is as large): point i of line c is at
// i * si + c * sc; w: the f.n roots exp(-2 pi i j / n).  dir = 1 forward, -1
// inverse, both unnormalised.  Every pass takes one factor p: groups g of
// points g + j n/p become points g + s r (p - 1) + s k, r = g / s, times
// w^(r k s), s the product of the factors before, so the result is in order
// after the last.  Called and left by the whole block; returns where the
// result is (x or y), after a barrier.
template <bool LINES_FAST>
__device__ double2 *fft_lines(const Factors &f, double2 *x, double2 *y, const double2 *w, int nl, int si, int sc,
                              double dir)
{
    const int n = f.n;
    int s = 1;
    __syncthreads();
    for (int st = 0; st < f.nf; ++st) {
        const int p = f.p[st], m = n / p;
        const int h = p > 4 || p == 3 ? (p + 1) / 2 : 1;   // items of a group: outputs 0 and (k, p - k), or all
        for (int t = threadIdx.x; t < nl * m * h; t += blockDim.x) {
            int c, g, k;
            if (LINES_FAST) {
                const int u = t / nl;
                c = t - u * nl;
                k = u / m;
                g = u - k * m;
            } else {
                const int u = t / m;
                g = t - u * m;
                k = u / nl;
                c = u - k * nl;
            }
            const int r = g / s, o = g + s * r * (p - 1);
            const double2 *xi = x + (long)c * sc + (long)g * si;
            double2 *yo = y + (long)c * sc + (long)o * si;
            const int dj = m * si, dk = s * si;
            // output kk times its root
            auto put = [&](int kk, double re, double im) {
                const double2 q = w[r * kk * s];
                const double qy = dir * q.y;
                yo[kk * dk] = make_double2(fma(re, q.x, -(im * qy)), fma(re, qy, im * q.x));
            };
            if (p == 4) {
                const double2 a0 = xi[0], a1 = xi[dj], a2 = xi[2 * dj], a3 = xi[3 * dj];
                const double s0x = a0.x + a2.x, s0y = a0.y + a2.y, d0x = a0.x - a2.x, d0y = a0.y - a2.y;
                const double s1x = a1.x + a3.x, s1y = a1.y + a3.y;
                const double d1x = dir * (a1.y - a3.y), d1y = dir * (a3.x - a1.x);   // -i (a1 - a3)
                put(0, s0x + s1x, s0y + s1y);
                put(1, d0x + d1x, d0y + d1y);
                put(2, s0x - s1x, s0y - s1y);
                put(3, d0x - d1x, d0y - d1y);
            } else if (p == 2) {
                const double2 a0 = xi[0], a1 = xi[dj];
                put(0, a0.x + a1.x, a0.y + a1.y);
                put(1, a0.x - a1.x, a0.y - a1.y);
            } else if (k == 0) {
                double re = xi[0].x, im = xi[0].y;
                for (int j = 1; j < p; ++j) {
                    re += xi[j * dj].x;
                    im += xi[j * dj].y;
                }
                put(0, re, im);
            } else {
                // points j and p - j carry conjugate roots: their sum goes with
                // the cosine, their difference with the sine, for outputs k
                // and p - k alike
                double px = xi[0].x, py = xi[0].y, qx = 0.0, qy = 0.0;
                const int step = k * m;
                int idx = 0;
#pragma unroll 4
                for (int j = 1; j <= (p - 1) / 2; ++j) {
                    idx += step;
                    idx -= idx >= n ? n : 0;
                    const double2 u = xi[j * dj], v = xi[(p - j) * dj], q = w[idx];
                    px = fma(u.x + v.x, q.x, px);
                    py = fma(u.y + v.y, q.x, py);
                    qx = fma(u.x - v.x, q.y, qx);
                    qy = fma(u.y - v.y, q.y, qy);
                }
                qx *= dir;
                qy *= dir;
                put(k, px - qy, py + qx);
                put(p - k, px + qy, py - qx);
            }
        }
        s *= p;
        double2 *z = x;
        x = y;
        y = z;
        __syncthreads();
    }
    return x;
}

__device__ static inline void roots(const Factors &f, double2 *w)
{
    for (int j = threadIdx.x; j < f.n; j += blockDim.x) {
        double sn, cs;
        sincospi(-2.0 * (double)j / (double)f.n, &sn, &cs);
        w[j] = make_double2(cs, sn);
    }
}

extern __shared__ double2 lds[];

// the first axis: np pairs of rows per block, a pair as the real and the
// imaginary part of one line.  Forward: rows of noise to their half spectra.
__global__ void __launch_bounds__(1024) k_rows_fwd(Factors f, double2 *c, int pitch, long long rows, int np,
                                                   unsigned long long seed)
{
    const int n = f.n, sc = n + 1;
    double2 *w = lds, *x = lds + n, *y = x + np * sc;
    const long long row0 = (long long)blockIdx.x * 2 * np;
    const unsigned long long key = mix64(seed);
    roots(f, w);
    for (int t = threadIdx.x; t < np * n; t += blockDim.x) {
        const int l = t / n, i = t - l * n;
        const long long row = row0 + 2 * l;
        x[l * sc + i] = make_double2(row < rows ? noise(key, row * n + i) : 0.0,
                                     row + 1 < rows ? noise(key, (row + 1) * n + i) : 0.0);
    }
    const double2 *z = fft_lines<false>(f, x, y, w, np, 1, sc, 1.0);
    const int nh = n / 2 + 1;
    for (int t = threadIdx.x; t < 2 * np * nh; t += blockDim.x) {
        const int l2 = t / nh, k = t - l2 * nh;
        const long long row = row0 + l2;
        if (row >= rows) break;
        const double2 a = z[(l2 >> 1) * sc + k], b = z[(l2 >> 1) * sc + (k ? n - k : 0)];
        c[row * pitch + k] = l2 & 1 ? make_double2(0.5 * (a.y + b.y), 0.5 * (b.x - a.x))
                                    : make_double2(0.5 * (a.x + b.x), 0.5 * (a.y - b.y));
    }
}

// Inverse: half spectra to real rows in their place (2 * pitch doubles a
// row), with the block's sum and sum of squares.
__global__ void __launch_bounds__(1024) k_rows_inv(Factors f, double2 *c, int pitch, long long rows, int np,
                                                   double *part)
{
    const int n = f.n, sc = n + 1, nh = n / 2 + 1;
    double2 *w = lds, *x = lds + n, *y = x + np * sc;
    const long long row0 = (long long)blockIdx.x * 2 * np;
    roots(f, w);
    for (int t = threadIdx.x; t < np * nh; t += blockDim.x) {
        const int l = t / nh, k = t - l * nh;
        const long long row = row0 + 2 * l;
        double2 a = make_double2(0.0, 0.0), b = a;
        if (row < rows) a = c[row * pitch + k];
        if (row + 1 < rows) b = c[(row + 1) * pitch + k];
        if (k == 0 || 2 * k == n) {   // real by symmetry
            x[l * sc + k] = make_double2(a.x, b.x);
        } else {
            x[l * sc + k] = make_double2(a.x - b.y, a.y + b.x);
            x[l * sc + n - k] = make_double2(a.x + b.y, b.x - a.y);
        }
    }
    const double2 *z = fft_lines<false>(f, x, y, w, np, 1, sc, -1.0);
    double sum = 0.0, sq = 0.0;
    for (int t = threadIdx.x; t < 2 * np * n; t += blockDim.x) {
        const int l2 = t / n, i = t - l2 * n;
        const long long row = row0 + l2;
        if (row >= rows) break;
        const double2 a = z[(l2 >> 1) * sc + i];
        const double v = l2 & 1 ? a.y : a.x;
        ((double *)(c + row * pitch))[i] = v;
        sum += v;
        sq += v * v;
    }
    for (int q = 32; q > 0; q >>= 1) {
        sum += __shfl_down(sum, q);
        sq += __shfl_down(sq, q);
    }
    __shared__ double2 s[16];
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = make_double2(sum, sq);
    __syncthreads();
    if (threadIdx.x == 0) {
        for (unsigned q = 1; q < blockDim.x >> 6; ++q) {
            s[0].x += s[q].x;
            s[0].y += s[q].y;
        }
        part[blockIdx.x] = s[0].x;
        part[gridDim.x + blockIdx.x] = s[0].y;
    }
}

// the other axes, in place: nl neighbouring columns (128 bytes where nl = 8)
// per block, points at a distance of step values; tiles of columns within each
// of the plane's rows, outer of them at a distance of ostep.  FILTER: the
// last axis, forward, filtered and back.
template <bool FILTER>
__global__ void __launch_bounds__(1024) k_cols(Factors f, double2 *c, int ncol, int ntile, long long step,
                                               long long ostep, int nl, double dir, FilterArgs fa)
{
    const int n = f.n;
    double2 *w = lds, *x = lds + n, *y = x + n * nl;
    const int tile = blockIdx.x % ntile, outer = blockIdx.x / ntile;
    const int c0 = tile * nl;
    const int have = min(nl, ncol - c0);
    double2 *p = c + outer * ostep + c0;
    roots(f, w);
    for (int t = threadIdx.x; t < n * nl; t += blockDim.x) {
        const int i = t / nl, l = t - i * nl;
        x[t] = l < have ? p[i * step + l] : make_double2(0.0, 0.0);
    }
    double2 *z = fft_lines<true>(f, x, y, w, nl, nl, 1, dir);
    if (FILTER) {
        for (int t = threadIdx.x; t < n * nl; t += blockDim.x) {
            const int i = t / nl, l = t - i * nl;
            z[t] = filtered(fa, c0 + l, outer, i, z[t]);
        }
        z = fft_lines<true>(f, z, z == x ? y : x, w, nl, nl, 1, -1.0);
    }
    for (int t = threadIdx.x; t < n * nl; t += blockDim.x) {
        const int i = t / nl, l = t - i * nl;
        if (l < have) p[i * step + l] = z[t];
    }
}

// mean and rms from the blocks' sums; DC is zero, so the mean is rounding
// only and takes nothing from the squares
__global__ void __launch_bounds__(256) k_stats(const double *part, int np, long long n, double *stats)
{
    __shared__ double2 s[256];
    double2 acc = make_double2(0.0, 0.0);
    for (int q = threadIdx.x; q < np; q += 256) {
        acc.x += part[q];
        acc.y += part[np + q];
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int q = 128; q > 0; q >>= 1) {
        if (threadIdx.x < q) {
            s[threadIdx.x].x += s[threadIdx.x + q].x;
            s[threadIdx.x].y += s[threadIdx.x + q].y;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double mean = s[0].x / (double)n;
        stats[0] = mean;
        stats[1] = sqrt(fmax(s[0].y / (double)n - mean * mean, 0.0));
    }
}

// rows of n1 doubles, 2 * pitch apart, scaled into the float field
__global__ void __launch_bounds__(256) k_scale(const double2 *c, int pitch, long long rows, int n1, const double *stats,
                                               double epsil, float *out)
{
    const double mean = stats[0], rms = stats[1];
    const double f = rms > 0.0 ? epsil / rms : 0.0;
    const long long row0 = (long long)blockIdx.x * 16;
    const int have = (int)(rows - row0 < 16 ? rows - row0 : 16);
    for (int t = threadIdx.x; t < have * n1; t += 256) {
        const int l = t / n1, i = t - l * n1;
        out[row0 * n1 + t] = (float)((((const double *)(c + (row0 + l) * pitch))[i] - mean) * f);
    }
}

struct Dev {
    void *p = nullptr;
    ~Dev() { if (p) (void)hipFree(p); }
};

}  // namespace

extern "C" const char *swpc_rmedia_last_error(void) { return g_err; }

#define RCHK(x)                                                                           \
    do {                                                                                  \
        hipError_t e_ = (x);                                                              \
        if (e_ != hipSuccess) return rfail(SWPC_EHIP, "%s: %s", #x, hipGetErrorString(e_)); \
    } while (0)
#define FCHK(x)                                                                 \
    do {                                                                        \
        hipfftResult r_ = (x);                                                  \
        if (r_ != HIPFFT_SUCCESS) return rfail(SWPC_EHIP, "%s: hipFFT error %d", #x, (int)r_); \
    } while (0)

namespace {

// how a block takes lines of one length: nl of them (8 columns are a 128-byte
// line of memory; fewer where they do not fit, 0 where not even one does), in
// threads that leave the fewest idle in the passes' last rounds
struct LinePlan {
    Factors f;
    int nl, threads;
    size_t lds;
};

LinePlan plan_lines(int n, size_t lds_max)
{
    LinePlan q;
    Factors &f = q.f;
    f.n = n;
    f.nf = 0;
    int m = n;
    q.nl = q.threads = 0;
    q.lds = 0;
    auto bytes = [&](int nl) { return ((size_t)n + 2 * (size_t)nl * (n + 1)) * sizeof(double2); };
    if (bytes(1) > lds_max) return q;
    while (m % 4 == 0) { f.p[f.nf++] = 4; m /= 4; }
    if (m % 2 == 0) { f.p[f.nf++] = 2; m /= 2; }
    for (int p = 3; m > 1; p += 2) {
        if (p * p > m) p = m;
        while (m % p == 0) { f.p[f.nf++] = p; m /= p; }
    }
    q.nl = 8;
    while (bytes(q.nl) > lds_max) q.nl /= 2;
    q.lds = bytes(q.nl);
    long best = 0;
    for (int t = 1024; t >= 256; t -= 64) {
        long cost = 0;
        for (int s = 0; s < f.nf; ++s) {
            const int p = f.p[s];
            const long items = (long)q.nl * (n / p) * (p > 4 || p == 3 ? (p + 1) / 2 : 1);
            cost += (items + t - 1) / t * t * (p + 4);
        }
        if (!q.threads || cost < best) { best = cost; q.threads = t; }
    }
    return q;
}

}  // namespace

extern "C" int swpc_rmedia_3d(int device, int ptype, int n1, int n2, int n3, float d1, float d2, float d3, float a1,
                              float a2, float a3, float epsil, float kappa, uint64_t seed, float *out)
{
    g_err[0] = 0;
    if (!out || n1 < 2 || n2 < 2 || n3 < 2 || ptype < 1 || ptype > 3 || !(d1 > 0) || !(d2 > 0) || !(d3 > 0) ||
        !(a1 > 0) || !(a2 > 0) || !(a3 > 0) || !(epsil >= 0) || (ptype == 3 && !(kappa > 0)))
        return rfail(SWPC_EINVAL, "swpc_rmedia_3d: bad arguments");
    RCHK(hipSetDevice(device));
    const long long n = (long long)n1 * n2 * n3;
    // out in device memory of this GPU: the field is written there directly
    hipPointerAttribute_t at;
    const bool out_dev = hipPointerGetAttributes(&at, out) == hipSuccess && at.type == hipMemoryTypeDevice &&
                         at.device == device;
    (void)hipGetLastError();
    const int n1h = n1 / 2 + 1;
    const long long nc = (long long)n1h * n2 * n3;
    // constants of the PSDFs of m_rmedia.f90:682-732 (they cancel in the final
    // scaling but are kept)
    FilterArgs fa;
    fa.n1h = n1h; fa.n2 = n2; fa.n3 = n3;
    fa.n1 = n1; fa.n2f = n2; fa.n3f = n3;
    const double PI = 3.14159265358979323846;
    fa.k1 = 2 * PI / ((double)n1 * d1);
    fa.k2 = 2 * PI / ((double)n2 * d2);
    fa.k3 = 2 * PI / ((double)n3 * d3);
    fa.a1 = a1; fa.a2 = a2; fa.a3 = a3;
    fa.ptype = ptype;
    const double e2a = (double)epsil * epsil * a1 * a2 * a3;
    if (ptype == 1) fa.coef = e2a * pow(PI, 1.5);
    else if (ptype == 2) fa.coef = 8 * e2a * PI;
    else fa.coef = 8 * pow(PI, 1.5) * e2a * std::tgamma((double)kappa + 1.5) / std::tgamma((double)kappa);
    fa.expo = (double)kappa + 1.5;
    fa.scale = (double)n * d1 * d2 * d3;
    int lds_max = 0;
    RCHK(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, device));
    const size_t lds_use = (size_t)lds_max - 1024;   // k_rows_inv's own
    const LinePlan ax[3] = {plan_lines(n1, lds_use), plan_lines(n2, lds_use), plan_lines(n3, lds_use)};
    // Wherever the lines fit (up to some 3390 points) their kernels are the
    // faster ones, also at primes: 198 x 262 x 262 cells 1.9 ms against 38.6,
    // 512^3 6.7 against 18.0, 509^3 30 against 67, 1031 x 1031 x 64 25 against
    // 62, 454 x 774 x 774 36 against 77; and the library takes another 0.6 to 3
    // s for the first grid of a size in a process.
    const bool lines = ax[0].nl && ax[1].nl && ax[2].nl;
    hipStream_t s;
    RCHK(hipStreamCreate(&s));
    struct StreamGuard { hipStream_t s; ~StreamGuard() { (void)hipStreamDestroy(s); } } sg{s};
    Dev dr, dc, dpart, dstats, dout;
    if (lines) {
        const int pitch = (n1h + 7) & ~7;   // rows start on a 128-byte line
        const long long rows = (long long)n2 * n3;
        const unsigned rowblk = (unsigned)((rows + 2 * ax[0].nl - 1) / (2 * ax[0].nl));
        RCHK(hipMalloc(&dc.p, (size_t)(rows * pitch) * sizeof(double2)));
        RCHK(hipMalloc(&dpart.p, (2 * (size_t)rowblk + 2) * sizeof(double)));
        if (!out_dev) RCHK(hipMalloc(&dout.p, (size_t)n * sizeof(float)));
        double2 *c = (double2 *)dc.p;
        double *part = (double *)dpart.p, *stats = part + 2 * (size_t)rowblk;
        const void *const kern[4] = {(const void *)k_rows_fwd, (const void *)k_rows_inv, (const void *)k_cols<false>,
                                     (const void *)k_cols<true>};
        for (const void *k : kern) RCHK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_use));
        const int nt2 = (n1h + ax[1].nl - 1) / ax[1].nl, nt3 = (n1h + ax[2].nl - 1) / ax[2].nl;
        const dim3 b1(ax[0].threads), b2(ax[1].threads), b3(ax[2].threads);
        const long long plane = (long long)n2 * pitch;
        // 1-2. noise and forward transform; 3-4. whitening and PSDF filter; 5. inverse transform
        hipLaunchKernelGGL(k_rows_fwd, dim3(rowblk), b1, ax[0].lds, s, ax[0].f, c, pitch, rows, ax[0].nl,
                           (unsigned long long)seed);
        hipLaunchKernelGGL(k_cols<false>, dim3((unsigned)nt2 * n3), b2, ax[1].lds, s, ax[1].f, c, n1h, nt2,
                           (long long)pitch, plane, ax[1].nl, 1.0, fa);
        hipLaunchKernelGGL(k_cols<true>, dim3((unsigned)nt3 * n2), b3, ax[2].lds, s, ax[2].f, c, n1h, nt3, plane,
                           (long long)pitch, ax[2].nl, 1.0, fa);
        hipLaunchKernelGGL(k_cols<false>, dim3((unsigned)nt2 * n3), b2, ax[1].lds, s, ax[1].f, c, n1h, nt2,
                           (long long)pitch, plane, ax[1].nl, -1.0, fa);
        hipLaunchKernelGGL(k_rows_inv, dim3(rowblk), b1, ax[0].lds, s, ax[0].f, c, pitch, rows, ax[0].nl, part);
        // 6. mean and rms (m_rmedia.f90:144-159)
        hipLaunchKernelGGL(k_stats, dim3(1), dim3(256), 0, s, part, (int)rowblk, n, stats);
        hipLaunchKernelGGL(k_scale, dim3((unsigned)((rows + 15) / 16)), dim3(256), 0, s, c, pitch, rows, n1, stats,
                           (double)epsil, out_dev ? out : (float *)dout.p);
        RCHK(hipGetLastError());
        if (!out_dev) RCHK(hipMemcpyAsync(out, dout.p, (size_t)n * sizeof(float), hipMemcpyDeviceToHost, s));
        RCHK(hipStreamSynchronize(s));
        return SWPC_OK;
    }
    const int nblk = 2048;
    RCHK(hipMalloc(&dr.p, (size_t)n * sizeof(double)));
    RCHK(hipMalloc(&dc.p, (size_t)nc * sizeof(double2)));
    RCHK(hipMalloc(&dpart.p, (size_t)nblk * sizeof(double)));
    RCHK(hipMalloc(&dstats.p, 2 * sizeof(double)));
    if (!out_dev) RCHK(hipMalloc(&dout.p, (size_t)n * sizeof(float)));
    double *r = (double *)dr.p;
    double2 *c = (double2 *)dc.p;
    double *part = (double *)dpart.p, *stats = (double *)dstats.p;

    // 1. noise
    hipLaunchKernelGGL(k_noise, dim3(nblk), dim3(256), 0, s, r, n, (unsigned long long)seed);
    RCHK(hipGetLastError());
    // 2. forward transform, axis 1 fastest (hipFFT lists the slowest axis first)
    hipfftHandle fwd, inv;
    FCHK(hipfftPlan3d(&fwd, n3, n2, n1, HIPFFT_D2Z));
    struct PlanGuard { hipfftHandle h; ~PlanGuard() { (void)hipfftDestroy(h); } } pf{fwd};
    FCHK(hipfftSetStream(fwd, s));
    FCHK(hipfftExecD2Z(fwd, (hipfftDoubleReal *)r, (hipfftDoubleComplex *)c));
    // 3-4. whitening and PSDF filter
    fa.b = c;
    hipLaunchKernelGGL(k_filter, dim3(nblk), dim3(256), 0, s, fa);
    RCHK(hipGetLastError());
    // 5. inverse transform (the output is real: the filtered spectrum keeps
    // the Hermitian symmetry of the noise's)
    FCHK(hipfftPlan3d(&inv, n3, n2, n1, HIPFFT_Z2D));
    struct PlanGuard pi{inv};
    FCHK(hipfftSetStream(inv, s));
    FCHK(hipfftExecZ2D(inv, (hipfftDoubleComplex *)c, (hipfftDoubleReal *)r));
    // 6. mean and rms (m_rmedia.f90:144-159)
    hipLaunchKernelGGL(k_partial, dim3(nblk), dim3(256), 0, s, r, n, 0.0, 0, part);
    hipLaunchKernelGGL(k_total, dim3(1), dim3(256), 0, s, part, nblk, stats);
    RCHK(hipGetLastError());
    double sum = 0.0;
    RCHK(hipMemcpyAsync(&sum, stats, sizeof(double), hipMemcpyDeviceToHost, s));
    RCHK(hipStreamSynchronize(s));
    const double mean = sum / (double)n;
    hipLaunchKernelGGL(k_partial, dim3(nblk), dim3(256), 0, s, r, n, mean, 1, part);
    hipLaunchKernelGGL(k_total, dim3(1), dim3(256), 0, s, part, nblk, stats + 1);
    RCHK(hipGetLastError());
    double ss = 0.0;
    RCHK(hipMemcpyAsync(&ss, stats + 1, sizeof(double), hipMemcpyDeviceToHost, s));
    RCHK(hipStreamSynchronize(s));
    const double st[2] = {mean, std::sqrt(ss / (double)n)};
    RCHK(hipMemcpyAsync(stats, st, sizeof st, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_finish, dim3(nblk), dim3(256), 0, s, r, n, stats, (double)epsil,
                       out_dev ? out : (float *)dout.p);
    RCHK(hipGetLastError());
    if (!out_dev) RCHK(hipMemcpyAsync(out, dout.p, (size_t)n * sizeof(float), hipMemcpyDeviceToHost, s));
    RCHK(hipStreamSynchronize(s));
    return SWPC_OK;
}
